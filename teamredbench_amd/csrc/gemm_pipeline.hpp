// Device helpers shared by the LDS-DMA pipelined GEMM kernels (gemm_tiled.hip
// for 16-bit and fp8 inputs, gemm_highp.hip for fp32): the global -> LDS DMA
// load, the vmcnt-bounded workgroup barrier, the A-row LDS swizzle and the
// XCD-aware tile order.
#pragma once

#include "gemm_common.hpp"

#define MB_LDS __attribute__((address_space(3)))

namespace mb {
namespace {

constexpr int kBufferFlags = 0x00020000;  // raw buffer resource word 3 on gfx9

// A-side rows of 64 bytes (4 chunks of 16 bytes): chunk c of row r is stored
// at chunk c ^ swz_a(r), which keeps the 16-byte operand reads of 32
// consecutive rows free of LDS bank conflicts (8- and 16-lane phases).
__device__ __forceinline__ int swz_a(int r) { return ((r >> 1) & 3) ^ ((r >> 3) & 1); }

// A-side rows of 128 bytes (8 chunks): chunk c of row r is stored at chunk
// c ^ swz_a2(r). For the operand reads (32 consecutive rows, one logical chunk
// per half wave) every 8 consecutive rows land on 8 distinct 16-byte bank
// groups and every 16 on 16 distinct (row parity, chunk) pairs: no bank
// conflicts for 8- or 16-lane LDS phases.
__device__ __forceinline__ int swz_a2(int r) { return ((r >> 1) & 7) ^ ((r & 1) << 2); }

// Wait until at most N vector-memory operations of this wave are pending and
// its LDS operations have drained, then join the workgroup barrier. The empty
// asm with a memory clobber keeps the compiler from moving LDS accesses
// across the barrier (the barrier builtin alone does not order memory).
template <int N>
__device__ __forceinline__ void wait_vmcnt_and_barrier() {
    static_assert(N >= 0 && N < 64, "vmcnt is a 6-bit counter");
    // gfx9 s_waitcnt encoding: vmcnt[3:0] | expcnt[6:4] | lgkmcnt[11:8] | vmcnt[5:4] at [15:14]
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0x0 << 8));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// One LDS-DMA load: every lane fetches 16 bytes at rsrc + voff + soff and the
// wave writes them to LDS bytes [lds_addr, lds_addr + 1024) in lane order.
// Issued as inline asm so the compiler's wait insertion, which cannot tell
// which ring slot the write lands in, does not put a full vmcnt drain in
// front of every later LDS read; the callers order these loads themselves.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"
__device__ __forceinline__ void lds_dma16(__amdgpu_buffer_rsrc_t rsrc, unsigned lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
}
// The same with 4 bytes per lane (256 LDS bytes per instruction): sources on 4 bytes.
__device__ __forceinline__ void lds_dma4(__amdgpu_buffer_rsrc_t rsrc, unsigned lds_addr, int voff, int soff) {
    asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rsrc), "s"(soff)
                 : "memory", "m0");
}
#pragma clang diagnostic pop

template <int BYTES>
__device__ __forceinline__ void lds_dma(__amdgpu_buffer_rsrc_t rsrc, unsigned lds_addr, int voff, int soff) {
    static_assert(BYTES == 16 || BYTES == 4, "bytes per lane of an LDS-DMA load");
    if constexpr (BYTES == 16) lds_dma16(rsrc, lds_addr, voff, soff);
    else lds_dma4(rsrc, lds_addr, voff, soff);
}

// Block -> (K split, tile row, tile column). Blocks are dispatched round-robin
// over the 8 XCDs (block b on XCD b % 8). Without splits, and with a split
// count that is no power of two, each XCD gets a contiguous run of (split,
// tile) pairs, split by split, a split's tiles in groups of `group_m` tile
// rows: its concurrent tiles form a compact patch of a split, whose A and B
// panels its L2 shares, whatever the counts. A power of two keeps the splits
// of a tile adjacent: up to 8 of them, the XCDs then divide the splits among
// them already. Over 349 plans of 2 to 32 splits on MI355X (1 to 512 tiles of
// 64 x 64 to 128 x 256, operands from HBM) either order is within 1.2% of the
// other in geometric mean, except with tile counts that are multiples of 8, as
// the plan's own few-row picks are: adjacent splits 2.4% faster at 4, 1.2% at 8,
// 3.2% at 16, equal at 2, 1.7% slower at 32. Tile counts that are no multiple of
// 8, dealt out over the XCDs before: 1.05x in geometric mean over 970 unsplit
// bf16 / fp16 / fp8 plans, multiples of 8 (the same map) 1.02x in the same runs;
// 5740 odd splits 1.04x.
__device__ __forceinline__ void block_coords(int b, int tiles_m, int tiles_n, int splits, int group_m, int* tm,
                                             int* tn, int* split) {
    const int tiles = tiles_m * tiles_n;
    int t;
    if (splits > 1 && (splits & (splits - 1)) == 0) {
        *split = b & (splits - 1);
        t = b / splits;
        if ((tiles & 7) == 0) t = (t & 7) * (tiles >> 3) + (t >> 3);
    } else {
        const int blocks = tiles * splits;
        t = (b & 7) * (blocks >> 3) + min(b & 7, blocks & 7) + (b >> 3);
        *split = splits > 1 ? t / tiles : 0;
        t -= *split * tiles;
    }
    const int per_group = group_m * tiles_n;
    const int g = t / per_group;
    const int first_m = g * group_m;
    const int rows = min(tiles_m - first_m, group_m);
    const int r = t - g * per_group;
    *tm = first_m + r % rows;
    *tn = r / rows;
}

}  // namespace
}  // namespace mb
