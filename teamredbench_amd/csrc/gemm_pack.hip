// 16-bit and fp8 GEMM whose rows are off 16 bytes (K or N not a multiple of 8,
// of 16 for fp8): the operands that are off are copied into the workspace with
// rows on 128 bytes, zeros after each row, and the LDS-DMA kernels run on the
// copies (their DMA loads need 16-byte sources; gemm_tiled_kernels.hpp, ANY_N).
//
// The copy is bound by HBM: it reads and writes each repacked operand once, a
// small part of a product with many rows (up to 64 go to gemm_strip.hip) and a
// long K; kPackMinK says from where on it pays.
#include "gemm_common.hpp"

namespace mb {
namespace {

typedef u32x4 u32x4_any __attribute__((aligned(1)));

// Rows of `row_bytes` bytes at any address into rows of `chunks` 16-byte
// pieces, zeros past row_bytes. Piece i is piece i - row * chunks of row
// (i * magic) >> shift (exact for i < 2^27).
struct PackJob {
    const unsigned char* src;
    unsigned char* dst;
    int64_t bytes;              // of src
    int row_bytes, chunks;
    unsigned pieces, blocks;
    unsigned magic, shift;
};

constexpr int kPackThreads = 256, kPackUnroll = 4;

// The first job's blocks, then the second's. A thread moves kPackUnroll pieces a
// block's width apart, all loads in flight before the first store.
__global__ void __launch_bounds__(kPackThreads)
pack_rows_kernel(PackJob first, PackJob second) {
    const bool two = blockIdx.x >= first.blocks;
    const PackJob& j = two ? second : first;
    const unsigned block = two ? blockIdx.x - first.blocks : blockIdx.x;
    const unsigned i0 = block * (kPackThreads * kPackUnroll) + threadIdx.x;
    u32x4 v[kPackUnroll];
#pragma unroll
    for (int u = 0; u < kPackUnroll; ++u) {
        const unsigned i = i0 + u * kPackThreads;
        v[u] = (u32x4){0u, 0u, 0u, 0u};
        if (i >= j.pieces) continue;
        const unsigned row = (unsigned)(((uint64_t)i * j.magic) >> j.shift);
        const int col = (int)(i - row * j.chunks) * 16;
        const int64_t at = (int64_t)row * j.row_bytes + col;
        const int left = j.row_bytes - col;                     // bytes of the row from here on
        if (left >= 16) {
            v[u] = *reinterpret_cast<const u32x4_any*>(j.src + at);
        } else if (left > 0) {
#pragma unroll
            for (int e = 0; e < 15; ++e)
                if (e < left) v[u][e >> 2] |= (unsigned)j.src[at + e] << 8 * (e & 3);
        }
    }
#pragma unroll
    for (int u = 0; u < kPackUnroll; ++u) {
        const unsigned i = i0 + u * kPackThreads;
        if (i < j.pieces) reinterpret_cast<u32x4*>(j.dst)[i] = v[u];
    }
}

PackJob pack_job(const void* src, void* dst, int64_t rows, int64_t row_bytes, int64_t pitch) {
    PackJob j{};
    if (src == nullptr) return j;
    j.src = static_cast<const unsigned char*>(src);
    j.dst = static_cast<unsigned char*>(dst);
    j.bytes = rows * row_bytes;
    j.row_bytes = (int)row_bytes;
    j.chunks = (int)(pitch / 16);
    j.pieces = (unsigned)(rows * j.chunks);
    j.blocks = (j.pieces + kPackThreads * kPackUnroll - 1) / (kPackThreads * kPackUnroll);
    unsigned bits = 0;
    while ((1u << bits) < (unsigned)j.chunks) ++bits;
    j.shift = 27 + bits;
    j.magic = (unsigned)(((uint64_t(1) << j.shift) + j.chunks - 1) / j.chunks);   // at most 2^28
    return j;
}

size_t align256(size_t v) { return (v + 255) & ~size_t(255); }

// The least K that pays for the copy and its launch (about 5 us together) against
// the bounds-checked kernel, whose time grows with K; columns under one of its
// tiles move its operands less often. 1800 random products on MI355X (M 1..8192,
// N and K 1..4096, all four types): repacked from these K on, one ran slower than
// on the bounds-checked kernel (0.96x) and all 1.28x faster in geometric mean;
// repacked everywhere, 977 ran slower, by up to 2.3x (fp16 5776 x 407 x 96 7.3
// against 14.7 us, e5m2 158 x 413 x 368 10.6 against 12.6 at worst beyond).
constexpr int64_t kPackMinK = 256, kPackMinKNarrow = 320, kPackNarrowN = 128;

}  // namespace

int gemm_packed_plan(int dtype, int64_t M, int64_t N, int64_t K, const DeviceProps& props, size_t scratch,
                     GemmPlan* plan) {
    const int64_t e = is_fp8(dtype) ? 1 : 2, grain = 16 / e;
    if (N >= (int64_t(1) << 31) || K >= (int64_t(1) << 31) || M >= (int64_t(1) << 31)) return MB_ERR_SHAPE;
    // (A forced tile is a call for these kernels.)
    if (K < (N < kPackNarrowN ? kPackMinKNarrow : kPackMinK) && tuning(MB_TUNE_GEMM_TILED_CONFIG) < 0) return MB_ERR_SHAPE;
    const int64_t np = (N + grain - 1) / grain * grain, kp = (K + grain - 1) / grain * grain;
    GemmPlan p;
    const char* why = "";
    if (gemm_tiled_plan(dtype, M, np, kp, props, Scratch{SIZE_MAX}, &p, &why) != MB_OK) return MB_ERR_SHAPE;
    p.pack_a = kp != K;
    p.pack_b = np != N;
    // Rows on 128 bytes: whole cache lines per tile row.
    p.lda = p.pack_a ? (K * e + 127) / 128 * 128 : K * e;
    p.ldb = p.pack_b ? (N * e + 127) / 128 * 128 : N * e;
    // 32-bit buffer offsets and piece counts (2^27 pieces are 2 GiB), as in gemm_tiled_plan.
    const int64_t k_end = ((K * e + 63) / 64 + p.split_k - 1) / p.split_k * p.split_k * 64 / e;
    if (k_end * p.ldb + 512 >= (int64_t(1) << 31) || 256 * (p.lda + 64 * p.split_k) >= (int64_t(1) << 31) ||
        M * p.lda >= (int64_t(1) << 31) || M * (np + 8) >= (int64_t(1) << 31))
        return MB_ERR_SHAPE;
    size_t at = 0;
    if (p.pack_b) p.b_offset = at, at = align256(at + (size_t)(K * p.ldb));
    if (p.pack_a) p.a_offset = at, at = align256(at + (size_t)(M * p.lda));
    p.partials_offset = at;
    if (p.split_k > 1) at += (size_t)p.split_k * (size_t)M * (size_t)((N + 7) / 8 * 8) * sizeof(float);
    if (at > scratch) return MB_ERR_SHAPE;
    p.packed = true;
    p.workspace = at;
    p.implementation = "gfx950_mfma_generic";   // the name of all shapes off 16 bytes; the family tells them apart
    p.family = "repacked_tiled";
    p.variant = kVariantPacked;
    *plan = p;
    return MB_OK;
}

int gemm_packed_launch(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                       float alpha, void* workspace, const GemmPlan& plan, hipStream_t stream) {
    const int64_t e = is_fp8(dtype) ? 1 : 2;
    auto* ws = static_cast<unsigned char*>(workspace);
    const PackJob b = pack_job(plan.pack_b ? B : nullptr, ws + plan.b_offset, K, N * e, plan.ldb);
    const PackJob a = pack_job(plan.pack_a ? A : nullptr, ws + plan.a_offset, M, K * e, plan.lda);
    hipLaunchKernelGGL(pack_rows_kernel, dim3(b.blocks + a.blocks), dim3(kPackThreads), 0, stream, b, a);
    MB_HIP_TRY(hipGetLastError());
    return gemm_tiled_launch(dtype, plan.pack_a ? a.dst : A, plan.pack_b ? b.dst : B, C, M, N, K, alpha,
                             ws + plan.partials_offset, plan, stream);
}

}  // namespace mb
