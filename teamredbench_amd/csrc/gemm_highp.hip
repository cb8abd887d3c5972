// fp32 and fp64 GEMM for gfx950 on the full-precision matrix cores:
// C = A * B, A (M x K), B (K x N), C (M x N) all row-major in the input type,
// accumulated in that type by the MFMAs (fp32: v_mfma_f32_32x32x2_f32; fp64:
// v_mfma_f64_16x16x4_f64), for any M, N, K >= 1.
//
// Two kernels. An LDS-DMA ring like the 16-bit pipelined kernel
// (gemm_f32_dma_kernel, gemm_f64_dma_kernel below: 95% and 93% of peak at
// 8192^3) runs every shape within 32-bit buffer offsets, on tiles from 256 x
// 256 (fp32) to 32 x 128, with K split over idle CUs when the caller gives a
// workspace (highp_choose). The rest, and some products of a short K (under 16,
// 24), run the register-staged kernel that follows, which indexes with 64 bits
// and stays near 80% of peak:
//
// Register-staged kernel. Operands come through registers into a
// double-buffered LDS tile (one barrier per stage), and the next stage's
// global loads are in flight while the current stage's MFMAs run. A 128 x 128
// block tile with 64 bytes of K per stage, 4 waves in a 2 x 2 grid owning
// 64 x 64 of C each.
//
// LDS layout per stage: A transposed to [BK][BM + pad] (the MFMA hands each
// lane one A row at a fixed k, so consecutive lanes read consecutive
// addresses) and B as [BK][BN + pad]. The threads that load A are laid out
// rows first, so the transposing stores of a wave also go to 64 consecutive
// rows of one k. The 128-byte pad puts the lanes that
// read the next k (fp32: lanes 32-63; fp64: every other group of 16) on the
// other half of the 64 banks, so operand reads are conflict-free.
//
// Global loads move 16 bytes per lane when the row pitches keep 16-byte
// alignment (K and N multiples of 16 / elem bytes); otherwise element-wise.
// Either way elements outside the matrices read as zero and stores outside C
// are skipped, so ragged edges need no separate kernel.
#include "gemm_pipeline.hpp"

#include <utility>

namespace mb {
namespace {

constexpr int kHpBM = 128, kHpBN = 128, kHpThreads = 256;

template <typename T>
struct HighpTraits;

// fp32: 32 x 32 fragments, K = 2 per MFMA; lane l supplies A[row l%32][k l/32]
// and B[k l/32][col l%32]; accumulator r = 4g + q holds row 8g + 4*(l/32) + q,
// col l%32.
template <>
struct HighpTraits<float> {
    static constexpr int kBK = 16;        // K elements per stage (64 bytes)
    static constexpr int kFrag = 32;
    static constexpr int kFragK = 2;
    static constexpr int kAcc = 16;
    typedef f32x16 Acc;
    __device__ static inline Acc mfma(float a, float b, Acc c) {
        return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
    }
    // Row (within the fragment) of accumulator register r for lane l.
    __device__ static inline int acc_row(int r, int lane) { return 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3); }
    __device__ static inline int lane_k(int lane) { return lane >> 5; }
    __device__ static inline int lane_mn(int lane) { return lane & 31; }
};

// fp64: 16 x 16 fragments, K = 4 per MFMA; lane l supplies A[row l%16][k l/16]
// and B[k l/16][col l%16]; accumulator r holds row 4r + l/16, col l%16 (each
// register is one group of 4 rows interleaved over the four 16-lane blocks,
// unlike the fp32 16x16 form, whose lane block owns 4 consecutive rows).
template <>
struct HighpTraits<double> {
    static constexpr int kBK = 8;         // K elements per stage (64 bytes)
    static constexpr int kFrag = 16;
    static constexpr int kFragK = 4;
    static constexpr int kAcc = 4;
    typedef f64x4 Acc;
    __device__ static inline Acc mfma(double a, double b, Acc c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    __device__ static inline int acc_row(int r, int lane) { return 4 * r + (lane >> 4); }
    __device__ static inline int lane_k(int lane) { return lane >> 4; }
    __device__ static inline int lane_mn(int lane) { return lane & 15; }
};

template <typename T, bool VEC>
__global__ void __launch_bounds__(kHpThreads)
gemm_highp_kernel(const T* __restrict__ A, const T* __restrict__ B, T* __restrict__ C, int64_t M, int64_t N,
                  int64_t K) {
    typedef HighpTraits<T> Tr;
    typedef typename Tr::Acc Acc;
    constexpr int BK = Tr::kBK;
    constexpr int F = Tr::kFrag;
    constexpr int FR = 64 / F;                    // fragments per wave side (wave tile 64 x 64)
    constexpr int V = 16 / (int)sizeof(T);        // elements per 16-byte vector
    constexpr int PAD = 128 / (int)sizeof(T);     // 128 bytes: half the LDS banks
    constexpr int A_LD = kHpBM + PAD;             // padded row of the transposed A tile
    constexpr int B_LD = kHpBN + PAD;
    constexpr int A_VECS = kHpBM * BK / V;        // 16-byte pieces per stage
    constexpr int B_VECS = BK * kHpBN / V;
    constexpr int PER_A = A_VECS / kHpThreads, PER_B = B_VECS / kHpThreads;
    static_assert(A_VECS % kHpThreads == 0 && B_VECS % kHpThreads == 0, "stage must split over the threads");

    __shared__ T sa[2][BK][A_LD];
    __shared__ __attribute__((aligned(16))) T sb[2][BK][B_LD];

    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int64_t m0 = (int64_t)blockIdx.y * kHpBM, n0 = (int64_t)blockIdx.x * kHpBN;

    T ra[PER_A][V], rb[PER_B][V];
    // Global -> registers for the stage at k0; zero outside the matrices.
    auto load = [&](int64_t k0) {
#pragma unroll
        for (int q = 0; q < PER_A; ++q) {
            const int v = tid + q * kHpThreads;
            const int row = v % kHpBM, kv = (v / kHpBM) * V;
            const int64_t gm = m0 + row, gk = k0 + kv;
            if constexpr (VEC) {
                if (gm < M && gk < K) {
                    *reinterpret_cast<u32x4*>(ra[q]) = *reinterpret_cast<const u32x4*>(A + gm * K + gk);
                } else {
#pragma unroll
                    for (int e = 0; e < V; ++e) ra[q][e] = T(0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) ra[q][e] = (gm < M && gk + e < K) ? A[gm * K + gk + e] : T(0);
            }
        }
#pragma unroll
        for (int q = 0; q < PER_B; ++q) {
            const int v = tid + q * kHpThreads;
            const int kr = v / (kHpBN / V), cv = (v % (kHpBN / V)) * V;
            const int64_t gk = k0 + kr, gn = n0 + cv;
            if constexpr (VEC) {
                if (gk < K && gn < N) {
                    *reinterpret_cast<u32x4*>(rb[q]) = *reinterpret_cast<const u32x4*>(B + gk * N + gn);
                } else {
#pragma unroll
                    for (int e = 0; e < V; ++e) rb[q][e] = T(0);
                }
            } else {
#pragma unroll
                for (int e = 0; e < V; ++e) rb[q][e] = (gk < K && gn + e < N) ? B[gk * N + gn + e] : T(0);
            }
        }
    };
    // Registers -> LDS buffer `buf` (A transposed).
    auto store = [&](int buf) {
#pragma unroll
        for (int q = 0; q < PER_A; ++q) {
            const int v = tid + q * kHpThreads;
            const int row = v % kHpBM, kv = (v / kHpBM) * V;
#pragma unroll
            for (int e = 0; e < V; ++e) sa[buf][kv + e][row] = ra[q][e];
        }
#pragma unroll
        for (int q = 0; q < PER_B; ++q) {
            const int v = tid + q * kHpThreads;
            const int kr = v / (kHpBN / V), cv = (v % (kHpBN / V)) * V;
            *reinterpret_cast<u32x4*>(&sb[buf][kr][cv]) = *reinterpret_cast<const u32x4*>(rb[q]);
        }
    };

    Acc acc[FR][FR];
#pragma unroll
    for (int i = 0; i < FR; ++i)
#pragma unroll
        for (int j = 0; j < FR; ++j)
#pragma unroll
            for (int r = 0; r < Tr::kAcc; ++r) acc[i][j][r] = T(0);

    const int lk = Tr::lane_k(lane), lmn = Tr::lane_mn(lane);
    const int64_t ksteps = (K + BK - 1) / BK;
    load(0);
    store(0);
    __syncthreads();
    for (int64_t kt = 0; kt < ksteps; ++kt) {
        const int buf = (int)(kt & 1);
        if (kt + 1 < ksteps) load((kt + 1) * BK);
#pragma unroll
        for (int kk = 0; kk < BK; kk += Tr::kFragK) {
            T a[FR], b[FR];
#pragma unroll
            for (int i = 0; i < FR; ++i) a[i] = sa[buf][kk + lk][wm * 64 + i * F + lmn];
#pragma unroll
            for (int j = 0; j < FR; ++j) b[j] = sb[buf][kk + lk][wn * 64 + j * F + lmn];
#pragma unroll
            for (int i = 0; i < FR; ++i)
#pragma unroll
                for (int j = 0; j < FR; ++j) acc[i][j] = Tr::mfma(a[i], b[j], acc[i][j]);
        }
        if (kt + 1 < ksteps) store(buf ^ 1);
        __syncthreads();
    }

    // Epilogue: a register index gives each lane one row; consecutive lanes
    // hold consecutive columns of it.
#pragma unroll
    for (int i = 0; i < FR; ++i) {
#pragma unroll
        for (int j = 0; j < FR; ++j) {
            const int64_t gn = n0 + wn * 64 + j * F + lmn;
#pragma unroll
            for (int r = 0; r < Tr::kAcc; ++r) {
                const int64_t gm = m0 + wm * 64 + i * F + Tr::acc_row(r, lane);
                if (gm < M && gn < N) C[gm * N + gn] = acc[i][j][r];
            }
        }
    }
}

// ---- fp32 on an LDS-DMA ring (256 x 256 and 128 x 128 tiles) ---------------
//
// The register-staged kernel above tops out near 80% of the fp32 peak: its
// load, LDS store and barrier phases leave the matrix pipe idle between MFMA
// groups. This one follows the 16-bit pipelined kernel instead: A and B go
// global -> LDS with buffer_load ... lds into a ring of 4 slots (one barrier
// per stage, loads of stage kt + 3 issued into the slot stage kt - 1 just
// vacated), and on 256 x 256 tiles each wave owns 128 x 128 of C as 4 x 4
// fragments of v_mfma_f32_32x32x2_f32, so a stage is 128 MFMAs (8192 cycles)
// against one barrier.
//
// K order inside a stage. The MFMA sums two K values, one from each lane
// half; here lane half h supplies K 8h + t at step t (t = 0..7), which is any
// fixed permutation of the stage's 16 K values and leaves the sum the same.
// So a lane's A operands for the whole stage are 8 consecutive floats of one
// row -- two ds_read_b128 per fragment from the [256 rows][64 B] A slot (the
// 16-bit kernel's layout and swizzle) -- and its B operand at step t is one
// float of row 8h + t, read with ds_read_b32. B keeps its HBM layout ([16
// rows][1024 B]); rows 8..15 have their 16-byte chunks XOR 8, so the two lane
// halves, which read rows 8 apart (8 KiB, the same banks), land 128 bytes
// apart and the read is conflict-free.
//
// The MFMA takes the B operand first, so a lane's 16 accumulators of a
// fragment hold one C row, 4 runs of 4 consecutive columns; the epilogue
// stores them as 16-byte pieces straight from registers (a tile computes for
// milliseconds; its 256 KiB of C do not need LDS staging).
constexpr int kHpStages = 4, kHpGroupM = 4;   // ring slots; tile rows per XCD group

// Chunk c of B row r sits at chunk c ^ swz_b32(r). Rows of 32 columns (128
// bytes) have no chunk 8; there rows 8..15 are swapped in pairs instead
// (f32_b_row), so that the halves' rows, 8 apart, differ in parity: the odd
// row lies on the other half of the banks.
template <int BN, int SK>
__device__ __forceinline__ int swz_b32(int row) { return BN >= 64 ? (row >= SK / 2 ? 8 : 0) : 0; }
template <int BN, int SK>
__device__ __forceinline__ int f32_b_row(int row) { return BN >= 64 ? row : row ^ (row >= SK / 2 ? 1 : 0); }

// A rows of 64 or 128 bytes.
template <int ROW>
__device__ __forceinline__ int swz_hp_a(int row) { return ROW == 64 ? swz_a(row) : swz_a2(row); }

typedef f32x4 f32x4_any __attribute__((aligned(4)));

// The loads that go out after MFMA s of `mfmas`: load l follows MFMA
// l * mfmas / loads; the first such l at or after MFMA s.
constexpr int load_at(int s, int mfmas, int loads) { return (s * loads + mfmas - 1) / mfmas; }

template <int LO, int HI, class F>
__device__ __forceinline__ void issue_range(F f) {
    [&]<int... I>(std::integer_sequence<int, I...>) {
        (f(std::integral_constant<int, LO + I>{}), ...);
    }(std::make_integer_sequence<int, HI - LO>{});
}

// Tile shapes. Waves form a WGM x WGN grid of 32 x 32 fragments; a stage is SK
// K values, 64 or 128 bytes of an A row. 128 x 128 tiles run eight waves, two
// per SIMD, so one's barrier waits hide under the other's MFMAs (2048^3 fp32
// 127.7 us against 137.9 with four; 4% over 335 shapes of one block per CU).
// DMA pieces are PA / PB bytes of A / B per lane: 16, or 4 for rows off 16
// bytes (K or N not a multiple of 4), where a lane's 16 bytes would not start
// on 16 in memory. A 4-byte piece costs four times the load instructions,
// which the 64-cycle MFMAs cover: fp32 4096 x 4001 x 4096 951 us against 929 at
// N = 4096 (1659 on the register-staged kernel).
template <int BM, int BN, int WGM, int WGN, int SK, int PA, int PB, bool RAGGED_K>
__global__ void __launch_bounds__(64 * WGM * WGN)
gemm_f32_dma_kernel(const float* __restrict__ A, const float* __restrict__ B, float* __restrict__ C, int M, int N,
                    int K, int tiles_m, int tiles_n, int splits, int k_len, float* __restrict__ ws) {
    constexpr int W = WGM * WGN;
    constexpr int WTM = BM / WGM, WTN = BN / WGN, FM = WTM / 32, FN = WTN / 32;
    constexpr int ARow = SK * 4, ABytes = BM * ARow, BRow = BN * 4, BBytes = SK * BRow, Slot = ABytes + BBytes;
    constexpr int AInstr = ABytes / (64 * PA) / W, BInstr = BBytes / (64 * PB) / W, Loads = AInstr + BInstr;
    static_assert(AInstr * W * 64 * PA == ABytes && BInstr * W * 64 * PB == BBytes, "a stage splits over the waves");
    static_assert(WTM % 32 == 0 && WTN % 32 == 0 && BRow >= 128, "tile shape");
    __shared__ __attribute__((aligned(1024))) unsigned char ring[kHpStages][Slot];
    const int tid = threadIdx.x, lane = tid & 63, half = lane >> 5;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    int tm, tn, split;
    block_coords((int)blockIdx.x, tiles_m, tiles_n, splits, kHpGroupM, &tm, &tn, &split);
    const int lda = K * 4, ldb = N * 4;
    const int k0 = split * k_len;
    // Buffer ranges end at A's row M and at B's last byte: rows of a partial
    // last M tile, and B's rows past K, load zeros; the columns of a partial
    // last N tile load the start of B's next row and are not stored.
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(A) + (int64_t)tm * BM * K, (short)0, min(BM, M - tm * BM) * lda, kBufferFlags);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<float*>(B) + (int64_t)tn * BN, (short)0, K * ldb - tn * BN * 4, kBufferFlags);
    int a_voff[AInstr], a_kbyte[AInstr], b_voff[BInstr];
#pragma unroll
    for (int q = 0; q < AInstr; ++q) {
        const int lin = (wave * AInstr + q) * 64 * PA + lane * PA;
        const int row = lin / ARow, pchunk = (lin % ARow) >> 4;
        a_kbyte[q] = ((pchunk ^ swz_hp_a<ARow>(row)) << 4) + (lin & 15);
        a_voff[q] = row * lda + a_kbyte[q];
    }
#pragma unroll
    for (int q = 0; q < BInstr; ++q) {
        const int lin = (wave * BInstr + q) * 64 * PB + lane * PB;
        const int slot_row = lin / BRow, pchunk = (lin % BRow) >> 4;
        b_voff[q] = f32_b_row<BN, SK>(slot_row) * ldb + ((pchunk ^ swz_b32<BN, SK>(slot_row)) << 4) + (lin & 15);
    }
    // DMA instruction q of stage kt into `slot`: A pieces first, then B.
    // RAGGED_K (the splits' stages run past K): A pieces at or past K load zeros.
    auto issue_one = [&](int kt, int slot, auto idx) {
        constexpr int q = decltype(idx)::value;
        const unsigned base = (unsigned)(uintptr_t)(MB_LDS unsigned char*)ring[slot];
        const int kb = k0 * 4 + kt * ARow;
        if constexpr (q < AInstr) {
            lds_dma<PA>(ra, base + (wave * AInstr + q) * 64 * PA,
                            RAGGED_K && a_kbyte[q] >= K * 4 - kb ? (int)0x80000000u : a_voff[q], kb);
        } else {
            lds_dma<PB>(rb, base + ABytes + (wave * BInstr + q - AInstr) * 64 * PB, b_voff[q - AInstr],
                        (k0 + kt * SK) * ldb);
        }
    };
    auto issue = [&](int kt, int slot) {
        [&]<int... Q>(std::integer_sequence<int, Q...>) {
            (issue_one(kt, slot, std::integral_constant<int, Q>{}), ...);
        }(std::make_integer_sequence<int, Loads>{});
    };

    f32x16 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;

    const int ksteps = k_len / SK, last = ksteps - 1;
#pragma unroll
    for (int st = 0; st < kHpStages - 1; ++st) issue(min(st, last), st);
    const int a_row = wm * WTM + (lane & 31);
    const int b_col = wn * WTN + (lane & 31);
    // A operands: a[i][t] is K SK / 2 * h + t of fragment i's row. The next
    // stage's first half is read into the registers this stage's first half of
    // steps is done with (after the mid-stage barrier), its second half at the
    // stage boundary, half a stage before it is needed: one register set.
    float a[FM][SK / 2];
    float b[4][FN];     // B operands of steps t .. t + 3, read two steps ahead
    auto read_a = [&](int kt, auto hc) {
        constexpr int hf = decltype(hc)::value;
        const unsigned char* slot = ring[kt % kHpStages];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int row = a_row + 32 * i;
#pragma unroll
            for (int e = hf * (SK / 16); e < (hf + 1) * (SK / 16); ++e) {
                // Whole float vectors: __builtin_bit_cast of a single ext_vector
                // element (bit_cast(float, v[w]) on a u32x4) is miscompiled by this
                // clang -- it reuses element 0 and drops the other loads.
                const f32x4 v = *reinterpret_cast<const f32x4*>(
                    slot + row * ARow + (((SK / 8 * half + e) ^ swz_hp_a<ARow>(row)) << 4));
#pragma unroll
                for (int w = 0; w < 4; ++w) a[i][4 * e + w] = v[w];
            }
        }
    };
    auto read_b = [&](int kt, int t, int set) {
        const unsigned char* sb = ring[kt % kHpStages] + ABytes;
        const int row = f32_b_row<BN, SK>(SK / 2 * half + t);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int col = b_col + 32 * j;
            b[set][j] = *reinterpret_cast<const float*>(sb + row * BRow + (((col >> 2) ^ swz_b32<BN, SK>(row)) << 4) +
                                                        4 * (col & 3));
        }
    };
    // One barrier per stage, at its middle: it certifies that stage kt + 1 has
    // landed for every wave and that every wave is done with stage kt - 1's
    // slot, which takes stage kt + 3's loads. Those loads are spread over the
    // stage's second half, evenly between its MFMAs (issued back to back after
    // the barrier, they held the wave's issue for longer than the one MFMA in
    // flight covers). The next stage's operands are read under this stage's
    // MFMAs (A's first chunk after the barrier, its first two B operands in
    // the last two steps, A's second chunk at the boundary), so a stage
    // boundary has no wait. B is read two steps (8 or 32 MFMAs) ahead of its
    // use: on 128 x 128 tiles one step (4 MFMAs) did not cover the LDS
    // latency when two blocks share a CU (3072 x 6144 x 4096 ran 17% faster
    // with two; other shapes within 0.7%). Past the last stage the loads
    // repeat it (in bounds, never used).
    constexpr int kSteps = SK / 2, kMid = kSteps / 2;
    static_assert(kSteps % 4 == 0 && kMid >= 2, "B sets cycle with the stage; next-stage reads follow the barrier");
    constexpr int kMfma = FM * FN;                               // MFMAs per step
    constexpr int kLoadMfma = kMfma * (kSteps - kMid);           // MFMAs of the second half
    wait_vmcnt_and_barrier<Loads * (kHpStages - 2)>();
    read_a(0, std::integral_constant<int, 0>{});
    read_a(0, std::integral_constant<int, 1>{});
    read_b(0, 0, 0);
    read_b(0, 1, 1);
    for (int kt = 0; kt < ksteps; ++kt) {
        const int load_kt = min(kt + kHpStages - 1, last), load_slot = (kt + kHpStages - 1) % kHpStages;
        [&]<int... T>(std::integer_sequence<int, T...>) {
            ([&] {
                constexpr int t = T;
                if (t == 0 && kt > 0) read_a(kt, std::integral_constant<int, 1>{});
                if constexpr (t == kMid) {
                    wait_vmcnt_and_barrier<Loads * (kHpStages - 3)>();
                    read_a(kt + 1, std::integral_constant<int, 0>{});
                }
                // (t + 2) & 3 is also the set of step t + 2 - kSteps of the next stage: kSteps % 4 == 0
                if constexpr (t + 2 < kSteps) read_b(kt, t + 2, (t + 2) & 3);
                else read_b(kt + 1, t + 2 - kSteps, (t + 2) & 3);
                __builtin_amdgcn_sched_barrier(0);
                [&]<int... Q>(std::integer_sequence<int, Q...>) {
                    ([&] {
                        constexpr int m = Q, i = m / FN, j = m % FN;
                        acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(b[t & 3][j], a[i][t], acc[i][j], 0, 0, 0);
                        // Load l follows MFMA l * kLoadMfma / Loads of the second half.
                        if constexpr (t >= kMid)
                            issue_range<load_at((t - kMid) * kMfma + m, kLoadMfma, Loads),
                                        load_at((t - kMid) * kMfma + m + 1, kLoadMfma, Loads)>(
                                [&](auto idx) { issue_one(load_kt, load_slot, idx); });
                        __builtin_amdgcn_sched_barrier(0);   // keeps each load where it is placed
                    }(), ...);
                }(std::make_integer_sequence<int, kMfma>{});
            }(), ...);
        }(std::make_integer_sequence<int, kSteps>{});
    }
    wait_vmcnt_and_barrier<0>();

    // Accumulator register 4g + q of lane l holds C[row 32i + l % 32]
    // [col 32j + 8g + 4 * (l / 32) + q] of the wave's tile. Rows at or past M
    // and columns at or past N are not stored; with K splits the block stores
    // its partial plane ws[split][M][N] instead of C.
    float* out = splits > 1 ? ws + (int64_t)split * M * N : C;
    const int col0 = tn * BN + wn * WTN + 4 * half;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const int row = tm * BM + wm * WTM + 32 * i + (lane & 31);
        if (row >= M) continue;
        float* crow = out + (int64_t)row * N + col0;
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 v = {acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
                const int left = N - (col0 + 32 * j + 8 * g);   // columns of C from here on
                float* p = crow + 32 * j + 8 * g;
                if constexpr (PB == 16) {
                    if (left > 0) *reinterpret_cast<f32x4*>(p) = v;   // N is a multiple of 4
                } else if (left >= 4) {
                    *reinterpret_cast<f32x4_any*>(p) = v;
                } else {
#pragma unroll
                    for (int e = 0; e < 3; ++e)
                        if (e < left) p[e] = v[e];
                }
            }
    }
}

// ---- fp64 on the same LDS-DMA ring (128 x 128 tiles) -----------------------
//
// v_mfma_f64_16x16x4_f64 sums four K values, one from each 16-lane group g;
// here group g supplies K 2g + t at step t (t = 0, 1) of a stage's 8, so a
// lane's A operands for the stage are 2 consecutive doubles of one row -- one
// ds_read_b128 per fragment from the [128 rows][64 B] A slot -- and its B
// operand at step t is one double of row 2g + t (ds_read_b64). B keeps its HBM
// layout, [8 rows][128 doubles = 1024 B]; rows with bit 1 set have their
// 16-byte chunks XOR 8, so groups 0 and 1 (and 2 and 3), which read rows 2
// apart (the same banks), land 128 bytes apart. Waves own 64 x 64 of C as
// 4 x 4 fragments (64 accumulator registers); A is the MFMA's first operand,
// so accumulator r of lane l is C row 4r + l / 16, column l % 16, and a store
// instruction writes 4 rows x 128 bytes straight from registers. With 64 KiB
// of ring and under 200 registers per lane, two blocks fit a CU, one wave of
// each on every SIMD: on MI355X these tiles ran up to 21% faster than
// 256 x 128 tiles (one block per CU) on 12 shapes from 3072 x 6144 x 4096 to
// 10240^2 x 4096, 8192^3 included (73.3 against 72.1 TFLOP/s), and 0.5%
// slower on one (4608^3).
template <int SK>
__device__ __forceinline__ int swz_b64(int row) { return ((row / (SK / 4)) & 1) << 3; }

template <int BM, int BN, int WGM, int WGN, int SK, int PA, int PB, bool RAGGED_K>
__global__ void __launch_bounds__(64 * WGM * WGN)
gemm_f64_dma_kernel(const double* __restrict__ A, const double* __restrict__ B, double* __restrict__ C, int M,
                    int N, int K, int tiles_m, int tiles_n, int splits, int k_len, double* __restrict__ ws) {
    // Waves in a WGM x WGN grid of 16 x 16 fragments; pieces as in gemm_f32_dma_kernel.
    constexpr int W = WGM * WGN;
    constexpr int WTM = BM / WGM, WTN = BN / WGN, FM = WTM / 16, FN = WTN / 16;
    constexpr int ARow = SK * 8, ABytes = BM * ARow, BRow = BN * 8, BBytes = SK * BRow, Slot = ABytes + BBytes;
    constexpr int AInstr = ABytes / (64 * PA) / W, BInstr = BBytes / (64 * PB) / W, Loads = AInstr + BInstr;
    static_assert(AInstr * W * 64 * PA == ABytes && BInstr * W * 64 * PB == BBytes, "a stage splits over the waves");
    static_assert(WTM % 16 == 0 && WTN % 16 == 0 && BRow >= 256, "tile shape");
    __shared__ __attribute__((aligned(1024))) unsigned char ring[kHpStages][Slot];
    const int tid = threadIdx.x, lane = tid & 63, grp = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave / WGN, wn = wave % WGN;
    int tm, tn, split;
    block_coords((int)blockIdx.x, tiles_m, tiles_n, splits, kHpGroupM, &tm, &tn, &split);
    const int lda = K * 8, ldb = N * 8;
    const int k0 = split * k_len;
    // Buffer ranges as in gemm_f32_dma_kernel: partial last tiles and a ragged K.
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double*>(A) + (int64_t)tm * BM * K, (short)0, min(BM, M - tm * BM) * lda, kBufferFlags);
    const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<double*>(B) + (int64_t)tn * BN, (short)0, K * ldb - tn * BN * 8, kBufferFlags);
    int a_voff[AInstr], a_kbyte[AInstr], b_voff[BInstr];
#pragma unroll
    for (int q = 0; q < AInstr; ++q) {
        const int lin = (wave * AInstr + q) * 64 * PA + lane * PA;
        const int row = lin / ARow, pchunk = (lin % ARow) >> 4;
        a_kbyte[q] = ((pchunk ^ swz_hp_a<ARow>(row)) << 4) + (lin & 15);
        a_voff[q] = row * lda + a_kbyte[q];
    }
#pragma unroll
    for (int q = 0; q < BInstr; ++q) {
        const int lin = (wave * BInstr + q) * 64 * PB + lane * PB;
        const int row = lin / BRow, pchunk = (lin % BRow) >> 4;
        b_voff[q] = row * ldb + ((pchunk ^ swz_b64<SK>(row)) << 4) + (lin & 15);
    }
    auto issue_one = [&](int kt, int slot, auto idx) {
        constexpr int q = decltype(idx)::value;
        const unsigned base = (unsigned)(uintptr_t)(MB_LDS unsigned char*)ring[slot];
        const int kb = k0 * 8 + kt * ARow;
        if constexpr (q < AInstr) {
            lds_dma<PA>(ra, base + (wave * AInstr + q) * 64 * PA,
                            RAGGED_K && a_kbyte[q] >= K * 8 - kb ? (int)0x80000000u : a_voff[q], kb);
        } else {
            lds_dma<PB>(rb, base + ABytes + (wave * BInstr + q - AInstr) * 64 * PB, b_voff[q - AInstr],
                        (k0 + kt * SK) * ldb);
        }
    };
    auto issue = [&](int kt, int slot) {
        [&]<int... Q>(std::integer_sequence<int, Q...>) {
            (issue_one(kt, slot, std::integral_constant<int, Q>{}), ...);
        }(std::make_integer_sequence<int, Loads>{});
    };

    f64x4 acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.0;

    const int ksteps = k_len / SK, last = ksteps - 1;
#pragma unroll
    for (int st = 0; st < kHpStages - 1; ++st) issue(min(st, last), st);
    const int a_row = wm * WTM + (lane & 15);
    const int b_col = wn * WTN + (lane & 15);
    constexpr int kSteps = SK / 4, kMid = kSteps / 2;   // group g takes K kSteps * g + t at step t
    double a[2][FM][kSteps];  // A operands of this stage and the next
    double b[2][FN];          // B operands of this step and the next
    auto read_a = [&](int kt, auto setc) {
        constexpr int set = decltype(setc)::value;
        const unsigned char* slot = ring[kt % kHpStages];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const int row = a_row + 16 * i;
#pragma unroll
            for (int e = 0; e < kSteps / 2; ++e) {
                const f64x2 v = *reinterpret_cast<const f64x2*>(
                    slot + row * ARow + (((kSteps / 2 * grp + e) ^ swz_hp_a<ARow>(row)) << 4));
                a[set][i][2 * e] = v[0];
                a[set][i][2 * e + 1] = v[1];
            }
        }
    };
    auto read_b = [&](int kt, int t, int set) {
        const unsigned char* sb = ring[kt % kHpStages] + ABytes;
        const int row = kSteps * grp + t;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            const int col = b_col + 16 * j;
            b[set][j] = *reinterpret_cast<const double*>(sb + row * BRow + (((col >> 1) ^ swz_b64<SK>(row)) << 4) +
                                                         8 * (col & 1));
        }
    };
    // The fp32 kernel's schedule: one barrier per stage, at its middle, after
    // which stage kt + 1's A operands are read under the second half's MFMAs
    // and its first B operands at the end of the stage; the loads of stage
    // kt + kHpStages - 1 are spread evenly between the second half's MFMAs.
    constexpr int kMfma = FM * FN, kLoadMfma = kMfma * (kSteps - kMid);
    auto stage = [&](int kt, auto curc) {
        constexpr int cur = decltype(curc)::value;
        const int load_kt = min(kt + kHpStages - 1, last), load_slot = (kt + kHpStages - 1) % kHpStages;
        [&]<int... T>(std::integer_sequence<int, T...>) {
            ([&] {
                constexpr int t = T;
                if constexpr (t == kMid) {
                    wait_vmcnt_and_barrier<Loads * (kHpStages - 3)>();
                    read_a(kt + 1, std::integral_constant<int, cur ^ 1>{});
                }
                if constexpr (t + 1 < kSteps) read_b(kt, t + 1, (t + 1) & 1);
                else read_b(kt + 1, 0, 0);
                __builtin_amdgcn_sched_barrier(0);
                [&]<int... Q>(std::integer_sequence<int, Q...>) {
                    ([&] {
                        constexpr int m = Q, i = m / FN, j = m % FN;
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[cur][i][t], b[t & 1][j], acc[i][j], 0, 0, 0);
                        if constexpr (t >= kMid)
                            issue_range<load_at((t - kMid) * kMfma + m, kLoadMfma, Loads),
                                        load_at((t - kMid) * kMfma + m + 1, kLoadMfma, Loads)>(
                                [&](auto idx) { issue_one(load_kt, load_slot, idx); });
                        __builtin_amdgcn_sched_barrier(0);   // keeps each load where it is placed
                    }(), ...);
                }(std::make_integer_sequence<int, kMfma>{});
            }(), ...);
        }(std::make_integer_sequence<int, kSteps>{});
    };
    wait_vmcnt_and_barrier<Loads * (kHpStages - 2)>();
    read_a(0, std::integral_constant<int, 0>{});
    read_b(0, 0, 0);
    for (int kt = 0; kt < ksteps; kt += 2) {
        stage(kt, std::integral_constant<int, 0>{});
        if (kt + 1 < ksteps) stage(kt + 1, std::integral_constant<int, 1>{});
    }
    wait_vmcnt_and_barrier<0>();

    // Rows at or past M and columns at or past N are not stored; with K splits
    // the block stores its partial plane.
    double* out = splits > 1 ? ws + (int64_t)split * M * N : C;
    const int col0 = tn * BN + wn * WTN + (lane & 15);
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int row = tm * BM + wm * WTM + 16 * i + 4 * r + grp;
            if (row >= M) continue;
            double* crow = out + (int64_t)row * N + col0;
#pragma unroll
            for (int j = 0; j < FN; ++j)
                if (col0 + 16 * j < N) crow[16 * j] = acc[i][j][r];
        }
}

// Sum of the K-split partials: C[i] = sum_s ws[s][i] over planes of `mn`
// elements, in split order. A thread takes 16 bytes of C and has L splits'
// loads in flight (the planes were just written: the pass is latency-bound).
// Planes and C need only element alignment.
template <typename T, int L>
__global__ void __launch_bounds__(64)
highp_split_sum_kernel(const T* __restrict__ ws, T* __restrict__ C, int64_t mn, int splits) {
    constexpr int V = 16 / (int)sizeof(T);
    typedef T Vec __attribute__((ext_vector_type(V)));
    typedef Vec VecAny __attribute__((aligned(sizeof(T))));
    const int64_t i = ((int64_t)blockIdx.x * 64 + threadIdx.x) * V;
    if (i + V <= mn) {
        Vec sum = *reinterpret_cast<const VecAny*>(ws + i);
        for (int s0 = 1; s0 < splits; s0 += L) {
            Vec v[L];
#pragma unroll
            for (int u = 0; u < L; ++u)
                v[u] = s0 + u < splits ? (Vec)*reinterpret_cast<const VecAny*>(ws + (s0 + u) * mn + i) : (Vec)T(0);
#pragma unroll
            for (int u = 0; u < L; ++u)
                if (s0 + u < splits) sum += v[u];
        }
        *reinterpret_cast<VecAny*>(C + i) = sum;
    } else {
        for (int64_t e = i; e < mn; ++e) {
            T sum = ws[e];
            for (int s = 1; s < splits; ++s) sum += ws[s * mn + e];
            C[e] = sum;
        }
    }
}

// Tiles of the LDS-DMA rings, by plan->config (0: the register-staged kernel).
struct HighpTile {
    int bm, bn, wgm, wgn;
    int row;                // bytes of A's K per row and stage: 64, or 128 (whole cache lines)
};
constexpr HighpTile kHighpTiles[] = {
    {128, 128, 0, 0, 64},   // 0: register-staged
    {256, 256, 2, 2, 64},   // 1: fp32 only
    {128, 128, 4, 2, 64},   // 2
    {128, 128, 4, 2, 128},  // 3: fp64, one block per CU
    {64, 64, 2, 2, 64},     // 4
    {32, 128, 1, 4, 128},   // 5
    {128, 32, 4, 1, 128},   // 6
};

// The ring's tile and K splits for a shape, using at most `scratch` bytes of
// partial planes; config 0 with *why set for a shape only the register-staged
// kernel takes.
struct HighpChoice {
    int config = 0, splits = 1;
    bool pieces4 = false;    // A's or B's rows off 16 bytes: 4-byte DMA pieces
};

HighpChoice highp_choose(bool f64, int64_t M, int64_t N, int64_t K, int cus, size_t scratch, const char** why) {
    HighpChoice ch;
    if (tuning(MB_TUNE_GEMM_HIGHP_STAGED) == 1) {
        *why = "forced by the gemm_highp_staged override";
        return ch;
    }
    const int64_t e = f64 ? 8 : 4;
    auto k_len = [&](int c, int64_t sp) {   // K per split, whole stages
        const int64_t stage_k = kHighpTiles[c].row / e, stages = (K + stage_k - 1) / stage_k;
        return (stages + sp - 1) / sp * stage_k;
    };
    // 32-bit offsets: bytes of B up to tile c's last stage of the last split (whole stages, so up to 128
    // bytes of K past K itself) and a partial tile's columns, and of an A panel.
    auto fits = [&](int c, int64_t sp) {
        const int64_t k_end = k_len(c, sp) * sp;
        return (k_end * N + 256) * e < (int64_t(1) << 31) && 256 * k_end * e < (int64_t(1) << 31);
    };
    if (!fits(2, 1)) {   // 64-byte stages end nearest to K
        *why = "operand offsets exceed 32-bit buffer addressing (K*N or 256*K bytes >= 2 GiB)";
        return ch;
    }
    // The LDS-DMA kernels take M and N as int (row and column guards); the
    // register-staged kernel indexes with int64.
    if (M >= (int64_t(1) << 31) || N >= (int64_t(1) << 31)) {
        *why = "M or N >= 2^31 exceeds the 32-bit row and column indexes of the LDS-DMA kernels";
        return ch;
    }
    auto tiles = [&](int c) {
        return ((M + kHighpTiles[c].bm - 1) / kHighpTiles[c].bm) * ((N + kHighpTiles[c].bn - 1) / kHighpTiles[c].bn);
    };
    if (tiles(2) > INT32_MAX) {
        *why = "more than 2^31 tiles";
        return ch;
    }
    if ((K * e) % 16 != 0) *why = f64 ? "K is not a multiple of 2" : "K is not a multiple of 4";
    else if ((N * e) % 16 != 0) *why = f64 ? "N is not a multiple of 2" : "N is not a multiple of 4";
    ch.pieces4 = **why != 0;
    auto rounds = [&](int64_t blocks) { return (blocks + cus - 1) / cus; };
    // fp32: 256 x 256 tiles run 2.5% faster per FLOP than 128 x 128 ones
    // (8192^3, whole rounds of either: 150.1 against 145.8 TFLOP/s on MI355X) but
    // come in rounds of four times the work, so they are taken only when their
    // rounds cost no more: rounds(256 x 256) <= rounds(128 x 128) / 4 / 0.975.
    // This picked the faster tile on all of 12 shapes measured: 256 x 256 at
    // 4096^3, 8192^3, 6144 x 8192 x 4096 and 5632^2 x 4096 (1.9 rounds, 2%);
    // 128 x 128 where the last 256 x 256 round is partly empty, 1.05-1.32x
    // faster there (6144^3 124.5 against 109.5 TFLOP/s, 3072 x 6144 x 4096
    // 109.3 against 83.9). Ragged M or N: partial last tiles on either. Their
    // 32 loads per wave and stage leave no room in vmcnt for 4-byte pieces.
    if (!f64 && !ch.pieces4 && tiles(1) >= cus &&
        4.0 * 0.975 * (double)rounds(tiles(1)) <= (double)rounds(tiles(2))) {
        ch.config = 1;
        return ch;
    }
    // Under 16 of K the register-staged kernel is done before the ring's three
    // stages of loads are: with rows off 16 bytes on 128 x 128 tiles, whose 4-byte
    // pieces are 24 loads a wave (fp64 280 x 4073 x 2 6.5 us against 8.9; of 779
    // products off 16 bytes 93 ran more than 3% slower than there before this rule,
    // none with it; from 16 on the ring is 1.5x faster), and in fp32 with more than
    // a round of them (1570 x 2668 x 4 8.2 us against 10.3, 2941 x 2939 x 5 13.5
    // against 17.8; 18 such products on 16 bytes 1.20x faster; off 16 bytes up to
    // 24 of K, 4000 x 3630 x 16 18.0 against 21.7). Its grid holds 65535 rows of
    // tiles.
    auto short_k = [&](HighpChoice c) {
        const bool crowded = !f64 && tiles(2) > cus;
        if (c.config == 2 && c.splits == 1 && M <= 65535 * (int64_t)kHpBM && K < (c.pieces4 && crowded ? 24 : 16) &&
            (c.pieces4 || crowded)) {
            c.config = 0;
            if (!c.pieces4) *why = "K is under 16";
        }
        return c;
    };
    // 128 x 128 tiles where they fill whole rounds exactly, and for K of a few
    // stages, where the tile hardly matters (under one, up to 64 of them leave
    // the CUs idle: 64 x 64 tiles 1.1-1.6x faster). fp64 with one block per CU takes
    // 128-byte rows of A (2048^3 249 against 254 us; with more blocks their
    // 128 KiB of ring leave one block per CU and run 8-9% slower).
    const bool few_stages = K < 128 && M >= 512 && (K >= 16 || ch.pieces4 || tiles(2) > 64);
    if ((M % 128 == 0 && N % 128 == 0 && tiles(2) % cus == 0) || few_stages) {
        ch.config = f64 && tiles(2) <= cus && K >= 128 && fits(3, 1) ? 3 : 2;
        return short_k(ch);
    }
    // The rest: the tile and the K split that a cost model rates fastest,
    //   MFMA     = rounds x 2 * BM * BN * K / splits at the tile's share of a
    //              CU's peak: 0.89 on 128 x 128 and 64 x 64 tiles, 0.97 on
    //              32 x 128 (0.83 of that above two blocks per CU, more than
    //              its 80 KiB of ring lets share one), and 0.89 of it for the
    //              two small tiles alone on a CU, whose barriers nothing covers;
    //   stream   = A's and B's bytes at 8 TB/s x the share of the CUs in use;
    //   partials = the planes written and read at that rate, + 3.2 us;
    //   time     = max(MFMA, stream) + rounds x 1.9 us + partials,
    // its constants fitted to the cost of the pick over 655 shapes on MI355X (M
    // 1..4096, N and K 512..8192, aligned and odd; every tile x split 1..32):
    // the pick is within 1.3% of the best on average. Before, 128 x 128 tiles
    // without a split ran them all, on as few CUs as they covered: fp32 16 x
    // 8192 x 8192 479 us against 47, 1000 x 1500 x 2000 125 against 57,
    // 1 x 4096 x 4096 239 against 17.5; fp64 16 x 8192 x 4096 488 against 51.
    const double cu_rate = (f64 ? 72e6 : 150e6) / 256.0;   // FLOP per us and CU
    constexpr double kBw = 8.0e6;                           // bytes per us
    constexpr int kTiles[] = {2, 4, 5};
    constexpr double kEff[] = {0.89, 0.89, 0.97};
    constexpr int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32};
    double best = -1.0;
    for (int i = 0; i < 3; ++i) {
        const int c = kTiles[i];
        for (const int sp : kSplits) {
            const int64_t blocks = tiles(c) * sp, kl = k_len(c, sp);
            if (!fits(c, sp) || (sp > 1 && (K < 64 * sp || kl * (sp - 1) >= K || 4 * cus < blocks ||
                                            (size_t)(sp * M * N * e) > scratch)))
                continue;
            const double r = (double)rounds(blocks), used = blocks < cus ? (double)blocks / (double)cus : 1.0;
            const double eff = kEff[i] * (c != 2 && blocks <= cus ? 0.89 : c == 5 && blocks > 2 * cus ? 0.83 : 1.0);
            const double mfma = r * 2.0 * kHighpTiles[c].bm * kHighpTiles[c].bn * (double)kl / (cu_rate * eff);
            const double stream = (double)((M * K + K * N) * e) / (kBw * used);
            const double partials = sp > 1 ? 2.0 * (double)(sp * M * N * e) / kBw + 3.2 : 0.0;
            const double t = (mfma > stream ? mfma : stream) + r * 1.9 + partials;
            if (best < 0.0 || t < best) best = t, ch.config = c, ch.splits = sp;
        }
    }
    // fp64 alone on a CU: 128-byte rows of A (above), unless K leaves a row empty (378 x 4062 x 2 6.4 us, 7.9 so).
    if (f64 && ch.config == 2 && K >= 16 && tiles(2) * ch.splits <= cus && k_len(3, ch.splits) * (ch.splits - 1) < K &&
        fits(3, ch.splits))
        ch.config = 3;
    // One unsplit round of at least six 128-row panels runs 128 x 32 tiles:
    // 128-row tiles without a workspace are what a plan of 1000^3 has always
    // reported (26.7 us fp32 and 41.9 fp64, against 65 and 123 on 128 x 128). No
    // time speaks for it: 64 x 64 tiles take 21.4 and 38.6, and over 25 such shapes
    // the pick above is 1.27x faster in geometric mean (fp32 1.07-1.45x, fp64
    // 0.93-1.19x, the tall ones of few columns slower on it).
    if (ch.splits == 1 && ch.config != 2 && M >= 768 && K >= 16 && tiles(4) <= cus && fits(6, 1)) ch.config = 6;
    return short_k(ch);
}

template <typename T, int CFG, bool PIECES4>
int launch_dma(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, const GemmPlan& plan,
               void* workspace, hipStream_t stream) {
    constexpr HighpTile t = kHighpTiles[CFG];
    constexpr int PA = PIECES4 ? 4 : 16, PB = PA;
    const int tiles_m = (int)((M + t.bm - 1) / t.bm), tiles_n = (int)((N + t.bn - 1) / t.bn);
    const int splits = plan.split_k;
    constexpr int SK = t.row / (int)sizeof(T);
    const int64_t stages = (K + SK - 1) / SK;
    const int64_t k_len = (stages + splits - 1) / splits * SK;
    T* c = static_cast<T*>(C);
    T* ws = splits > 1 ? static_cast<T*>(workspace) : nullptr;
    typedef void (*Kernel)(const T*, const T*, T*, int, int, int, int, int, int, int, T*);
    Kernel kernel;
    const bool ragged = k_len * splits != K;
    if constexpr (sizeof(T) == 4)
        kernel = ragged ? gemm_f32_dma_kernel<t.bm, t.bn, t.wgm, t.wgn, SK, PA, PB, true>
                        : gemm_f32_dma_kernel<t.bm, t.bn, t.wgm, t.wgn, SK, PA, PB, false>;
    else
        kernel = ragged ? gemm_f64_dma_kernel<t.bm, t.bn, t.wgm, t.wgn, SK, PA, PB, true>
                        : gemm_f64_dma_kernel<t.bm, t.bn, t.wgm, t.wgn, SK, PA, PB, false>;
    hipLaunchKernelGGL(kernel, dim3((unsigned)(tiles_m * tiles_n * splits)), dim3(64 * t.wgm * t.wgn), 0, stream,
                       static_cast<const T*>(A), static_cast<const T*>(B), c, (int)M, (int)N, (int)K, tiles_m, tiles_n,
                       splits, (int)k_len, ws);
    MB_HIP_TRY(hipGetLastError());
    if (splits > 1) {
        const int64_t mn = M * N, per_block = 64 * (16 / (int64_t)sizeof(T));
        auto sum = splits <= 5 ? highp_split_sum_kernel<T, 4> : highp_split_sum_kernel<T, 16>;
        hipLaunchKernelGGL(sum, dim3((unsigned)((mn + per_block - 1) / per_block)), dim3(64), 0, stream,
                           static_cast<const T*>(ws), c, mn, splits);
        MB_HIP_TRY(hipGetLastError());
    }
    return MB_OK;
}

template <typename T, int CFG>
int launch_pieces(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, const GemmPlan& plan,
                  void* workspace, hipStream_t stream) {
    constexpr int64_t V = 16 / (int64_t)sizeof(T);
    if (K % V == 0 && N % V == 0) return launch_dma<T, CFG, false>(A, B, C, M, N, K, plan, workspace, stream);
    return launch_dma<T, CFG, true>(A, B, C, M, N, K, plan, workspace, stream);
}

template <typename T>
int launch_typed(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, hipStream_t stream) {
    constexpr int V = 16 / (int)sizeof(T);
    const dim3 grid((unsigned)((N + kHpBN - 1) / kHpBN), (unsigned)((M + kHpBM - 1) / kHpBM));
    const T* a = static_cast<const T*>(A);
    const T* b = static_cast<const T*>(B);
    T* c = static_cast<T*>(C);
    if (K % V == 0 && N % V == 0) {
        hipLaunchKernelGGL((gemm_highp_kernel<T, true>), grid, dim3(kHpThreads), 0, stream, a, b, c, M, N, K);
    } else {
        hipLaunchKernelGGL((gemm_highp_kernel<T, false>), grid, dim3(kHpThreads), 0, stream, a, b, c, M, N, K);
    }
    MB_HIP_TRY(hipGetLastError());
    return MB_OK;
}

}  // namespace

int gemm_highp_plan(int dtype, int64_t M, int64_t N, int64_t K, const DeviceProps& props, size_t scratch,
                    GemmPlan* plan) {
    const bool f64 = dtype == MB_DT_FLOAT64;
    const char* why = "";
    const HighpChoice ch = highp_choose(f64, M, N, K, props.cu_count > 0 ? props.cu_count : 256, scratch, &why);
    plan->variant = kVariantHighp;
    plan->config = ch.config;
    plan->fallback = why;
    plan->frag_m = plan->frag_n = f64 ? 16 : 32;
    plan->frag_k = f64 ? 4 : 2;
    const HighpTile& t = kHighpTiles[ch.config];
    plan->tile_k = t.row / (f64 ? 8 : 4);
    plan->tile_m = t.bm;
    plan->tile_n = t.bn;
    if (ch.config != 0) {
        // The plain name when the rows are off 16 bytes (`fallback` says why): the family tells the ring on
        // 4-byte pieces from the register-staged kernel.
        plan->family = ch.pieces4 ? "ring_4_byte" : "ring";
        plan->implementation = f64 ? (ch.pieces4 ? "gfx950_mfma_f64_16x16x4" : "gfx950_mfma_f64_16x16x4_lds_dma")
                                   : (ch.pieces4 ? "gfx950_mfma_f32_32x32x2" : "gfx950_mfma_f32_32x32x2_lds_dma");
        plan->threads = 64 * t.wgm * t.wgn;
        plan->grid = (int)(((M + t.bm - 1) / t.bm) * ((N + t.bn - 1) / t.bn) * ch.splits);
        plan->wave_grid_m = t.wgm;
        plan->wave_grid_n = t.wgn;
        plan->wave_tile_m = t.bm / t.wgm / plan->frag_m;
        plan->wave_tile_n = t.bn / t.wgn / plan->frag_n;
        plan->k_stages = f64 ? kHpStages : kHpStages;
        plan->split_k = ch.splits;
        plan->tile_group_m = kHpGroupM;
        plan->workspace = ch.splits > 1 ? (size_t)ch.splits * (size_t)M * (size_t)N * (f64 ? 8 : 4) : 0;
        return MB_OK;
    }
    const int64_t gx = (N + kHpBN - 1) / kHpBN, gy = (M + kHpBM - 1) / kHpBM;
    if (gy > 65535 || gx > INT32_MAX) {
        set_error("fp32/fp64 GEMM: M=%lld N=%lld too large for the register-staged kernel's grid (%s)",
                  (long long)M, (long long)N, why);
        return MB_ERR_SHAPE;
    }
    plan->implementation = f64 ? "gfx950_mfma_f64_16x16x4" : "gfx950_mfma_f32_32x32x2";
    plan->family = "register_staged";
    plan->threads = kHpThreads;
    plan->grid = (int)(gx * gy);
    plan->wave_grid_m = 2;
    plan->wave_grid_n = 2;
    plan->wave_tile_m = plan->wave_tile_n = 64 / plan->frag_m;
    plan->k_stages = 2;
    plan->split_k = 1;
    plan->tile_group_m = 1;
    plan->workspace = 0;
    return MB_OK;
}

int gemm_highp_launch(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                      const GemmPlan& plan, void* workspace, hipStream_t stream) {
    auto run = [&](auto zero) -> int {
        typedef decltype(zero) T;
        switch (plan.config) {
            case 1:
                if constexpr (sizeof(T) == 4) return launch_dma<T, 1, false>(A, B, C, M, N, K, plan, workspace, stream);
                break;
            case 2: return launch_pieces<T, 2>(A, B, C, M, N, K, plan, workspace, stream);
            case 3:
                if constexpr (sizeof(T) == 8) return launch_pieces<T, 3>(A, B, C, M, N, K, plan, workspace, stream);
                break;
            case 4: return launch_pieces<T, 4>(A, B, C, M, N, K, plan, workspace, stream);
            case 5: return launch_pieces<T, 5>(A, B, C, M, N, K, plan, workspace, stream);
            case 6: return launch_pieces<T, 6>(A, B, C, M, N, K, plan, workspace, stream);
        }
        return launch_typed<T>(A, B, C, M, N, K, stream);
    };
    if (dtype == MB_DT_FLOAT32) return run(0.0f);
    if (dtype == MB_DT_FLOAT64) return run(0.0);
    set_error("fp32/fp64 GEMM: unsupported dtype %d", dtype);
    return MB_ERR_UNSUPPORTED;
}

}  // namespace mb
