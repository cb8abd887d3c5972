// Few-row GEMM for rows off 16 bytes (K or N not a multiple of 8, of 16 for
// fp8; M <= 64): C = A * B, fp32 accumulation, one rounding.
//
// Bound: the stream over B. Repacking it first for the LDS-DMA kernels
// (gemm_pack.hip) moves every byte three times, which few rows of A cannot
// pay for. Here B goes from HBM to the matrix cores through registers alone:
// gfx950 loads 16 bytes at any address, so a lane takes 16 bytes (8 columns of
// a 16-bit type, 16 of fp8) of 8 consecutive K rows and transposes them with
// byte permutes into one MFMA operand per column (8 K values each). MFMA j of
// a step thus multiplies columns 8 * (lane % 16) + j (16 * ... for fp8), and a
// lane's accumulators are neighbouring columns of C. No LDS and no barrier in
// the loop, and no alignment asked of A, B or C.
//
// A block covers 128 columns (256 for fp8 with M <= 16); its waves take steps
// of 32 K rows in turn and add their sums through LDS; K is split over blocks
// too, the fp32 partials going to the caller's workspace.
//
// On MI355X against the repacked path, B from HBM: bf16 53 x 5039 x 6321 49.5
// -> 32.4 us, 4 x 9933 x 3689 49.0 -> 19.0, 16 x 8191 x 8192 26.6 (5.0 TB/s),
// e4m3 4 x 13027 x 9237 73.5 -> 28.4; 60 random shapes (M 1..64, N and K
// 64..16384) 1.81x faster in geometric mean, 0.99x at worst.
#include "gemm_common.hpp"

namespace mb {
namespace {

constexpr int kStripWaves = 4;
constexpr int kStripStep = 32;      // K rows per step: four groups of 16 lanes, 8 rows each
constexpr int kStripMaxM = 64;

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef u32x4 u32x4_any __attribute__((aligned(1)));
typedef u32x2 u32x2_any __attribute__((aligned(1)));
typedef f32x4 f32x4_any __attribute__((aligned(4)));

// CPL: columns per lane.
template <int DT, int CPL>
struct Strip {   // 16-bit types
    static_assert(CPL == 8, "16 bytes per lane and row");
    static constexpr int kElem = 2;
    typedef u32x4 Row;              // CPL columns of a row of B
    typedef u32x4_any RowAny;
    typedef u32x4 Frag;             // 8 K values
    typedef u32x4_any FragAny;
    __device__ static __forceinline__ f32x4 mfma(Frag a, Frag b, f32x4 c) {
        return Mfma16<DT>::run(&a, &b, c);
    }
    // Column j's operand from the lane's 8 rows of 8 columns.
    template <int J>
    __device__ static __forceinline__ Frag column(const Row (&rows)[8]) {
        constexpr unsigned sel = (J & 1) ? 0x07060302u : 0x05040100u;
        Frag f;
#pragma unroll
        for (int p = 0; p < 4; ++p) f[p] = __builtin_amdgcn_perm(rows[2 * p + 1][J >> 1], rows[2 * p][J >> 1], sel);
        return f;
    }
};

template <int DT, int CPL>
struct StripFp8 {
    static constexpr int kElem = 1;
    typedef std::conditional_t<CPL == 16, u32x4, u32x2> Row;
    typedef std::conditional_t<CPL == 16, u32x4_any, u32x2_any> RowAny;
    typedef u32x2 Frag;
    typedef u32x2_any FragAny;
    __device__ static __forceinline__ f32x4 mfma(Frag a, Frag b, f32x4 c) {
        const long la = __builtin_bit_cast(long, a), lb = __builtin_bit_cast(long, b);
        if constexpr (DT == MB_DT_FLOAT8_E4M3FN) return __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(la, lb, c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_bf8_bf8(la, lb, c, 0, 0, 0);
    }
    template <int J>
    __device__ static __forceinline__ Frag column(const Row (&rows)[8]) {
        // Bytes J of four rows: pairs of rows first, then pairs of pairs (the
        // pairs are shared by four columns; the compiler keeps them).
        constexpr unsigned pairs = (J & 2) ? 0x07030602u : 0x05010400u, quad = (J & 1) ? 0x07060302u : 0x05040100u;
        Frag f;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const unsigned lo = __builtin_amdgcn_perm(rows[4 * h + 1][J >> 2], rows[4 * h][J >> 2], pairs);
            const unsigned hi = __builtin_amdgcn_perm(rows[4 * h + 3][J >> 2], rows[4 * h + 2][J >> 2], pairs);
            f[h] = __builtin_amdgcn_perm(hi, lo, quad);
        }
        return f;
    }
};
template <int CPL>
struct Strip<MB_DT_FLOAT8_E4M3FN, CPL> : StripFp8<MB_DT_FLOAT8_E4M3FN, CPL> {};
template <int CPL>
struct Strip<MB_DT_FLOAT8_E5M2, CPL> : StripFp8<MB_DT_FLOAT8_E5M2, CPL> {};

constexpr int strip_cols(int dtype, int fm) { return is_fp8(dtype) && fm <= 1 ? 16 : 8; }

template <int DT>
__device__ __forceinline__ unsigned pack2(float a, float b) {
    if constexpr (DT == MB_DT_FLOAT16)
        return (unsigned)__builtin_bit_cast(uint16_t, (_Float16)a) |
               (unsigned)__builtin_bit_cast(uint16_t, (_Float16)b) << 16;
    else
        return (unsigned)__builtin_bit_cast(uint16_t, (__bf16)a) | (unsigned)__builtin_bit_cast(uint16_t, (__bf16)b) << 16;
}

// FM: fragments of 16 rows of A. `steps_per_split`: steps of 32 K rows.
// Lanes whose columns would pass N take the last kCols columns instead (N is
// at least that), and rows past M row M - 1: every load is in range, and C or
// partial elements covered twice get the same value twice.
template <int DT, int FM>
__global__ void __launch_bounds__(64 * kStripWaves, 2)
gemm_strip_kernel(const unsigned char* __restrict__ A, const unsigned char* __restrict__ B,
                  uint16_t* __restrict__ C, int M, int N, int K, int groups, int splits,
                  int steps_per_split, float alpha, float* __restrict__ ws) {
    constexpr int CPL = strip_cols(DT, FM);
    typedef Strip<DT, CPL> S;
    typedef typename S::Row Row;
    typedef typename S::Frag Frag;
    constexpr int E = S::kElem, COLS = 16 * CPL, W = kStripWaves;
    const int lane = threadIdx.x & 63, l16 = lane & 15, g = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // Block b runs on XCD b % 8: each XCD takes a contiguous run of (split,
    // column group) pairs, so that neighbouring groups, whose rows of B share
    // cache lines, read them through one L2 (bf16 16 x 8191 x 8192 33.1 us
    // with groups dealt out over the XCDs, 26.6 so).
    const int total = groups * splits, xcd = (int)blockIdx.x % 8, per_xcd = total / 8, extra = total % 8;
    const int index = xcd * per_xcd + min(xcd, extra) + (int)blockIdx.x / 8;
    const int split = index / groups;
    const int group_col = (index - split * groups) * COLS;
    const int col = min(group_col + CPL * l16, N - CPL);
    const unsigned ldb = (unsigned)N * E;
    const int64_t lda = (int64_t)K * E;

    unsigned b_off[8];
#pragma unroll
    for (int r = 0; r < 8; ++r) b_off[r] = (unsigned)(8 * g + r) * ldb + (unsigned)col * E;
    const unsigned char* a_row[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) a_row[i] = A + min(16 * i + l16, M - 1) * lda + 8 * g * E;

    auto load = [&](int step, Row (&b)[8], Frag (&a)[FM]) {
        const unsigned char* base = B + (int64_t)step * kStripStep * ldb;
#pragma unroll
        for (int r = 0; r < 8; ++r) b[r] = *reinterpret_cast<const typename S::RowAny*>(base + b_off[r]);
#pragma unroll
        for (int i = 0; i < FM; ++i)
            a[i] = *reinterpret_cast<const typename S::FragAny*>(a_row[i] + (int64_t)step * kStripStep * E);
    };

    f32x4 acc[FM][CPL];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < CPL; ++j) acc[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    auto multiply = [&](const Row (&b)[8], const Frag (&a)[FM]) {
        [&]<int... J>(std::integer_sequence<int, J...>) {
            ([&] {
                const Frag f = S::template column<J>(b);
#pragma unroll
                for (int i = 0; i < FM; ++i) acc[i][J] = S::mfma(a[i], f, acc[i][J]);
            }(), ...);
        }(std::make_integer_sequence<int, CPL>{});
    };

    // Whole steps, the next one's loads in flight under this one's MFMAs.
    const int first = split * steps_per_split, whole = K / kStripStep;
    const int end = min(whole, first + steps_per_split);
    Row b0[8], b1[8];
    Frag a0[FM], a1[FM];
    int step = first + wave;
    if (step < end) load(step, b0, a0);
    for (; step < end; step += 2 * W) {
        if (step + W < end) load(step + W, b1, a1);
        multiply(b0, a0);
        if (step + W < end) {
            if (step + 2 * W < end) load(step + 2 * W, b0, a0);
            multiply(b1, a1);
        }
    }
    // The last K % 32 rows: rows of B and K values of A past K are zeros.
    if (K % kStripStep != 0 && whole >= first && whole < first + steps_per_split && (whole - first) % W == wave) {
        const int left = K - whole * kStripStep - 8 * g;        // K values of this lane's 8
        const unsigned char* base = B + (int64_t)whole * kStripStep * ldb;
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            b0[r] = Row{};
            if (r < left) b0[r] = *reinterpret_cast<const typename S::RowAny*>(base + b_off[r]);
        }
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const unsigned char* p = a_row[i] + (int64_t)whole * kStripStep * E;
            Frag f = {};
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (k < left) {
                    if constexpr (E == 2) f[k >> 1] |= (unsigned)reinterpret_cast<const uint16_t*>(p)[k] << 16 * (k & 1);
                    else f[k >> 2] |= (unsigned)p[k] << 8 * (k & 3);
                }
            a0[i] = f;
        }
        multiply(b0, a0);
    }

    // Accumulator r of acc[i][j] is C[16i + 4g + r][col + j]. The waves' sums
    // meet in LDS, 16 rows at a time, and are added in wave order.
    __shared__ __attribute__((aligned(16))) float red[W][16][COLS];
    const int orow = threadIdx.x >> 4;                          // the row and the lane columns this thread adds
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        if (i > 0) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int j = 0; j < CPL; j += 4)
                *reinterpret_cast<f32x4*>(&red[wave][4 * g + r][CPL * l16 + j]) =
                    f32x4{acc[i][j][r], acc[i][j + 1][r], acc[i][j + 2][r], acc[i][j + 3][r]};
        __syncthreads();
        const int m = 16 * i + orow;
        if (m >= M || group_col + CPL * l16 >= N) continue;
        f32x4 sum[CPL / 4];
#pragma unroll
        for (int j = 0; j < CPL / 4; ++j) {
            sum[j] = *reinterpret_cast<const f32x4*>(&red[0][orow][CPL * l16 + 4 * j]);
#pragma unroll
            for (int w = 1; w < W; ++w) sum[j] += *reinterpret_cast<const f32x4*>(&red[w][orow][CPL * l16 + 4 * j]);
        }
        if (ws != nullptr) {
            float* p = ws + ((int64_t)split * M + m) * N + col;
#pragma unroll
            for (int j = 0; j < CPL / 4; ++j) reinterpret_cast<f32x4_any*>(p)[j] = sum[j];
        } else {
            uint16_t* p = C + (int64_t)m * N + col;
#pragma unroll
            for (int j = 0; j < CPL / 8; ++j) {
                const f32x4 lo = sum[2 * j] * alpha, hi = sum[2 * j + 1] * alpha;
                reinterpret_cast<u32x4_any*>(p)[j] = (u32x4){pack2<DT>(lo[0], lo[1]), pack2<DT>(lo[2], lo[3]),
                                                             pack2<DT>(hi[0], hi[1]), pack2<DT>(hi[2], hi[3])};
            }
        }
    }
}

template <int DT>
int launch_dt(const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K, float alpha,
              const GemmPlan& plan, void* workspace, hipStream_t stream) {
    typedef void (*Kernel)(const unsigned char*, const unsigned char*, uint16_t*, int, int, int, int, int, int, float, float*);
    const Kernel kernel = M <= 16   ? gemm_strip_kernel<DT, 1>
                          : M <= 32 ? gemm_strip_kernel<DT, 2>
                          : M <= 48 ? gemm_strip_kernel<DT, 3>
                                    : gemm_strip_kernel<DT, 4>;
    const int64_t steps = (K + kStripStep - 1) / kStripStep;
    const int steps_per_split = (int)((steps + plan.split_k - 1) / plan.split_k);
    const int cols = plan.tile_n;
    float* ws = plan.split_k > 1 ? static_cast<float*>(workspace) : nullptr;
    const int groups = (int)((N + cols - 1) / cols);
    hipLaunchKernelGGL(kernel, dim3((unsigned)(groups * plan.split_k)), dim3(64 * kStripWaves), 0, stream,
                       static_cast<const unsigned char*>(A), static_cast<const unsigned char*>(B),
                       static_cast<uint16_t*>(C), (int)M, (int)N, (int)K, groups, plan.split_k, steps_per_split, alpha, ws);
    MB_HIP_TRY(hipGetLastError());
    if (plan.split_k > 1) return gemm_sum_planes(DT, ws, C, M * N, plan.split_k, alpha, stream);
    return MB_OK;
}

}  // namespace

int gemm_strip_plan(int dtype, int64_t M, int64_t N, int64_t K, const DeviceProps& props, size_t scratch,
                    GemmPlan* plan) {
    if (M < 1 || M > kStripMaxM) return MB_ERR_SHAPE;
    // Under one step of K only the tail runs, which loads A element by element:
    // three or four fragments of rows of a 16-bit type then take 5.1-6.5 us, the
    // bounds-checked kernel 4.8-5.9 (139 products, 0.76-1.32x; from one step of K
    // on 0.96-2.0x, fp8 1.0-2.4x but for one at 0.90, fewer rows 1.1-3.3x).
    if (M > 32 && K < kStripStep && !is_fp8(dtype)) return MB_ERR_SHAPE;
    const int fm = (int)(M + 15) / 16;
    const int64_t e = is_fp8(dtype) ? 1 : 2, cols = strip_cols(dtype, fm);
    // 32-bit offsets within a step (32 rows of B) and 32-bit K and column indices.
    if (N < cols || N * e > (int64_t(1) << 25) || K > (int64_t(1) << 30)) return MB_ERR_SHAPE;
    const int64_t cus = props.cu_count > 0 ? props.cu_count : 256;
    const int64_t groups = (N + 16 * cols - 1) / (16 * cols), steps = (K + kStripStep - 1) / kStripStep;
    // K splits: one block per CU (a block's loads in flight stream a CU's share
    // of HBM; 2 to 6 blocks per CU ran the same or up to 3x slower on 44 random
    // shapes, by the partials they add), or, with more column groups than that
    // leaves, the count whose last round is fullest; every wave keeps a step.
    // The partials' cost weighs each split by 1/32 of a round.
    int64_t splits = 1;
    double best = 0.0;
    for (int64_t s = 1; s == 1 || (s <= (cus / groups > 4 ? cus / groups : 4) && s <= steps / 5); ++s) {
        const double cost = (double)((groups * s + cus - 1) / cus) / (double)s * (1.0 + (double)s / 32.0);
        if (s == 1 || cost < best) best = cost, splits = s;
    }
    const int64_t force_splits = tuning(MB_TUNE_GEMM_SPLITS);
    if (force_splits >= 1) splits = force_splits < steps ? force_splits : steps;
    const size_t plane = (size_t)(M * N) * sizeof(float);
    if (splits > 1 && (size_t)splits > scratch / plane) splits = scratch / plane > 1 ? (int64_t)(scratch / plane) : 1;
    const int64_t per = (steps + splits - 1) / splits;
    splits = (steps + per - 1) / per;                           // no split without a step
    *plan = GemmPlan{};
    plan->implementation = "gfx950_mfma_generic";   // as gemm_pack.hip
    plan->family = "few_rows";
    plan->threads = 64 * kStripWaves;
    plan->grid = (int)(groups * splits);
    plan->tile_m = 16 * fm;
    plan->tile_n = (int)(16 * cols);
    plan->tile_k = kStripStep * kStripWaves;
    plan->wave_grid_m = plan->wave_grid_n = 1;
    plan->wave_tile_m = plan->tile_m / 16;
    plan->wave_tile_n = (int)cols;
    plan->frag_m = plan->frag_n = 16;
    plan->frag_k = 32;
    plan->k_stages = 2;
    plan->split_k = (int)splits;
    plan->tile_group_m = 1;
    plan->workspace = splits > 1 ? (size_t)splits * plane : 0;
    plan->variant = kVariantStrip;
    return MB_OK;
}

int gemm_strip_launch(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N, int64_t K,
                      float alpha, void* workspace, const GemmPlan& plan, hipStream_t stream) {
    switch (dtype) {
        case MB_DT_BFLOAT16: return launch_dt<MB_DT_BFLOAT16>(A, B, C, M, N, K, alpha, plan, workspace, stream);
        case MB_DT_FLOAT16: return launch_dt<MB_DT_FLOAT16>(A, B, C, M, N, K, alpha, plan, workspace, stream);
        case MB_DT_FLOAT8_E4M3FN: return launch_dt<MB_DT_FLOAT8_E4M3FN>(A, B, C, M, N, K, alpha, plan, workspace, stream);
        case MB_DT_FLOAT8_E5M2: return launch_dt<MB_DT_FLOAT8_E5M2>(A, B, C, M, N, K, alpha, plan, workspace, stream);
        default:
            set_error("few-row GEMM: unsupported dtype %d", dtype);
            return MB_ERR_UNSUPPORTED;
    }
}

}  // namespace mb
