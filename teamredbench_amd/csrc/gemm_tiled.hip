// Plan and dispatch of the LDS-pipelined MFMA GEMM (gemm_tiled_kernels.hpp). Its
// kernels are compiled per input type (gemm_tiled_<type>.hip).
#include "gemm_tiled_kernels.hpp"

namespace mb {

namespace {

// Estimated time (us) of a plan: `blocks` blocks of configuration c, `stages` K
// stages each, `bytes` of A, B and C, `feed` bytes of A and B into the blocks'
// LDS, `outputs` elements of C.
//   loop     rounds of blocks, the last one weighed by how full it is (idle CUs
//            leave clock and bandwidth to the busy ones), each a block's stages
//            plus its prologue and epilogue;
//   stream   the operands from HBM, at a rate of the configuration's rows of B;
//   feed     the panels that several blocks read, from the caches;
//   splits   the reduction's launch, the partials written and read back.
// The constants fit 10596 timings on MI355X (bf16, fp16, fp8; 300 random shapes
// of M 1..8192, N and K 512..16384, every configuration, 15 split counts), the
// near-best plans of a shape weighing most: 12% rms.
struct TiledLoad {
    double bytes, feed, outputs, cus;
};

double tiled_reduce_us(int splits, double outputs) {
    constexpr double kReduce = 2.203, kPartialTBs = 5.142;
    return splits > 1 ? kReduce + splits * outputs * 8.0 / (kPartialTBs * 1e6) : 0.0;
}

// Estimates that cannot come below `limit` end early.
double tiled_estimate_us(int64_t e, int c, int64_t blocks, unsigned stages, int splits, const TiledLoad& load,
                         double limit) {
    // us per stage: 16-bit, fp8 16x16x128 (128 rows and more, an even stage count), fp8 32x32x64.
    static constexpr double kStage[3][5] = {{0.705, 0.4243, 0.2606, 0.1358, 0.0836},
                                            {0.6155, 0.3986, 0.2482, 0.0, 0.0},
                                            {0.6778, 0.4372, 0.2759, 0.1403, 0.1067}};
    static constexpr double kBlock[5] = {5.775, 2.869, 1.783, 1.158, 0.6144};      // us
    static constexpr double kLastRound[5] = {0.672, 0.5805, 0.5087, 0.7886, 0.9845};  // nearly empty, of a full one
    static constexpr double kStreamTBs[5] = {3.784, 6.407, 6.819, 5.621, 5.35};
    constexpr double kLaunch = 2.478, kFeedTBs = 21.11;
    const int cls = e == 2 ? 0 : c <= 2 && stages % 2 == 0 ? 1 : 2;
    const double all = (double)blocks / load.cus, full = std::floor(all), part = all - full;
    const double rounds = full + (part > 0.0 ? kLastRound[c] + (1.0 - kLastRound[c]) * part : 0.0);
    const double bounds[3] = {rounds * ((double)stages * kStage[cls][c] + kBlock[c]),
                              load.bytes / (kStreamTBs[c] * 1e6), load.feed / (kFeedTBs * 1e6)};
    const double fixed = kLaunch + tiled_reduce_us(splits, load.outputs);
    if (fixed + bounds[0] >= limit || fixed + bounds[1] >= limit) return limit;
    double sum = 0.0;
    for (double t : bounds) sum += t * t * t * t;   // the largest, the others showing where they come near
    return fixed + std::sqrt(std::sqrt(sum));
}

constexpr int64_t kSplitCounts[] = {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32};

// How much of the rules' estimated time another plan may take to replace it (what
// it gives: below).
constexpr double kMargin = 0.9;

// Two kinds of plans run longer than the model says:
// - a K split where the rules have none launches a second kernel: under
//   kShortPlan us the estimate must win kAddedPass us beside the margin;
// - a smaller tile with fewer splits reads the panels more often, in narrower
//   rows, for the partials it saves: the rules' partials must come to kSavedShare
//   of the panels' added bytes, and fp8 blocks, whose rows are half as long, to
//   at most kNarrowStages stages.
// Of 1300 shapes on MI355X (M 1..8192, N and K 64..16384, all four types) whose
// plan the model changes, with operands from HBM, 9 ran more than 2% slower than
// on the rules' plan (10% at most) and all 1.48x faster in geometric mean; with
// the margin alone 67 did (45% at most: e5m2 276 x 5120 x 14592 45 us on 128 x
// 256 tiles at 4 splits, 82 on 64 x 128 unsplit), at the same mean.
constexpr double kAddedPass = 1.2, kShortPlan = 8.0, kSavedShare = 0.24;
constexpr int64_t kNarrowStages = 48;

}  // namespace

// Picks the tiled configuration for a shape, or returns MB_ERR_SHAPE with
// *why set when the shape does not divide into any of them (or its buffers
// need offsets beyond the 32-bit range of buffer addressing).
int gemm_tiled_plan(int dtype, int64_t M, int64_t N, int64_t K, const DeviceProps& props,
                    Scratch scratch, GemmPlan* plan, const char** why) {
    const int64_t e = is_fp8(dtype) ? 1 : 2;
    const int64_t stage_k = kStageK / e;
    // B's rows must start on 16 bytes (N a multiple of 8, or of 16 for fp8)
    // for the 16-byte DMA loads. N a multiple of 256 takes any tile width; a
    // multiple of 128 only the 128-column tiles (configurations 2 and 3),
    // which then cover N exactly. Any other N (ragged) takes any tile width,
    // with a partial last column of tiles: its columns past N load the start
    // of B's next row (or zeros past B's end) and are not stored.
    if ((N * e) % 16 != 0) {
        *why = e == 1 ? "N is not a multiple of 16" : "N is not a multiple of 8";
        return MB_ERR_SHAPE;
    }
    const bool ragged_n = N % 128 != 0;
    const bool n128_only = !ragged_n && N % 256 != 0;
    // A's rows must start on 16 bytes too. K that is not a multiple of the
    // stage (ragged) runs over k_pad, K rounded up to whole stages: the A
    // pieces past K load zeros, and B's rows past K lie past B's end.
    if ((K * e) % 16 != 0) {
        *why = e == 1 ? "K is not a multiple of 16" : "K is not a multiple of 8";
        return MB_ERR_SHAPE;
    }
    const int64_t k_pad = (K + stage_k - 1) / stage_k * stage_k;
    // 32-bit buffer offsets: B's rows up to k_pad (plus a partial tile's 256
    // columns past the last), a 256-row A panel, and the C / partial planes.
    if ((k_pad * N + 256) * e >= (int64_t(1) << 31) || 256 * k_pad * e >= (int64_t(1) << 31) ||
        M >= (int64_t(1) << 31) || M * N >= (int64_t(1) << 31)) {
        *why = "operand offsets exceed 32-bit buffer addressing (K*N or 256*K bytes, or M*N, >= 2^31)";
        return MB_ERR_SHAPE;
    }
    // K splits. A whole-stage K splits into s parts of K / s when they are
    // whole stages. A ragged K splits into ceil(stages / s) stages each, the
    // last split running furthest past K, for any s up to the stage count
    // whose rows stay within 32-bit offsets.
    const bool ragged_k = k_pad != K;
    const int64_t stages = k_pad / stage_k;
    auto split_ok = [&](int64_t sp) {
        if (!ragged_k) return K % (stage_k * sp) == 0;
        return sp <= stages && ((stages + sp - 1) / sp * sp * stage_k * N + 256) * e < (int64_t(1) << 31);
    };
    // Any other count whose last split still holds a stage (the kernels for a
    // ragged K run it, the A pieces past K being zeros).
    auto uneven_ok = [&](int64_t sp) {
        const int64_t per = (stages + sp - 1) / sp;
        return (sp - 1) * per < stages && (per * sp * stage_k * N + 256) * e < (int64_t(1) << 31);
    };
    auto split_k_len = [&](int64_t sp) { return (stages + sp - 1) / sp * stage_k; };
    const int64_t cus = props.cu_count > 0 ? props.cu_count : 256;
    auto tiles = [&](int i) {
        return ((M + kConfigs[i].bm - 1) / kConfigs[i].bm) * ((N + kConfigs[i].bn - 1) / kConfigs[i].bn);
    };
    const int forced_cfg = (int)tuning(MB_TUNE_GEMM_TILED_CONFIG);  // -1 unless forced
    const int pinned = forced_cfg >= 0 && n128_only && forced_cfg < 2 ? 2 : forced_cfg;
    // 256 x 256 tiles once they occupy more than half the CUs. Short of a
    // full round they still beat the smaller tiles, whose twice-as-many
    // blocks need a second round: on MI355X, with A and B cycled through
    // copies that exceed the Infinity Cache, 16 shapes with 132 to 240 such
    // tiles (M 1536..4096, N 3072..8192, K 512..8192) ran 1.12-1.64x faster on
    // them than on the cost model's pick, 1.29x in geometric mean over bf16
    // and fp8 e4m3 (bf16 3072 x 3072 x 4096 74.8 against 104.6 us on 128 x 256
    // tiles at 2 splits, fp8 4096 x 3072 x 8192 74.5 against 122.4 on 128 x
    // 128), while at 128 or 64 of them (1024 x 8192, 2048 x 4096, 2048^2) they
    // ran 27-125% slower.
    int cfg = pinned >= 0 ? pinned : (!n128_only && 2 * tiles(0) > cus && M % kConfigs[0].bm == 0) ? 0 : -1;
    // Last-round fill. 128 x 256 tiles run 7-14% below 256 x 256 per FLOP on
    // MI355X, and a partly filled last round costs less than a full one (the
    // busy CUs clock up under the power limit), so the smaller tile pays only
    // when the last 256 x 256 round is at most a quarter full and there are
    // few rounds: 2560 x 8192 x 8192 ran 11-14% faster on 128 x 256 tiles,
    // 6144^3 1-5%, while 2.5- and 3.5-round shapes ran 3-15% slower.
    // Such shapes have at least one tile per CU: no K split.
    bool fill_rule = false;
    if (pinned < 0 && cfg == 0) {
        const int64_t full = tiles(0) / cus, rest = tiles(0) % cus;
        fill_rule = full <= 2 && rest > 0 && 4 * rest <= cus;
        if (fill_rule) cfg = 1;
    }
    // Problems with too few 256 x 256 tiles to fill half the GPU: the tile
    // configuration (128 x 256, 128 x 128 or 64 x 128) and the K split count s
    // (1, 2, 4 .. 32, whole stages per split) that a cost model rates fastest:
    //   blocks  = tiles * s, in ceil(blocks / CUs) rounds;
    //   MFMA    = rounds x one block's 2 * BM * BN * K / s FLOP at a per-CU
    //             rate of the configuration (3.70 / 2.87 / 1.99 TFLOP/s for
    //             16-bit inputs, twice that for fp8);
    //   stream  = the A and B bytes at 6.26 TB/s times the fraction of the
    //             CUs the blocks occupy (each block keeps a fixed number of
    //             loads in flight, so too few blocks leave HBM idle);
    //   partials (s > 1): the fp32 partials written and read back at the
    //             same rate, plus 4.72 us for the reduction pass;
    //   time    = max(MFMA, stream) + rounds x 2.71 us (prologue, epilogue)
    //             + partials.
    // The constants minimise the measured cost of the model's pick, not its
    // timing error (they are effective figures, not the part's rates), over
    // 906 timings on MI355X (bf16, fp16, fp8 e4m3; 61 shapes, M = 8..4096,
    // N = 256..16384, K = 768..16384; every configuration x split 1..16),
    // with B cycled through copies that exceed the 256 MB Infinity Cache:
    // the pick is within 0.65% of the measured best in geometric mean (11%
    // at worst), against 1.8% (24%) for constants fitted to the timings
    // themselves. On 48 further shapes where the two sets pick differently
    // (splits up to 32), these picks ran 7.6% faster in geometric mean
    // (0.89x - 1.39x): fp8 128 x 14336 x 8192 37.7 us on 128 x 128 tiles at
    // 2 splits against 43.5 on 64 x 128 at 1, fp8 8 x 1024 x 2048 7.9 us at 32
    // splits against 11.0 at 1, bf16 32 x 14336 x 8192 55.5 us at 4 splits
    // against 49.4 at 2.
    int splits = 1;
    if (!fill_rule && (cfg < 0 || kConfigs[cfg].bm <= 128)) {
        // kRate[4] (64 x 64 tiles) only prices the split count when that configuration is forced.
        constexpr double kRate[5] = {0.0, 3.70e12, 2.87e12, 1.99e12, 1.20e12}, kBw = 6.26e12, kRound = 2.71e-6,
                         kReduce = 4.72e-6;
        int cands[3] = {1, 2, 3}, n_cands = 3, first = 0;
        if (cfg >= 0) cands[0] = cfg, n_cands = 1;
        else if (n128_only) first = 1;
        double best = -1.0;
        for (int ci = first; ci < n_cands; ++ci) {
            const int c = cands[ci];
            const double bm = kConfigs[c].bm, bn = kConfigs[c].bn;
            const double rate = kRate[c] * (e == 1 ? 2.0 : 1.0);
            for (int64_t sp = 1; sp <= 32; sp *= 2) {
                if (!split_ok(sp)) continue;
                const double blocks = (double)(tiles(c) * sp);
                const double rounds = std::ceil(blocks / (double)cus);
                const double mfma = rounds * 2.0 * bm * bn * (double)split_k_len(sp) / rate;
                const double occupancy = blocks < (double)cus ? blocks / (double)cus : 1.0;
                const double stream = (double)((K * N + M * K) * e) / (kBw * occupancy);
                const double partials = sp > 1 ? 2.0 * (double)sp * (double)M * (double)N * 4.0 / kBw + kReduce : 0.0;
                const double t = (mfma > stream ? mfma : stream) + rounds * kRound + partials;
                if (best < 0.0 || t < best) {
                    best = t;
                    cfg = c;
                    splits = (int)sp;
                }
            }
        }
    }
    // 64 x 64 tiles for narrow problems: a plan of 64 x 128 tiles with N at
    // most 2048 takes them with half its K splits (the same block count, each
    // block half the columns over twice the K: one reduction pass less, or
    // none), or, unsplit, when twice its blocks still fit one round. On
    // MI355X, B from HBM, 61 such shapes (M 8..1024, N 256..2048, K
    // 512..16384, bf16 and fp8 e4m3) ran 1.128x faster in geometric mean
    // (0.96x - 1.33x): 1024^3 bf16 6.3 against 7.6 us, 1024 x 1024 x 2048 7.8
    // against 14.0 (no split instead of two), 128 x 1024 x 8192 12.8 against
    // 14.6. Wider N keeps 64 x 128 tiles: their 256-byte B rows stream HBM
    // better (16 x 8192 x 8192 fp8 19.7 against 22.1 us on 64 x 64).
    if (pinned < 0 && cfg == 3 && N <= 2048) {
        const int s4 = splits > 1 ? splits / 2 : 1;
        if (splits > 1 || tiles(4) <= cus) {
            cfg = 4;
            splits = s4;
        }
    }
    // Those rules look at powers of two that divide K into whole stages, and at
    // 256 x 256 tiles for whole panels of M only. A model of the measured times
    // over every configuration and split count replaces their pick where it
    // expects another to take less than kMargin of the time. Rating them costs the
    // host 0.1-1.0 us a call (16 x 8192 x 8192 0.24 us for the whole plan, 0.26 by
    // the rules alone; 1024^3 0.32 and 0.22, 9 x 2512 x 15136 1.0 and 0.09), beside
    // about 2.5 us for a launch.
    const int64_t force_splits = tuning(MB_TUNE_GEMM_SPLITS);
    // A plan that fills the CUs exactly once stays (fp8 128 x 8192 x 8192: 25.2 us
    // on 128 x 128 tiles at 4 splits, 28.0 on 64 x 128 at 2).
    const int64_t rules_blocks = tiles(cfg) * splits;
    // (An unsplit pick stays with a workspace off 16 bytes, which it leaves alone.)
    if (pinned < 0 && force_splits < 1 && !fill_rule && cfg > 0 && (splits == 1 ? scratch.on_16 : rules_blocks != cus)) {
        const double a_bytes = (double)(M * K * e), b_bytes = (double)(K * N * e), outputs = (double)(M * N);
        auto estimate = [&](int c, int64_t tiles_m, int64_t tiles_n, int64_t sp, double limit) {
            const TiledLoad load{a_bytes + b_bytes + 2.0 * outputs, (double)tiles_m * b_bytes + (double)tiles_n * a_bytes,
                                 outputs, (double)cus};
            return tiled_estimate_us(e, c, tiles_m * tiles_n * sp, (unsigned)(stages + sp - 1) / (unsigned)sp, (int)sp, load,
                                     limit);
        };
        auto partials = [&](int64_t sp) { return sp > 1 ? (size_t)(sp * M * N) * sizeof(float) : 0; };
        int best_cfg = cfg;
        int64_t best_splits = splits;
        const int64_t rules_tm = (M + kConfigs[cfg].bm - 1) / kConfigs[cfg].bm;
        const int64_t rules_tn = (N + kConfigs[cfg].bn - 1) / kConfigs[cfg].bn;
        const double rules_us = estimate(cfg, rules_tm, rules_tn, splits, 1e30);
        const double added_pass = splits == 1 && rules_us < kShortPlan ? kAddedPass : 0.0;
        double best = kMargin * rules_us;
        for (int c = n128_only ? 2 : 0; c < 5; ++c) {
            // fp8 rows of 64 bytes stream a wide B poorly: e5m2 7 x 13568 x 2560
            // 11.8 us unsplit on 64 x 64 tiles, 9.7 on 64 x 128 at 2 splits; so do
            // rows of 128 where the rules take 256: e5m2 284 x 12272 x 4144 34.8 us
            // on 128 x 256 tiles, 42.6 on 64 x 128.
            if (e == 1 && N > 8192 && (c == 4 || (c == 3 && kConfigs[cfg].bn == 256))) continue;
            const int64_t tm = (M + kConfigs[c].bm - 1) / kConfigs[c].bm, tn = (N + kConfigs[c].bn - 1) / kConfigs[c].bn;
            for (int64_t sp : kSplitCounts) {
                // More splits only add partials: past a round of blocks, or once
                // the reduction alone takes what is left, no more of them.
                if (sp > 1 && (c == 0 || 4 * tm * tn * sp > 5 * cus || tiled_reduce_us((int)sp, outputs) >= best)) break;
                // Fewer blocks than 0.7 of the CUs keep too little in flight: e4m3
                // 11 x 16064 x 3968 18.5 us on 126 blocks, 14.8 on 252.
                const int64_t blocks = tm * tn * sp;
                if (10 * blocks < 7 * cus && blocks < rules_blocks) continue;
                if (sp < splits && kConfigs[c].bm * kConfigs[c].bn < kConfigs[cfg].bm * kConfigs[cfg].bn) {
                    const double added_feed = (double)(tm - rules_tm) * b_bytes + (double)(tn - rules_tn) * a_bytes;
                    if ((double)splits * outputs * 4.0 < kSavedShare * added_feed ||
                        (e == 1 && stages > kNarrowStages * sp))
                        continue;
                }
                const double added = sp > 1 ? added_pass : 0.0;
                const double t = estimate(c, tm, tn, sp, best - added);
                if (t < best - added && uneven_ok(sp)) best = t + added, best_cfg = c, best_splits = sp;
            }
        }
        // A call whose workspace would not hold the new plan's partials keeps
        // the rules' plan; one that lacks a workspace the rules' plan needs is
        // served from the library's own array, or refused, under either.
        const size_t held = partials(splits), own = (size_t)MB_NOALLOC_SCRATCH_BYTES;
        const size_t limit = scratch.bytes < held && held <= own ? own : scratch.bytes;
        if (partials(best_splits) <= limit) cfg = best_cfg, splits = (int)best_splits;
    }
    if (force_splits >= 1 && (split_ok(force_splits) || uneven_ok(force_splits))) splits = (int)force_splits;
    if (kConfigs[cfg].bm > 128) splits = 1;   // the 256-row kernels carry no split path
    if (tiles(cfg) * splits > INT32_MAX) {
        *why = "more than 2^31 tiles";
        return MB_ERR_SHAPE;
    }
    const TiledConfig& c = kConfigs[cfg];
    // fp8 takes v_mfma_scale_f32_16x16x128_f8f6f4 on tiles of 128 rows or
    // more when every split holds an even number of stages (one MFMA spans
    // two): on MI355X 2.3-4.2% faster than the 32x32x64 kernel at 4096^3 -
    // 16384^3 (256 x 256), 2.6-3.9% on 128 x 256 tiles, and on 128 x 128 tiles
    // 2-5.5% faster on 8 of 10 shapes (2048^3 13.5 against 14.3 us, e4m3 and
    // e5m2 alike), equal at 128 x 8192 x 8192 and 1% slower at 1024 x 1024 x
    // 4096. The 64 x 128 tiles (two fragment rows per wave) keep 32x32x64:
    // within 0.6% either way there. The gemm_fp8_mfma override (16 or 32)
    // forces either.
    const int64_t mfma_force = tuning(MB_TUNE_GEMM_FP8_MFMA);
    const bool mi16 = e == 1 && (split_k_len(splits) / stage_k) % 2 == 0 && c.bn >= 128 &&
                      (mfma_force == 16 || (mfma_force != 32 && c.bm >= 128));
    const int frag = mi16 ? 16 : 32;
    plan->implementation = mi16 ? "gfx950_mfma16_lds_dma" : "gfx950_mfma32_lds_dma";
    plan->family = "tiled";
    plan->threads = 64 * c.wgm * c.wgn;
    plan->grid = (int)(tiles(cfg) * splits);
    plan->tile_m = c.bm;
    plan->tile_n = c.bn;
    plan->tile_k = (int)stage_k;
    plan->wave_grid_m = c.wgm;
    plan->wave_grid_n = c.wgn;
    plan->wave_tile_m = c.bm / c.wgm / frag;
    plan->wave_tile_n = c.bn / c.wgn / frag;
    plan->frag_m = frag;
    plan->frag_n = frag;
    plan->frag_k = mi16 ? 128 : is_fp8(dtype) ? 64 : 16;
    plan->k_stages = c.nb;
    plan->split_k = splits;
    plan->tile_group_m = c.group_m;
    plan->workspace = splits > 1 ? (size_t)splits * (size_t)M * (size_t)N * sizeof(float) : 0;
    plan->variant = kVariantTiled;
    plan->config = cfg;
    return MB_OK;
}

int gemm_tiled_launch(int dtype, const void* A, const void* B, void* C, int64_t M, int64_t N,
                      int64_t K, float alpha, void* workspace, const GemmPlan& plan, hipStream_t stream) {
    switch (dtype) {
        case MB_DT_BFLOAT16: return gemm_tiled_launch_bf16(plan, A, B, C, M, N, K, alpha, workspace, stream);
        case MB_DT_FLOAT16: return gemm_tiled_launch_f16(plan, A, B, C, M, N, K, alpha, workspace, stream);
        case MB_DT_FLOAT8_E4M3FN: return gemm_tiled_launch_e4m3(plan, A, B, C, M, N, K, alpha, workspace, stream);
        case MB_DT_FLOAT8_E5M2: return gemm_tiled_launch_e5m2(plan, A, B, C, M, N, K, alpha, workspace, stream);
        default:
            set_error("tiled GEMM: unsupported dtype %d", dtype);
            return MB_ERR_UNSUPPORTED;
    }
}

}  // namespace mb
