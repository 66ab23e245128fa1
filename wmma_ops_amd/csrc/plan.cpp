// Host-only GEMM planner.  Chooses the kernel family, tile and split-K partition.
//
// The reference picks a tile from gfx1151-tuned thresholds (select_optimal_tile,
// wmma_tile_selection.hpp:30-66) and has an unreachable split-K config
// (compute_config, wmma_xor_swizzle.hpp:293-332: target tiles = 4 x CUs, split capped at
// 32 and at K/256, k_per_split = ceil(K/split)).  Here the choice is made against a
// 256-CU device, in four tiers: exact shapes from the autotuned table; M <= 16 with
// K > 1024 on the streaming kernel with its split rule; every other M <= 256 and larger M
// by two launch models fitted to measured times of every plan (model_plan, tiled_plan),
// the latter with bulk + edge plans.  The result never depends on the plan beyond fp32
// summation order.
#include "plan.hpp"

#include <algorithm>
#include <cstdint>

namespace wmma_amd {

static void finish_split(int M, int N, int K, int tiles, int split, wmma_gemm_plan* p) {
    // k_per_split is a whole number of 64-deep stages so that every split but the last
    // is full; the split count is then recomputed so no split is empty.
    int kps = ceil_div(ceil_div(K, split), kBlockK) * kBlockK;
    if (kps < kBlockK) kps = kBlockK;
    split = std::max(1, ceil_div(K, kps));
    p->split_k = split;
    p->k_per_split = split > 1 ? kps : std::max(K, 0);
    p->grid = tiles * split;
    p->workspace_bytes = split > 1 ? (size_t)split * (size_t)M * (size_t)N * sizeof(float) : 0;
}

// Lower the split of p until its partial sums fit max_ws (a plan without a split needs none).
static void fit_split(int M, int N, int K, size_t max_ws, wmma_gemm_plan* p) {
    const int tiles = p->grid / std::max(p->split_k, 1);
    for (int split = p->split_k - 1; p->workspace_bytes > max_ws && split >= 1; --split)
        finish_split(M, N, K, tiles, split, p);
}

double plan_time_us(const wmma_gemm_plan& p, int M, int N, int K, int num_cus) {
    if (M <= 0 || N <= 0 || K <= 0) return 0.0;
    if (num_cus <= 0) num_cus = 256;
    const int split = std::max(p.split_k, 1);
    const double hbm_mb = (2.0 * M * K + 2.0 * K * N + 4.0 * M * N) / 1e6;
    double t = hbm_mb / kHbmMBPerUs;
    if (p.kernel == WMMA_KERNEL_TILED) {
        const TileShape& ts = kTiles[p.tile_cfg];
        const TileTime& tt = kTileTime[p.tile_cfg];
        const int64_t wgs = (int64_t)ceil_div(M, ts.bm) * ceil_div(N, ts.bn) * split;
        const int64_t rounds = ceil_div64(wgs, num_cus);
        const double stages = (split > 1 ? p.k_per_split : K) / (double)kBlockK;
        const double last = (double)(wgs - (rounds - 1) * num_cus) / num_cus;
        const double last_stage = tt.stage_lat_us + (tt.stage_us - tt.stage_lat_us) * last;
        t = std::max(t, kLaunchUs + (rounds - 1) * (tt.fixed_us + stages * tt.stage_us) +
                            tt.fixed_us + stages * last_stage);
    }
    if (split > 1) t += kReduceUs + kReduceUsPerMB * (split + 1) * 4.0 * M * N / 1e6;
    return t;
}

double model_time_us(const wmma_gemm_plan& p, int M, int N, int K, int num_cus) {
    if (num_cus <= 0) num_cus = 256;
    const int split = std::max(p.split_k, 1);
    const double kk = split > 1 ? p.k_per_split : K;
    double t;
    if (p.kernel == WMMA_KERNEL_SKINNY) {
        const int mb = M <= 16 ? 16 : 32;
        const int64_t wgs = (int64_t)ceil_div(N, kSkinnyBlockN) * split;
        const double kb = (kSkinnyBlockN + mb) * kk * 2.0 / 1000.0;
        t = (double)ceil_div64(wgs, num_cus) * (kSkinnyWgFixedUs + kb / kSkinnyKbPerUs);
    } else {
        const TileShape& ts = kTiles[p.tile_cfg];
        const int64_t wgs = (int64_t)ceil_div(M, ts.bm) * ceil_div(N, ts.bn) * split;
        const double kb = (std::min(M, ts.bm) + ts.bn) * kk * 2.0 / 1000.0;
        const double mflop = 2.0 * ts.bm * ts.bn * kk / 1e6;
        const TileRate& r = kTileRate[p.tile_cfg];
        t = (double)ceil_div64(wgs, num_cus) *
            (kWgFixedUs + std::max(kb / r.kb_per_us, mflop / r.mflop_per_us));
    }
    const double mb_io = (2.0 * M * K + 2.0 * K * N + 4.0 * M * N) / 1e6;
    t = std::max(t, mb_io / kModelHbmMBPerUs);
    if (split > 1) t += kSplitFixedUs + kPartialUsPerMB * (split + 1) * 4.0 * M * N / 1e6;
    return t;
}

// Modelled time of a skinny plan for B stored [N][K], read off a sweep of 16, 32 and 64
// columns x splits 1-8 at 44 shapes (M = 1-32, N = 256-14336, K = 1024-14336): a workgroup
// streams its operand bytes at 27 KB/us, all of them together at 5.1 TB/s from HBM and
// 7.3 TB/s from L2 (every workgroup reads all of A's K range again), and past one wave the
// busiest CU sets the pace (N = 11008: 344 workgroups of 32 columns 29 us, 688 of 16 21 us).
// A K split adds its reduction.  Its choices take 3% more time than the fastest of each
// shape.
static double skinny_nt_time_us(const wmma_gemm_plan& p, int M, int N, int K, int num_cus) {
    const int split = std::max(p.split_k, 1);
    const double kk = split > 1 ? p.k_per_split : K;
    const int64_t wgs = (int64_t)ceil_div(N, p.tile_n) * split;
    const int64_t waves = ceil_div64(wgs, num_cus);
    const double kb = (p.tile_n + std::min(M, p.tile_m)) * kk * 2.0 / 1000.0;
    const double uneven = wgs > num_cus ? (double)(waves * num_cus) / (double)wgs : 1.0;
    const double hbm_mb = (2.0 * M * K + 2.0 * K * N + 4.0 * M * N) / 1e6;
    double t = 2.0 + std::max(waves * kb / 27.0,
                              uneven * std::max(hbm_mb / 5.1, wgs * kb / 1000.0 / 7.3));
    if (split > 1) t += 3.0 + 0.5 * (split + 1) * 4.0 * M * N / 1e6;
    return t;
}

// The plan with the shortest modelled time: every tile with K splits 1, 2, 4, 8, 16 (a
// split only from K = 2048, at least 256 of K per part, and only while the workgroups fit
// one wave of the CUs), and for M <= 32 the streaming kernel with splits up to K / 256.
// Over the fitted shapes the choice cost 0.65% more time than the fastest plan of each
// shape (the previous heuristics: 14%), and 0.8% on a second sweep of 63 shapes, with four-wave
// 128x128 and 256x128 tiles; with those of now 1.5% over 80 random shapes of 17 to 256 rows.
static wmma_gemm_plan model_plan(int M, int N, int K, int num_cus, size_t max_ws,
                                 bool skinny = true) {
    wmma_gemm_plan best{};
    double best_t = 1e300;
    for (int cfg = 0; cfg < WMMA_TILE_COUNT; ++cfg) {
        const TileShape& ts = kTiles[cfg];
        const int64_t tiles = (int64_t)ceil_div(M, ts.bm) * ceil_div(N, ts.bn);
        for (int sp : {1, 2, 4, 8, 16}) {
            if (sp > 1 && (K / sp < 256 || K < 2048 || tiles * sp > num_cus)) break;
            wmma_gemm_plan c{};
            if (make_custom_plan(M, N, K, WMMA_KERNEL_TILED, cfg, sp, &c) != WMMA_OK ||
                c.workspace_bytes > max_ws)
                continue;
            const double t = model_time_us(c, M, N, K, num_cus);
            if (t < best_t * 0.999) {
                best_t = t;
                best = c;
            }
        }
    }
    if (skinny && M <= 32) {
        for (int sp : {1, 2, 3, 4, 5, 6, 8, 12, 16, 24, 32}) {
            if (sp > std::max(1, K / 256)) break;
            wmma_gemm_plan c{};
            if (make_custom_plan(M, N, K, WMMA_KERNEL_SKINNY, -1, sp, &c) != WMMA_OK ||
                c.workspace_bytes > max_ws)
                continue;
            const double t = model_time_us(c, M, N, K, num_cus);
            if (t < best_t * 0.999) {
                best_t = t;
                best = c;
            }
        }
    }
    return best;
}

// The autotuned table: exact shapes measured on a 256-CU MI355X.
#include "tuned_table.inc"

const TunedPlan* tuned_plans(int* count) {
    *count = (int)(sizeof(kTunedPlans) / sizeof(kTunedPlans[0]));
    return kTunedPlans;
}

int make_custom_plan(int M, int N, int K, int kernel, int tile_cfg, int split,
                     wmma_gemm_plan* out) {
    if (!out || M < 0 || N < 0 || K < 0 || split < 1 || split > kMaxSplitK)
        return WMMA_ERR_INVALID_ARG;
    wmma_gemm_plan p{};
    int tiles;
    if (kernel == WMMA_KERNEL_SKINNY) {
        if (M > kSkinnyMaxMWide) return WMMA_ERR_INVALID_ARG;
        p.kernel = WMMA_KERNEL_SKINNY;
        p.tile_cfg = -1;
        p.tile_m = M <= 16 ? 16 : (M <= 32 ? 32 : 64);
        p.tile_n = kSkinnyBlockN;
        tiles = ceil_div(std::max(N, 1), kSkinnyBlockN);
    } else if (kernel == WMMA_KERNEL_TILED) {
        if (tile_cfg < 0 || tile_cfg >= WMMA_TILE_COUNT) return WMMA_ERR_INVALID_ARG;
        const TileShape& t = kTiles[tile_cfg];
        p.kernel = WMMA_KERNEL_TILED;
        p.tile_cfg = tile_cfg;
        p.tile_m = t.bm;
        p.tile_n = t.bn;
        tiles = ceil_div(std::max(M, 1), t.bm) * ceil_div(std::max(N, 1), t.bn);
    } else {
        return WMMA_ERR_INVALID_ARG;
    }
    if (split > 1 && K < split * kBlockK) return WMMA_ERR_INVALID_ARG;
    finish_split(M, N, K, tiles, split, &p);
    *out = p;
    return WMMA_OK;
}

// The tiled plan with the shortest plan_time_us: every tile with K splits up to 16 (from
// K = 2048, at least 256 of K per part, at most two rounds of the CUs).
static wmma_gemm_plan tiled_plan(int M, int N, int K, int num_cus, size_t max_ws) {
    wmma_gemm_plan best{};
    double best_t = 1e300;
    // larger tiles first: they win a tie
    for (int cfg : {WMMA_TILE_256x256, WMMA_TILE_256x128, WMMA_TILE_128x128, WMMA_TILE_256x64,
                    WMMA_TILE_128x64, WMMA_TILE_64x64}) {
        const TileShape& ts = kTiles[cfg];
        const int64_t tiles = (int64_t)ceil_div(M, ts.bm) * ceil_div(N, ts.bn);
        for (int sp : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (sp > 1 && (K < 2048 || K / sp < 256 || tiles * sp > 2 * (int64_t)num_cus)) break;
            wmma_gemm_plan c{};
            if (make_custom_plan(M, N, K, WMMA_KERNEL_TILED, cfg, sp, &c) != WMMA_OK ||
                c.split_k != sp || c.workspace_bytes > max_ws)
                continue;
            const double t = plan_time_us(c, M, N, K, num_cus);
            if (t < best_t * 0.999) {
                best_t = t;
                best = c;
            }
        }
    }
    return best;
}

// Bulk + edge: when the 256x256 tiles of the shape fill W >= 1 whole waves plus part of
// another, the whole tile rows (or columns) that fit in W waves run as one launch and the
// rest as a GEMM of its own, planned on its own (it is small, so it may take a smaller
// tile or a K split and spread over the chip).  Measured on MI355X (N = K = 4096): M = 4352
// one launch of 128x128 tiles 193 us, 4096 + 256 rows 148 us; M = 5000: 209 vs 171 us;
// M = 9192: 347 vs 295 us.  Taken when the modelled time gains more than kEdgeGain asks for.
// The edge is planned and priced for the layout it runs in, as the launch plans it: the
// streaming kernels of the layouts differ in their K splits, hence in their workspaces.
static void two_part(GemmLayout layout, int M, int N, int K, int num_cus, size_t max_ws,
                     wmma_gemm_plan* p) {
    const int64_t tm = ceil_div(M, 256), tn = ceil_div(N, 256);
    const int64_t whole = tm * tn / num_cus * num_cus;  // 256x256 tiles in whole waves
    if (whole == 0) return;
    double best_t = kEdgeGain * plan_time_us(*p, M, N, K, num_cus);
    for (int dim : {WMMA_EDGE_ROWS, WMMA_EDGE_COLS}) {
        const int64_t lines = whole / (dim == WMMA_EDGE_ROWS ? tn : tm);
        const int extent = dim == WMMA_EDGE_ROWS ? M : N;
        if (lines < 1 || lines * 256 >= extent) continue;
        const int at = (int)(lines * 256);
        const int bm = dim == WMMA_EDGE_ROWS ? at : M, bn = dim == WMMA_EDGE_ROWS ? N : at;
        const int em = dim == WMMA_EDGE_ROWS ? M - at : M, en = dim == WMMA_EDGE_ROWS ? N : N - at;
        wmma_gemm_plan bulk{}, edge{};
        if (make_custom_plan(bm, bn, K, WMMA_KERNEL_TILED, WMMA_TILE_256x256, 1, &bulk) != WMMA_OK ||
            make_layout_plan(layout, em, en, K, WMMA_TILE_AUTO, num_cus, max_ws, &edge) != WMMA_OK ||
            edge.edge_dim != WMMA_EDGE_NONE)
            continue;
        const bool skinny_nt = layout == GemmLayout::NT && edge.kernel == WMMA_KERNEL_SKINNY;
        const double t = plan_time_us(bulk, bm, bn, K, num_cus) + kSecondLaunchUs +
                         (skinny_nt ? skinny_nt_time_us(edge, em, en, K, num_cus)
                                    : plan_time_us(edge, em, en, K, num_cus));
        // columns only where they are 2% better than rows: each row of their edge is a short
        // run of B and C (2560 x 14336 x 4096: 280 us by rows, 286 by columns, modelled level)
        if (t < (p->edge_dim == WMMA_EDGE_ROWS ? 0.98 : 1.0) * best_t) {
            best_t = t;
            bulk.workspace_bytes = edge.workspace_bytes;
            bulk.edge_dim = dim;
            bulk.edge_at = at;
            *p = bulk;
        }
    }
}

int make_plan(int M, int N, int K, int tile_cfg, int num_cus, wmma_gemm_plan* out) {
    return make_plan_within(M, N, K, tile_cfg, num_cus, SIZE_MAX, out);
}

int make_plan_within(int M, int N, int K, int tile_cfg, int num_cus, size_t max_ws,
                     wmma_gemm_plan* out) {
    return make_layout_plan(GemmLayout::NN, M, N, K, tile_cfg, num_cus, max_ws, out);
}

// The plan of the kernels that take every layout, and of the plain layout's streaming kernel;
// `layout` is that of a two-part plan's edge.
static int plain_plan(GemmLayout layout, int M, int N, int K, int tile_cfg, int num_cus,
                      size_t max_ws, wmma_gemm_plan* out) {
    if (!out || M < 0 || N < 0 || K < 0) return WMMA_ERR_INVALID_ARG;
    if (tile_cfg < WMMA_TILE_AUTO || tile_cfg >= WMMA_TILE_COUNT) return WMMA_ERR_INVALID_ARG;
    if (num_cus <= 0) num_cus = 256;
    wmma_gemm_plan p{};

    if (tile_cfg == WMMA_TILE_AUTO && num_cus == 256) {
        for (const TunedPlan& e : kTunedPlans)
            if (e.M == M && e.N == N && e.K == K &&
                make_custom_plan(M, N, K, e.kernel, e.tile_cfg, e.split, &p) == WMMA_OK &&
                p.workspace_bytes <= max_ws) {
                *out = p;
                return WMMA_OK;
            }
    }

    if (tile_cfg != WMMA_TILE_AUTO) {
        // Explicit tile (matmul_tiled): exactly that tile, no split.
        const TileShape& t = kTiles[tile_cfg];
        p.kernel = WMMA_KERNEL_TILED;
        p.tile_cfg = tile_cfg;
        p.tile_m = t.bm;
        p.tile_n = t.bn;
        int tiles = ceil_div(M, t.bm) * ceil_div(N, t.bn);
        finish_split(M, N, K, tiles, 1, &p);
        *out = p;
        return WMMA_OK;
    }

    if (M <= kSkinnyAutoMaxM && M > 0 && N > 0 && K > 1024) {
        // Streaming kernel (M <= 16 with K > 1024; the launch model takes shorter K, where
        // an unsplit 64x64 tile measured 10-30% faster): each workgroup owns
        // kSkinnyBlockN columns and one K range.
        // The launch lasts as long as the busiest CU, which streams ceil(W / CUs) of the
        // W = tiles x split workgroups, each 1/W of the bytes.  M <= 16: pick the split
        // that minimises ceil(W / CUs) / W over W <= 3 x CUs (measured on MI355X: a split
        // that leaves some CUs one workgroup more than the rest costs 10-25%, and beyond
        // three workgroups per CU the extra partial sums cost more than the balance gains),
        // the smaller split on a tie (fewer partial sums to write and reduce).
        p.kernel = WMMA_KERNEL_SKINNY;
        p.tile_cfg = -1;
        p.tile_m = 16;
        p.tile_n = kSkinnyBlockN;
        const int tiles = ceil_div(N, kSkinnyBlockN);
        const int smax = std::min(std::max(1, K / 256), kMaxSplitK);
        int split = 1;
        double best = 1e300;
        for (int sp = 1; sp <= smax; ++sp) {
            const int64_t w = (int64_t)tiles * sp;
            if (sp > 1 && w > 3 * (int64_t)num_cus) break;
            const double cost = (double)ceil_div64(w, num_cus) / (double)w;
            if (cost < best * 0.99) {
                best = cost;
                split = sp;
            }
        }
        finish_split(M, N, K, tiles, split, &p);
        fit_split(M, N, K, max_ws, &p);
        *out = p;
        return WMMA_OK;
    }

    if (M > 0 && N > 0 && K > 0 && M <= kModelMaxM) {
        *out = model_plan(M, N, K, num_cus, max_ws);
        return WMMA_OK;
    }

    // No output or an empty sum: any tile, the kernels write what there is to write.
    if (M <= 0 || N <= 0 || K <= 0) {
        make_custom_plan(M, N, K, WMMA_KERNEL_TILED, WMMA_TILE_64x64, 1, out);
        return WMMA_OK;
    }
    p = tiled_plan(M, N, K, num_cus, max_ws);
    if (p.split_k == 1) two_part(layout, M, N, K, num_cus, max_ws, &p);
    *out = p;
    return WMMA_OK;
}

// The skinny kernel for B stored [N][K]: columns per workgroup and K split.
static wmma_gemm_plan skinny_nt_plan(int M, int N, int K, int num_cus, size_t max_ws) {
    wmma_gemm_plan best{};
    double best_t = 1e300;
    const int mb = M <= 16 ? 1 : 2;
    for (int cols : {16, 32, 64}) {
        const int tiles = ceil_div(N, cols);
        for (int sp : {1, 2, 3, 4, 6, 8, 12, 16}) {
            if (sp > 1 && (K < sp * kSkinnyNtRound || (int64_t)tiles * sp > 4 * (int64_t)num_cus)) break;
            wmma_gemm_plan c{};
            c.kernel = WMMA_KERNEL_SKINNY;
            c.tile_cfg = -1;
            c.tile_m = 16 * mb;
            c.tile_n = cols;
            finish_split(M, N, K, tiles, sp, &c);
            if (c.workspace_bytes > max_ws) continue;
            const double t = skinny_nt_time_us(c, M, N, K, num_cus);
            if (t < best_t * 0.999) {
                best_t = t;
                best = c;
            }
        }
    }
    return best;
}

int make_layout_plan(GemmLayout layout, int M, int N, int K, int tile_cfg, int num_cus,
                     size_t max_ws, wmma_gemm_plan* out) {
    if (num_cus <= 0) num_cus = 256;
    const bool some = M > 0 && N > 0 && K > 0 && tile_cfg == WMMA_TILE_AUTO;
    if (some && layout == GemmLayout::NT && M <= kSkinnyNtMaxM) {
        *out = skinny_nt_plan(M, N, K, num_cus, max_ws);
        return WMMA_OK;
    }
    int rc = plain_plan(layout, M, N, K, tile_cfg, num_cus, max_ws, out);
    if (rc == WMMA_OK && layout != GemmLayout::NN && out->kernel == WMMA_KERNEL_SKINNY)
        *out = model_plan(M, N, K, num_cus, max_ws, /*skinny=*/false);
    return rc;
}

}  // namespace wmma_amd
