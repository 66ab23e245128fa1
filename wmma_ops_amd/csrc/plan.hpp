// Host-only GEMM planning: tile table, tile choice, split-K partition and workspace size.
// Pure C++ (no HIP), so the dispatch math is testable on a machine without a GPU.
#pragma once

#include <cstddef>
#include <cstdint>

#include "../../include/wmma_ops_amd.h"

namespace wmma_amd {

// One row of the tile menu: workgroup output tile and its wave grid.
struct TileShape {
    int bm, bn;    // workgroup tile
    int wm, wn;    // waves along M and N (wm*wn*64 threads)
};

// Tile menu indexed by WMMA_TILE_*.  Rows 0..3 keep the reference's matmul_tiled block
// shapes (wmma_gemm.hip:1500-1520); 4 and 5 are the CDNA4 large tiles.
constexpr TileShape kTiles[WMMA_TILE_COUNT] = {
    {64, 64, 2, 2},    // 0: wave tile 32x32
    {128, 64, 4, 2},   // 1: wave tile 32x32 (8 waves; 5-9% faster than 4 waves of 64x32)
    {256, 64, 4, 1},   // 2: wave tile 64x64
    {128, 128, 2, 4},  // 3: wave tile 64x32 (8 waves: 0-5% faster than 4 of 64x64 at K to 8192,
                       //    128 rows at K = 14336 unsplit or in two parts 1-4% slower)
    {256, 128, 4, 2},  // 4: wave tile 64x64 (8 waves: 3-12% faster than 4 of 128x64)
    {256, 256, 2, 4},  // 5: wave tile 128x64 (8 waves, two per SIMD)
};

constexpr int kBlockK = 64;        // K depth of one LDS stage (fp16: 128-byte rows)
constexpr int kSkinnyAutoMaxM = 16; // M at or below this (K > 1024): the streaming kernel's own rule
constexpr int kModelMaxM = 256;     // M at or below this: model_time_us picks the plan
constexpr int kSkinnyMaxMWide = 64; // the streaming kernel's limit (four 16-row blocks)
constexpr int kSkinnyBlockN = 128; // columns per skinny workgroup
constexpr int kMaxSplitK = 32;     // cap from the reference's split-K config (wmma_xor_swizzle.hpp:318)

inline int ceil_div(int a, int b) { return (a + b - 1) / b; }
inline int64_t ceil_div64(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Launch model for M <= kModelMaxM, fitted on MI355X (256 CUs) to the autotuner's timings
// of every plan (6 tiles x splits 1-16, the streaming kernel with splits 1-32) at 819
// shapes, M = 1-768, N = 512-14336, K = 512-14336, when the 128x128 and 256x128 tiles ran four
// waves; it has served M to 256 since the model below.  With the tiles of now its choices take
// 1.5% more than the fastest plan of each of 80 random shapes (M = 17-256), at worst 1.2 times
// (80 x 768 x 1664 unsplit, 12.4 us; 64x64 in seven parts 10.3).  A workgroup streams its operand bytes
// (the rows of A that exist plus the tile's columns of B, over its K range) at a per-CU
// rate, or is held by its MFMA work, whichever is longer, plus a fixed cost; the launch
// takes as many such times as it has waves of workgroups (one per CU), at least the HBM
// time of its operands, plus, with a K split, a fixed cost and the partial sums' bytes.
struct TileRate {
    double kb_per_us;     // operand bytes a workgroup streams per microsecond (KB)
    double mflop_per_us;  // its MFMA rate (MFLOP per microsecond, full tile rows)
};
constexpr TileRate kTileRate[WMMA_TILE_COUNT] = {
    {40, 2}, {40, 4}, {10, 4}, {40, 4}, {30, 3}, {35, 5}};
constexpr double kWgFixedUs = 2.0;         // per workgroup: prologue, epilogue
constexpr double kSkinnyKbPerUs = 50;      // the streaming kernel's per-workgroup rate
constexpr double kSkinnyWgFixedUs = 3.0;
constexpr double kSplitFixedUs = 2.0;      // a K split: the reduction launch
constexpr double kPartialUsPerMB = 0.5;    // and (split + 1) x M x N x 4 bytes of partial sums
constexpr double kModelHbmMBPerUs = 8.0;   // operand bytes per microsecond at most

// Modelled duration (microseconds) of a one-launch plan for M <= kModelMaxM.
double model_time_us(const wmma_gemm_plan& p, int M, int N, int K, int num_cus);

// Launch model for M > kModelMaxM, fitted on MI355X (256 CUs) to 320 shapes (M = 33-4096,
// N, K = 256-14336 over their logarithms, up to 4096^3) x 6 tiles x splits 1-16, each plan
// timed in a settled clock: 6% RMS error over the plans within twice the fastest.  A
// workgroup takes a fixed time (prologue, epilogue) and a time per 64-deep stage, which
// grows from its latency to what the chip's power and memory sustain with all CUs busy; the
// launch takes that per round of workgroups, at least its operands' bytes at 4.4 TB/s, plus,
// with a K split, the reduction launch and the partial sums' bytes.  Its choices take 2.0%
// more time than the fastest plan of each shape; the rules before (the model above to
// M = 768, full waves of tiles past it, a split only under half a wave) 5.3%, and up to 2.5
// times at long K and few tiles (1665 x 384 x 12544: 50 us unsplit, 34 us split).
struct TileTime {
    double fixed_us, stage_us, stage_lat_us;
};
constexpr TileTime kTileTime[WMMA_TILE_COUNT] = {{2.51, 0.280, 0.220}, {2.88, 0.412, 0.258},
                                                 {5.26, 0.766, 0.564}, {4.30, 0.635, 0.300},
                                                 {5.03, 1.022, 0.626}, {8.14, 1.612, 1.001}};
constexpr double kLaunchUs = 1.77;
constexpr double kHbmMBPerUs = 4.4;
constexpr double kReduceUs = 2.58;
constexpr double kReduceUsPerMB = 0.217;   // per MB of (split + 1) x M x N x 4 bytes
constexpr double kSecondLaunchUs = 3.0;    // a two-part plan's edge behind its bulk

// Modelled duration (microseconds) of one launch of tiled plan p.
double plan_time_us(const wmma_gemm_plan& p, int M, int N, int K, int num_cus);

// A two-part plan is taken when its estimate is below this fraction of the best one-launch
// plan's.  Of 60 shapes timed both ways, those modelled below it ran 4-24% faster in two
// parts (2106 x 8320 x 2552: 106 us against 138), those from there to 1 between 3% faster
// and 4% slower.
constexpr double kEdgeGain = 0.97;

// Fill `out` for a GEMM of this shape; returns WMMA_OK or WMMA_ERR_INVALID_ARG.  With
// tile_cfg == WMMA_TILE_AUTO on a 256-CU device, a shape found in the autotuned table
// (tuned_table.inc) takes the measured plan; every other shape the heuristics in
// plan.cpp, which may split it into a bulk and an edge GEMM (out->edge_dim).
int make_plan(int M, int N, int K, int tile_cfg, int num_cus, wmma_gemm_plan* out);

// A GEMM whose A or B is given transposed (A stored [K][M], or B stored [N][K]; at most one).
enum class GemmLayout { NN, TN, NT };

// Skinny kernel for B stored [N][K] (gemm_skinny_nt_kernel): its rows, column counts per
// workgroup and 8 x 128 of K that the waves of a workgroup take per round.
constexpr int kSkinnyNtMaxM = 32;
constexpr int kSkinnyNtRound = 1024;

// make_plan_within for a transposed operand.  The tiled kernel takes either operand in
// either layout and keeps the plan of the plain layout (its tiles read whole 64-byte or
// longer runs of every operand in each of them); the streaming kernel reads B row-major
// only: TN takes a tiled plan instead, NT at M <= kSkinnyNtMaxM a plan of its own kernel
// (tile_m 16 or 32, tile_n 16, 32 or 64 columns per workgroup).  The same holds for the edge
// of a two-part plan, whose workspace_bytes is what this function's plan of the edge needs.
int make_layout_plan(GemmLayout layout, int M, int N, int K, int tile_cfg, int num_cus,
                     size_t max_ws, wmma_gemm_plan* out);

// make_plan among the plans whose split-K partial sums fit max_ws bytes: a tuned-table
// entry or a split that needs more is passed over for the next choice (a plan without a
// split needs none, so there always is one).
int make_plan_within(int M, int N, int K, int tile_cfg, int num_cus, size_t max_ws,
                     wmma_gemm_plan* out);

// A plan with an explicit kernel (WMMA_KERNEL_*), tile (WMMA_TILE_*; ignored by the skinny
// kernel) and K split, completed as the planner completes its own (k_per_split a whole
// number of 64-deep stages, no empty split).  WMMA_ERR_INVALID_ARG for a combination the
// kernels cannot run.
int make_custom_plan(int M, int N, int K, int kernel, int tile_cfg, int split,
                     wmma_gemm_plan* out);

// One entry of the autotuned dispatch table: the fastest measured plan for one shape.
struct TunedPlan {
    int M, N, K;
    int kernel, tile_cfg, split;
};
// The table (generated by wmma_ops_amd/autotune.py) and its length.
const TunedPlan* tuned_plans(int* count);

}  // namespace wmma_amd
