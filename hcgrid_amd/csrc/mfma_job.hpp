// mfma_job.hpp -- the multi-channel job descriptor shared by the one-job
// launch (hcg_grid_mfma) and the persistent batched launch (hcg_batch_*).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "plain_tile.hpp"

namespace hcg {

constexpr int kMcCols = 64;                   // cells per workgroup
constexpr uint32_t kMcDefaultTileCols = 16;   // default block: 4 rows x 16 columns
constexpr int kMcNB = 4;                      // 16-channel blocks per wave
constexpr int kMcMaxWaves = 8;
constexpr uint32_t kMcChanPerWave = 16 * kMcNB;

// Tile plan: per tile, its ring span and the sorted range of each ring's
// union window, for up to kPlanRings rings (rings past that are searched in
// the gridding kernel itself).  Layout per tile, kPlanStride uint32:
// [r_begin, r_end, lo_0, hi_0, lo_1, hi_1, ...]; lo >= hi: no samples.
constexpr uint32_t kPlanRings = 64;
constexpr uint32_t kPlanStride = 2 + 2 * kPlanRings;
// After the ring ranges, at kPlanHeadWords: the block's 64 cell windows
// (Window, as block_cell_window gives them), then their unit vectors as
// three arrays of 64 doubles (x, y, z): the gridding kernel reads them
// instead of evaluating the cells' trigonometry and its dependent loads.
// kPlanTileWords uint32 per tile in all.
constexpr uint32_t kPlanHeadWords = (kPlanStride + 3u) & ~3u;
constexpr uint32_t kPlanWinWords = kMcCols * (uint32_t)sizeof(Window) / 4u;
constexpr uint32_t kPlanTileWords = kPlanHeadWords + kPlanWinWords + kMcCols * 3u * 2u;
static_assert(sizeof(Window) % 8 == 0 && kPlanHeadWords % 2 == 0 && kPlanTileWords % 4 == 0, "plan alignment");

// The weight form of a job (MfmaJob::kt): the kernel type, or
// kKtGaussSmall (GAUSS1D whose radius rules out the exponent's asin branch
// and the exp clamp, gauss_small_radius), or kKtGaussLean (also
// lean_weight_ok: the p.q candidate test and gauss_weight_lean of the tile
// loop).
constexpr uint32_t kKtGaussSmall = HCG_GAUSS1D + 16u;
constexpr uint32_t kKtGaussLean = HCG_GAUSS1D + 32u;

inline uint32_t mfma_weight_form(const GridParams& P, int kernel_type) {
  if (kernel_type != HCG_GAUSS1D || !gauss_small_radius(P)) return (uint32_t)kernel_type;
  return lean_weight_ok(P) ? kKtGaussLean : kKtGaussSmall;
}

// One multi-channel job: geometry, sorted channel values and outputs, with
// its launch shape (tiles of (64 >> tc_shift) x (1 << tc_shift) cells).
struct MfmaJob {
  GridParams P;
  GridBuffers B;
  const void* vs;     // sorted channel values [nchan][n_pad], BF16 or FP16
  float* cube;        // [nchan][side * side]
  float* wsum;        // [side * side] or NULL
  uint32_t kt, n_pad, nchan, dtype;  // kt: mfma_weight_form
  uint32_t tc_shift, tiles_x, ntiles, normalize;
  uint32_t* plan;     // [ntiles][kPlanTileWords], or NULL (windows and searches in the gridding kernel)
};

// The routes of a job: the MFMA contraction, or the FP64 tile loop (tiles_x
// and ntiles then count kTileCols x kTileRows tiles): one channel with four
// ring streams per tile (one_channel_streams) or one, or few channels.
enum : uint32_t { kRouteMfma = 0, kRouteOne4 = 1, kRouteOne1 = 2, kRouteFew = 3, kRoutes = 4 };
inline uint32_t route_of(const GridParams& P, uint32_t kernel_type, bool weighted, uint32_t nchan, uint32_t n) {
  if (one_channel_tiles(P, kernel_type, weighted, nchan))
    return one_channel_streams(P.side) == kOneChannelStreams ? kRouteOne4 : kRouteOne1;
  return few_channel_tiles(P, kernel_type, weighted, nchan, n) ? kRouteFew : kRouteMfma;
}

// The tile-route jobs of a batch: job `job`'s tiles are workgroups first,
// first + 1, ... of its route's launch.
struct TileRange {
  uint32_t first, job;
};
// Launches one tile route's workgroups (`blocks` of them over `nranges`
// ranges): the same tile bodies as the one-job launches, so a job's cube is
// the same alone or batched.
int launch_batch_tiles(uint32_t route, const TileRange* ranges, uint32_t nranges, uint32_t blocks,
                       const MfmaJob* jobs, hipStream_t s);

// One unit of the persistent launch: a tile of one job, one channel group.
struct MfmaItem {
  uint32_t job, tile, group, pad;
};

inline uint32_t tile_shift_of(uint32_t tile_cols) {
  return tile_cols == 8 ? 3u : tile_cols == 16 ? 4u : tile_cols == 32 ? 5u : 6u;
}

// Batch preparation in one launch: each job's channel gather (input values,
// permutation and non-finite counter here; output J.vs) and tile plan.
struct PrepJob {
  const void* in;          // the caller's channel values (layout per prep_ranges)
  const uint32_t* perm;    // [n]
  uint32_t* nonfinite;     // counter, or NULL
  uint32_t n, pad;
};
enum : uint32_t { kPrepPlan = 0, kPrepGatherCm = 1, kPrepGatherSm = 2 };
struct PrepRange {
  uint32_t first, job, kind, gx;  // first workgroup; for gathers, workgroups per channel block row
};
// The ranges of one prep launch (layouts[j]: job j's value layout, 0
// channel-major, 1 sample-major; at most 2 per job) and their workgroup
// total.
int prep_ranges(uint32_t njobs, const MfmaJob* jobs, const uint32_t* layouts, std::vector<PrepRange>& out,
                uint32_t* blocks);
int launch_batch_prep(const PrepRange* ranges, uint32_t nranges, uint32_t blocks, const PrepJob* pj,
                      const MfmaJob* jobs, hipStream_t s);

// Enqueues the tile-plan kernel of a job into J.plan (non-NULL).
int launch_mfma_plan(const MfmaJob& J, hipStream_t s);

// Grid size of the persistent kernel: CUs x resident workgroups per CU.
int mfma_batch_blocks(uint32_t chunk, uint32_t waves, uint32_t* blocks);

// Launches the persistent kernel with `blocks` workgroups of `waves` waves
// over `nitems` work items (head: a device counter that reads 0 at launch).
int launch_mfma_batch(uint32_t chunk, uint32_t waves, uint32_t blocks, const MfmaJob* jobs, const MfmaItem* items,
                      uint32_t nitems, uint32_t* head, hipStream_t s);

}  // namespace hcg
