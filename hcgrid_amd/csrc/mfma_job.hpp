// mfma_job.hpp -- the multi-channel job descriptor shared by the one-job
// launch (hcg_grid_mfma) and the batched launches (hcg_batch_*).
#pragma once

#include <hip/hip_runtime.h>

#include <vector>

#include "plain_tile.hpp"

namespace hcg {

constexpr int kMcCols = 64;                   // cells per workgroup
constexpr uint32_t kMcDefaultTileCols = 16;   // default block: 4 rows x 16 columns
constexpr int kMcWaves = 4;                   // waves per workgroup, 16 cells each

constexpr size_t kPlanBytes = 3600;  // a block's plan (MfmaPlan), as hcg_grid_mfma_workspace_size documents

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
  void* plan;         // [ntiles] x kPlanBytes (instances with mfma_uses_plan), or NULL: set-up in the kernel
};

// The routes of a job: the MFMA contraction, or the FP64 tile loop (tiles_x
// and ntiles then count kTileCols x kTileRows tiles): one channel with four
// ring streams per tile (one_channel_streams) or one, or few channels.  In a
// batch, contraction jobs are told apart by their kernel instance too
// (kRouteMfma + mfma_instance).
enum : uint32_t { kRouteOne4 = 0, kRouteOne1 = 1, kRouteFew = 2, kRouteMfma = 3 };
constexpr uint32_t kMfmaInstances = 20, kRoutes = kRouteMfma + kMfmaInstances;
inline uint32_t route_of(const GridParams& P, uint32_t kernel_type, bool weighted, uint32_t nchan, uint32_t n) {
  if (one_channel_tiles(P, kernel_type, weighted, nchan))
    return one_channel_streams(P.side) == kOneChannelStreams ? kRouteOne4 : kRouteOne1;
  return few_channel_tiles(P, kernel_type, weighted, nchan, n) ? kRouteFew : kRouteMfma;
}

// The jobs of one route of a batch: job `job`'s tiles are workgroups first,
// first + 1, ... of its route's launch.
struct TileRange {
  uint32_t first, job;
};
// Launches one tile route's workgroups (`blocks` of them over `nranges`
// ranges): the same tile bodies as the one-job launches, so a job's cube is
// the same alone or batched.
int launch_batch_tiles(uint32_t route, const TileRange* ranges, uint32_t nranges, uint32_t blocks,
                       const MfmaJob* jobs, hipStream_t s);

// The contraction kernel's instance of a job, and the workgroups it takes (a
// multiple of 8).
uint32_t mfma_instance(const MfmaJob& J);
bool mfma_uses_plan(uint32_t instance);
uint64_t mfma_blocks(const MfmaJob& J);
// Launches one instance's workgroups.
int launch_mfma_batch(uint32_t instance, const TileRange* ranges, uint32_t nranges, uint32_t blocks,
                      const MfmaJob* jobs, hipStream_t s);

inline uint32_t tile_shift_of(uint32_t tile_cols) {
  return tile_cols == 8 ? 3u : tile_cols == 16 ? 4u : tile_cols == 32 ? 5u : 6u;
}

// Batch preparation in one launch: each job's channel gather (input values,
// permutation and non-finite counter here; output J.vs) and block plan.
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

}  // namespace hcg
