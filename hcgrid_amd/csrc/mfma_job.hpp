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
constexpr uint32_t kMfmaInstances = 22, kRoutes = kRouteMfma + kMfmaInstances;

// The contraction kernel's forms: 16-channel blocks per wave (mfma_tile), or
// 0: mfma_wide.  A wave's registers grow with its channel blocks, so its SIMD
// holds fewer waves; more than kNarrow blocks (kNarrowGeneral with the general
// weights) take mfma_wide.  An instance is a form for each value type: first
// the lean weight's forms, then the general weights', kNbOf[kGeneral[...]].
constexpr uint32_t kWideWaves = 8;  // waves of a mfma_wide workgroup, 64 channels each
constexpr uint32_t kNbs = 8, kNbOf[kNbs] = {1, 2, 4, 6, 8, 12, 16, 0};
constexpr uint32_t kNarrow = 16, kNarrowGeneral = 4;
constexpr uint32_t kGenerals = 3, kGeneral[kGenerals] = {0, 2, 7};
static_assert(kMfmaInstances == 2 * (kNbs + kGenerals), "instances");

// The form of a job (index as instances count): the narrowest that holds its channels.
constexpr uint32_t mfma_form(uint32_t nchan, bool lean) {
  const uint32_t blocks = (nchan + 15) / 16;
  uint32_t i = 0;
  if (lean) {
    while (i < kNbs - 1 && kNbOf[i] < blocks) ++i;
    return i;
  }
  while (i < kGenerals - 1 && kNbOf[kGeneral[i]] < blocks) ++i;
  return kNbs + i;
}
constexpr uint32_t nb_of_form(uint32_t form) { return kNbOf[form < kNbs ? form : kGeneral[form - kNbs]]; }

// A lane reads whole 16-channel blocks of a value block: the rows that the
// form of a job reads, counted from the value block's first, and those that
// are there after the first row of the last sample's block (its own and the
// padding's eight blocks, hcg_channels_padded_len).  Rows past the last channel
// fill MFMA columns that nothing reads, but they have to be in the buffer.
constexpr uint64_t value_rows_read(uint32_t nchan, bool lean) {
  const uint64_t nb = nb_of_form(mfma_form(nchan, lean));
  if (nchan == 1) return nb ? (nb - 1) * 16 + 1 : 49;  // (every lane reads its block's first row)
  const uint64_t step = nb ? 16 * nb : 64;
  return (nchan + step - 1) / step * step;
}
constexpr uint64_t value_rows_held(uint32_t nchan) { return 9ull * nchan; }
// (past kNarrow blocks a form reads fewer than 64 rows beyond the last one;
// a single channel takes the lean weight on the tile loop only)
constexpr bool value_rows_ok() {
  for (uint32_t c = 1; c <= 1024; ++c)
    for (uint32_t lean = 0; lean < 2; ++lean)
      if (value_rows_read(c, lean != 0) > value_rows_held(c)) return false;
  return true;
}
static_assert(value_rows_ok(), "a form reads past the padded channel values");
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
