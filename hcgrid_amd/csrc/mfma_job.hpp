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

// The weight form of a job (MfmaJob::kt): the kernel type for the general
// evaluation (which calls asin, atan2, sin and exp), or one of the forms without
// such calls: kKtGaussSmall (GAUSS1D, gauss_small_radius), kKtGaussLean (also
// lean_weight_ok: the p.q candidate test and gauss_weight_lean of the tile
// loop), and for radii below ~9.9 deg, from longer series than the tile loop's,
// kKtGaussSeries (GAUSS1D), kKtFrame2d (GAUSS2D) and kKtSincSeries
// (TAPERED_SINC, sinc_triple_ok).
constexpr uint32_t kKtGaussSmall = HCG_GAUSS1D + 16u;
constexpr uint32_t kKtGaussLean = HCG_GAUSS1D + 32u;
constexpr uint32_t kKtGaussSeries = HCG_GAUSS1D + 48u;
constexpr uint32_t kKtFrame2d = HCG_GAUSS2D + 48u;
constexpr uint32_t kKtSincSeries = HCG_TAPERED_SINC + 48u;

inline uint32_t mfma_weight_form(const GridParams& P, int kernel_type) {
  if (kernel_type == HCG_GAUSS1D && gauss_small_radius(P)) return lean_weight_ok(P) ? kKtGaussLean : kKtGaussSmall;
  if (!(P.c_hi < kSeriesMaxC2)) return (uint32_t)kernel_type;
  if (kernel_type == HCG_GAUSS1D) return kKtGaussSeries;
  if (kernel_type == HCG_GAUSS2D) return frame_finite(P) ? kKtFrame2d : (uint32_t)kernel_type;
  return sinc_triple_ok(P, P.c_hi * 1.003) ? kKtSincSeries : (uint32_t)kernel_type;
}

// How the contraction evaluates a job's weights: the lean weight (no sample
// weights), from series (one kind for each: merged, their constants alone fill
// the scalar registers), or by calls.  A call's clobbered registers cost the
// many-channel kernel 46 spills around it, and the transcendental functions
// themselves several times a series: 1M samples onto 512^2 with GAUSS2D, 64
// channels, 6.62 ms by calls and 0.78 by series; 300 channels 12.3 and 1.72.
enum : uint32_t {
  kWeightLean = 0,
  kWeightSmall = 1,   // kKtGaussSmall, and kKtGaussLean with sample weights
  kWeightSeries = 2,  // kKtGaussSeries
  kWeight2d = 3,      // kKtFrame2d
  kWeightSinc = 4,    // kKtSincSeries
  kWeightCall = 5,
  kWeightKinds = 6
};
inline uint32_t mfma_weight_kind(uint32_t kt, bool weighted) {
  switch (kt) {
    case kKtGaussLean: return weighted ? kWeightSmall : kWeightLean;
    case kKtGaussSmall: return kWeightSmall;
    case kKtGaussSeries: return kWeightSeries;
    case kKtFrame2d: return kWeight2d;
    case kKtSincSeries: return kWeightSinc;
    default: return kWeightCall;
  }
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
constexpr uint32_t kMfmaInstances = 60, kRoutes = kRouteMfma + kMfmaInstances;

// The contraction kernel's forms: 16-channel blocks per wave (mfma_tile), or
// 0: mfma_wide, for each kind of weight.  A wave's registers grow with its
// channel blocks, so its SIMD holds fewer waves; jobs of more than 16 blocks
// take mfma_wide.  An instance is a form for each value type.
constexpr uint32_t kWideWaves = 8;  // waves of a mfma_wide workgroup, 64 channels each
constexpr uint32_t kForms = 30, kFormNb[kForms] = {1, 2, 4, 6, 8, 12, 16, 0,        // kWeightLean
                                                   1, 4, 8, 16, 0, 1, 4, 16, 0,     // Small, Series
                                                   1, 4, 8, 16, 0, 1, 4, 16, 0,     // 2d, Sinc
                                                   1, 4, 16, 0};                    // Call
constexpr uint32_t kFormFirst[kWeightKinds + 1] = {0, 8, 13, 17, 22, 26, kForms};
static_assert(kMfmaInstances == 2 * kForms, "instances");

// The form of a job: the narrowest of its weight's kind that holds its channels.
constexpr uint32_t mfma_form(uint32_t nchan, uint32_t kind) {
  uint32_t i = kFormFirst[kind];
  while (i + 1 < kFormFirst[kind + 1] && 16 * kFormNb[i] < nchan) ++i;
  return i;
}
constexpr uint32_t kind_of_form(uint32_t form) {
  uint32_t k = 0;
  while (form >= kFormFirst[k + 1]) ++k;
  return k;
}

// A lane reads whole 16-channel blocks of a value block: the rows that the
// form of a job reads, counted from the value block's first, and those that
// are there after the first row of the last sample's block (its own and the
// padding's eight blocks, hcg_channels_padded_len).  Rows past the last channel
// fill MFMA columns that nothing reads, but they have to be in the buffer.
constexpr uint64_t value_rows_read(uint32_t nchan, uint32_t kind) {
  const uint64_t nb = kFormNb[mfma_form(nchan, kind)];
  if (nchan == 1) return nb ? (nb - 1) * 16 + 1 : 49;  // (every lane reads its block's first row)
  const uint64_t step = nb ? 16 * nb : 64;
  return (nchan + step - 1) / step * step;
}
constexpr uint64_t value_rows_held(uint32_t nchan) { return 9ull * nchan; }
// (mfma_wide reads fewer than 64 rows beyond the last channel's)
constexpr bool value_rows_ok() {
  for (uint32_t c = 1; c <= 1024; ++c)
    for (uint32_t kind = 0; kind < kWeightKinds; ++kind)
      if (value_rows_read(c, kind) > value_rows_held(c)) return false;
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
// One launch of an instance (launch_form), and the instances of mfma_gauss.hip
// and mfma_gauss2d_sinc.hip.
struct MfmaLaunch {
  const MfmaJob* job;
  uint32_t groups;
  const TileRange* ranges;
  uint32_t nranges;
  const MfmaJob* jobs;
  uint32_t first, count;
  hipStream_t stream;
};
void launch_gauss_forms(uint32_t instance, const MfmaLaunch& L);
void launch_gauss2d_sinc_forms(uint32_t instance, const MfmaLaunch& L);
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
