// grid_plain.hip -- the single-channel gather-convolution on gfx950.
//
// Replaces the `hcgrid` kernel (HCGrid/gridding.cu:277-403).  Selection is
// the reference's, per window anchor a (first cell of a `factor` group):
//   rings r in [uring(a), dring(a)], r != firstring (the reference's
//   start_int-1 wrap skips the first used ring, gridding.cu:326,363-367),
//   sorted samples with lpix_r(a) <= key <= rpix_r(a) (whole ring when the
//   anchor colatitude is <= 20 or >= 160 deg, gridding.cu:341-356),
//   great-circle distance from the cell itself < sphere_radius.
// Sums are FP64.  The order is the reference's (ring ascending, sorted index
// ascending) within each of a cell's partial sums: four lane phases, in each of
// the ring streams that share a tile of a small map (plain_tile.hpp).
//
// What differs from the reference's arithmetic (not its selection):
//  * ring windows use the per-ring cos/sin table built with the LUT instead
//    of recomputing pix2ang + cos per cell and ring (same values);
//  * the end-of-window test reads the sorted key instead of recomputing
//    ang2pix for every candidate (gridding.cu:373; equal by construction);
//  * distance: h = |p - q|^2 / 4 = sin^2(d/2) from precomputed unit vectors
//    (the haversine quantity of helpers.cu:128-130, exact in real
//    arithmetic, ~1e-12 relative in FP64); for GAUSS1D at radii with
//    c2 threshold >= 1e-7 (dot_distance_ok) c2 = 2 - 2 p.q instead, which
//    tests a candidate in four FP64 operations rather than seven and is
//    good to ~1.2e-15 absolute (weights to ~5e-8 relative at worst).  Pairs
//    within the guard band of the radius threshold (1e-9 relative + 4e-15
//    absolute) are decided with the reference's haversine formula itself,
//    so selection is exact in both forms; d^2 for the Gaussian comes from the series
//    4 asin^2(sqrt h) = 4 (h + h^2/3 + 8h^3/45 + 4h^4/35 + ...), exact to
//    <1e-17 relative for h < 1e-4 (radius < 1.1 deg), asin otherwise.
//
// Work decomposition: one wave per 16 x 4 tile of cells, or several waves
// sharing a tile's rings on small maps (plain_tile.hpp).
#include <hip/hip_runtime.h>

#include "common.hpp"
#include "expneg.hpp"
#include "healpix.hpp"

#include "mfma_job.hpp"
#include "plain_tile.hpp"

namespace hcg {

// The tile of workgroup b.  XCD-aware order: workgroups are dealt
// round-robin over the 8 XCDs, so block b runs on XCD b % 8; give each XCD a
// contiguous run of tiles so neighbouring tiles (which stage overlapping
// samples) share its L2.
__device__ inline uint32_t xcd_tile(uint32_t b, uint32_t ntiles) {
  return (ntiles & 7u) == 0 ? (b & 7u) * (ntiles >> 3) + (b >> 3) : b;
}

// WMODE: grid_tile.  S waves per tile, each walking every S-th non-empty
// ring; their sums are added in stream order.
// One-wave tiles have 168 registers at three waves per SIMD: at four (128) some
// 70 spill around the sample loop, 3.7 GB of scratch writes on the 20M-sample
// map (a pass 4.39 -> 4.28 ms; 250k samples onto 400^2 175 -> 160 us).  Tiles
// of several waves, on maps that fill the chip less, are the slower for it
// (5 sigma beam onto 347^2 1.17 -> 1.35 ms).
template <int KT, bool HAS_W, int WMODE, uint32_t S, int ROWS>
__global__ void __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(S == 1 ? 3 : 4)))
    k_grid_tiles(GridParams P, GridBuffers B, uint32_t tiles_x, uint32_t tiles_y, uint32_t first) {
  constexpr uint32_t kCap = S >= 16 ? 128 : S >= 4 ? 192 : kStageCap;
  constexpr size_t kSlice = kCap * ((HAS_W ? 5 : 4) * sizeof(double) + sizeof(uint32_t));
  __shared__ __attribute__((aligned(16))) char lds[S * kSlice];
  __shared__ double s_exp[64];
  const uint32_t wave = S > 1 ? threadIdx.x >> 6 : 0u;
  if (wave == 0) exp_table_load(s_exp);
  if constexpr (S > 1)
    __syncthreads();
  else
    tile_sync();
  if (B.meta->usedrings == 0) return;  // uniform: no samples, nothing to add
  const uint32_t tile = xcd_tile(first + blockIdx.x, tiles_x * tiles_y);
  TileSums<0> t;
  if constexpr (S == 1) {
    grid_tile<KT, HAS_W, WMODE, false, 0, kCap, ROWS>(P, B, tile, tiles_x, lds, s_exp, TileOut{}, RingStream{0, 1},
                                                      t);
  } else {
    __shared__ TileShared sh;
    grid_tile<KT, HAS_W, WMODE, false, 0, kCap, ROWS, true>(P, B, tile, tiles_x, lds + wave * kSlice, s_exp,
                                                            TileOut{}, RingStream{wave, S}, t, &sh);
    static_assert(kSlice >= 64 * 2 * sizeof(double), "a wave's sums fit its slice");
    const uint32_t lane = __lane_id();
    tile_sync();
    double* red = reinterpret_cast<double*>(lds + wave * kSlice);
    red[lane] = t.d;
    red[64 + lane] = t.w;
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (uint32_t q = 1; q < S; ++q) {
      const double* o = reinterpret_cast<const double*>(lds + q * kSlice);
      t.d += o[lane];
      t.w += o[64 + lane];
    }
  }
  uint32_t cell;
  if (tile_cell<ROWS>(P.side, tile, tiles_x, cell)) {
    B.dc[cell] += t.d;
    B.wc[cell] += t.w;
  }
}

// A one-channel job of the multi-channel entry points on the tile path:
// 16-bit values in, FP32 cube and weight sum out; one tile per workgroup of
// S waves, one partial ring stream per wave (one_channel_tile).
template <uint32_t S, int WMODE>
__global__ void __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(4)))
    k_grid_tiles_1ch(GridParams P, GridBuffers B, TileOut O, uint32_t tiles_x, uint32_t tiles_y, uint32_t first) {
  __shared__ __attribute__((aligned(16))) char lds[one_channel_lds_bytes(S, S)];
  __shared__ double s_exp[64];
  if (threadIdx.x < 64) exp_table_load(s_exp);
  __syncthreads();
  one_channel_tile<WMODE>(P, B, O, xcd_tile(first + blockIdx.x, tiles_x * tiles_y), tiles_x, S, S, lds, s_exp);
}

// A few-channel job of the multi-channel entry points on the tile path: one
// wave per tile (few_channel_tile_body).  Two waves per SIMD: with its sums and
// values of eight channels the sample loop takes some 200 registers (a grid
// pass of 300k samples x 2 onto 2048^2 655 us so, 732 at three waves, 2156 at
// four, where it spills; 20k x 8 onto 512^2 48, 68 and 146 us).
constexpr int kFewWaves = 2;
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(kFewWaves)))
    k_grid_tiles_few(GridParams P, GridBuffers B, TileOut O, uint32_t tiles_x, uint32_t tiles_y, uint32_t first) {
  __shared__ __attribute__((aligned(16))) char lds[kFewTileLdsBytes];
  __shared__ double s_exp[64];
  exp_table_load(s_exp);
  tile_sync();
  few_channel_tile_body(P, B, O, xcd_tile(first + blockIdx.x, tiles_x * tiles_y), tiles_x, lds, s_exp);
}

int launch_tiles_few_channels(const GridParams& P, const GridBuffers& B, const TileOut& O, hipStream_t s) {
  const uint32_t tiles_x = tile_cols_of(P.side);
  const uint32_t tiles_y = (P.side + kTileRows - 1) / kTileRows;
  if ((uint64_t)tiles_x * tiles_y == 0) return HCG_OK;
  launch_runs((uint64_t)tiles_x * tiles_y, 64, [&](uint32_t first, uint32_t count) {
    k_grid_tiles_few<<<count, 64, 0, s>>>(P, B, O, tiles_x, tiles_y, first);
  });
  HCG_CHECK_LAUNCH("k_grid_tiles_few");
  return HCG_OK;
}

// The tile-route jobs of a batch, one route per launch: a workgroup finds its
// job by binary search over the range starts and works one tile of it.
template <uint32_t ROUTE>
__global__ void __launch_bounds__(ROUTE == kRouteOne4 ? 64 * kOneChannelStreams : 64)
    __attribute__((amdgpu_waves_per_eu(ROUTE == kRouteFew ? kFewWaves : 4)))
    k_batch_tiles(const TileRange* __restrict__ ranges, uint32_t nranges, const MfmaJob* __restrict__ jobs,
                  uint32_t first) {
  constexpr uint32_t S = ROUTE == kRouteOne4 ? kOneChannelStreams : 1;
  __shared__ __attribute__((aligned(16))) char lds[ROUTE == kRouteFew ? kFewTileLdsBytes : one_channel_lds_bytes(S, S)];
  __shared__ double s_exp[64];
  if (threadIdx.x < 64) exp_table_load(s_exp);
  if constexpr (S > 1)
    __syncthreads();
  else
    tile_sync();
  const uint32_t block = first + blockIdx.x;
  uint32_t lo = 0, hi = nranges;  // last range with first <= block
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (ranges[mid].first <= block)
      lo = mid;
    else
      hi = mid;
  }
  const MfmaJob& J = jobs[ranges[lo].job];
  const uint32_t tile = block - ranges[lo].first;
  const TileOut O{static_cast<const uint16_t*>(J.vs), J.cube, J.wsum, J.dtype == HCG_DTYPE_BF16 ? 1u : 0u,
                  J.normalize, J.nchan};
  if constexpr (ROUTE == kRouteFew)
    few_channel_tile_body(J.P, J.B, O, tile, J.tiles_x, lds, s_exp);
  else if (J.kt == kKtGaussLean)  // uniform; as launch_tiles_one_channel chooses
    one_channel_tile<3>(J.P, J.B, O, tile, J.tiles_x, S, S, lds, s_exp);
  else
    one_channel_tile<2>(J.P, J.B, O, tile, J.tiles_x, S, S, lds, s_exp);
}

int launch_batch_tiles(uint32_t route, const TileRange* ranges, uint32_t nranges, uint32_t blocks,
                       const MfmaJob* jobs, hipStream_t s) {
  if (nranges == 0 || blocks == 0) return HCG_OK;
  constexpr uint32_t kThreads4 = 64 * kOneChannelStreams;
  launch_runs(blocks, route == kRouteOne4 ? kThreads4 : 64, [&](uint32_t first, uint32_t count) {
    if (route == kRouteOne4)
      k_batch_tiles<kRouteOne4><<<count, kThreads4, 0, s>>>(ranges, nranges, jobs, first);
    else if (route == kRouteOne1)
      k_batch_tiles<kRouteOne1><<<count, 64, 0, s>>>(ranges, nranges, jobs, first);
    else
      k_batch_tiles<kRouteFew><<<count, 64, 0, s>>>(ranges, nranges, jobs, first);
  });
  HCG_CHECK_LAUNCH("k_batch_tiles");
  return HCG_OK;
}

template <int WMODE>
static void launch_1ch(const GridParams& P, const GridBuffers& B, const TileOut& O, uint32_t tiles_x,
                       uint32_t tiles_y, hipStream_t s) {
  const bool several = one_channel_streams(P.side) == kOneChannelStreams;
  const uint32_t threads = several ? 64 * kOneChannelStreams : 64;
  launch_runs((uint64_t)tiles_x * tiles_y, threads, [&](uint32_t first, uint32_t count) {
    if (several)
      k_grid_tiles_1ch<kOneChannelStreams, WMODE><<<count, threads, 0, s>>>(P, B, O, tiles_x, tiles_y, first);
    else
      k_grid_tiles_1ch<1, WMODE><<<count, threads, 0, s>>>(P, B, O, tiles_x, tiles_y, first);
  });
}

int launch_tiles_one_channel(const GridParams& P, const GridBuffers& B, const TileOut& O, hipStream_t s) {
  const uint32_t tiles_x = tile_cols_of(P.side);
  const uint32_t tiles_y = (P.side + kTileRows - 1) / kTileRows;
  if ((uint64_t)tiles_x * tiles_y == 0) return HCG_OK;
  if (lean_weight_ok(P))
    launch_1ch<3>(P, B, O, tiles_x, tiles_y, s);
  else
    launch_1ch<2>(P, B, O, tiles_x, tiles_y, s);
  HCG_CHECK_LAUNCH("k_grid_tiles_1ch");
  return HCG_OK;
}

template <int KT, bool HAS_W, int WMODE, uint32_t S, int ROWS>
static void launch_tiles_as(const GridParams& P, const GridBuffers& B, hipStream_t s) {
  const uint32_t tiles_x = tile_cols_of(P.side), tiles_y = (P.side + ROWS - 1) / ROWS;
  launch_runs((uint64_t)tiles_x * tiles_y, 64 * S, [&](uint32_t first, uint32_t count) {
    k_grid_tiles<KT, HAS_W, WMODE, S, ROWS><<<count, 64 * S, 0, s>>>(P, B, tiles_x, tiles_y, first);
  });
}

// Rows of a tile and waves per tile (each walking its share of the rings) by
// the map's size, so that the chip is filled: 256 CUs hold about 4096 waves.
// One wave per tile needs the fewest set-ups (a tile's windows and ring
// ranges), but a map of few tiles then takes as long as one tile.  Grid
// kernel, us, as (waves, rows): 20^2 map (1, 4) 311, (16, 1) 28; 64^2 433,
// 52; 128^2 (1, 4) 192, (4, 1) 55, (16, 1) 89; 256^2 (1, 4) 175, (4, 1) 148,
// (4, 4) 92; 347^2 at 390 samples per 16 x 4 cells (1, 4) 1924, (4, 4) 1164;
// 400^2 at 100 (1, 4) 106, (4, 4) 139; 512^2 at 980 (1, 4) 739, (4, 4) 921.
template <int KT, bool HAS_W, int WMODE>
static void launch_tiles(const GridParams& P, const GridBuffers& B, uint32_t n, hipStream_t s) {
  // GAUSS2D's tangent frames take twelve registers a row: two rows
  constexpr int R = KT == HCG_GAUSS2D && WMODE >= 4 ? 2 : 4;
  const uint32_t tiles = tile_count_of(P.side);
  if (tiles >= 4096 || (tiles >= 2048 && n < 256 * tiles))
    launch_tiles_as<KT, HAS_W, WMODE, 1, R>(P, B, s);
  else if (tiles >= 512)
    launch_tiles_as<KT, HAS_W, WMODE, 4, R>(P, B, s);
  else if (tiles >= 128)
    launch_tiles_as<KT, HAS_W, WMODE, 4, 1>(P, B, s);
  else
    launch_tiles_as<KT, HAS_W, WMODE, 16, 1>(P, B, s);
}

template <int KT, bool HAS_W>
int launch_grid(const GridParams& P, const GridBuffers& B, uint32_t n, hipStream_t s) {
  // GAUSS1D with a radius whose pairs all take the exponent's series branch
  // (and stay clear of the exp clamp): the forms without either check
  if constexpr (KT == HCG_GAUSS1D) {
    if (lean_weight_ok(P))
      launch_tiles<KT, HAS_W, 3>(P, B, n, s);
    else if (gauss_tiny_radius(P))
      launch_tiles<KT, HAS_W, 2>(P, B, n, s);
    else if (gauss_small_radius(P))
      launch_tiles<KT, HAS_W, 1>(P, B, n, s);
    else
      launch_tiles<KT, HAS_W, 0>(P, B, n, s);
  } else if (frame_weight_ok(P, KT)) {
    if (KT != HCG_GAUSS2D || frame_weight_short(P))
      launch_tiles<KT, HAS_W, 4>(P, B, n, s);
    else if constexpr (KT == HCG_GAUSS2D)
      launch_tiles<KT, HAS_W, 5>(P, B, n, s);
  } else {
    launch_tiles<KT, HAS_W, 0>(P, B, n, s);
  }
  HCG_CHECK_LAUNCH("k_grid_tiles");
  return HCG_OK;
}

__global__ void __launch_bounds__(256) k_normalize(uint64_t n, const double* __restrict__ dc,
                                                   const double* __restrict__ wc, double* __restrict__ map) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) map[i] = dc[i] / wc[i];
}

}  // namespace hcg

using namespace hcg;

extern "C" int hcg_grid_plain(const hcg_healpix* hp, const hcg_kernel* kern, uint32_t side, uint32_t n,
                              const hcg_sample* records, const uint32_t* keys_sorted, const double* lon_sorted,
                              const double* lat_sorted, const double* weights_sorted, const uint32_t* lut,
                              const double* ring_z, const double* ring_s, const hcg_ring_meta* meta,
                              const double* xwcs, const double* ywcs, double* datacube, double* weightscube,
                              void* stream) {
  HCG_REQUIRE(hp && kern, "hcg_grid_plain: NULL hp/kern");
  if (hp->nside == 0 || hp->nside > HCG_MAX_NSIDE)
    return set_error(HCG_ERR_UNSUPPORTED, "hcg_grid_plain: nside must be <= 8192");
  HCG_REQUIRE(kern->kernel_type >= HCG_GAUSS1D && kern->kernel_type <= HCG_TAPERED_SINC,
              "hcg_grid_plain: unknown kernel type");
  HCG_REQUIRE(kern->factor >= 1, "hcg_grid_plain: factor must be >= 1");
  HCG_REQUIRE(kern->selection <= HCG_SELECT_DISC,
              "hcg_grid_plain: selection must be HCG_SELECT_COMPAT or HCG_SELECT_DISC");
  HCG_REQUIRE(side <= 65535, "hcg_grid_plain: side must be <= 65535");
  if (side == 0) return HCG_OK;
  HCG_REQUIRE(records && keys_sorted && lon_sorted && lat_sorted && lut && ring_z && ring_s && meta && xwcs &&
                  ywcs && datacube && weightscube,
              "hcg_grid_plain: NULL buffer");
  GridParams P = make_grid_params(hp, kern, side);
  GridBuffers B{records, keys_sorted, lon_sorted, lat_sorted, weights_sorted, lut, ring_z, ring_s, meta,
                xwcs,    ywcs,        datacube,   weightscube};
  hipStream_t s = as_stream(stream);
  const bool hw = weights_sorted != nullptr;
  switch (kern->kernel_type) {
    case HCG_GAUSS1D: return hw ? launch_grid<HCG_GAUSS1D, true>(P, B, n, s) : launch_grid<HCG_GAUSS1D, false>(P, B, n, s);
    case HCG_GAUSS2D: return hw ? launch_grid<HCG_GAUSS2D, true>(P, B, n, s) : launch_grid<HCG_GAUSS2D, false>(P, B, n, s);
    default: return hw ? launch_grid<HCG_TAPERED_SINC, true>(P, B, n, s) : launch_grid<HCG_TAPERED_SINC, false>(P, B, n, s);
  }
}

extern "C" int hcg_normalize(uint64_t ncells, const double* datacube, const double* weightscube, double* map,
                             void* stream) {
  if (ncells == 0) return HCG_OK;
  HCG_REQUIRE(datacube && weightscube && map, "hcg_normalize: NULL buffer");
  const uint32_t blocks = (uint32_t)std::min<uint64_t>((ncells + 255) / 256, 8192);
  k_normalize<<<blocks, 256, 0, as_stream(stream)>>>(ncells, datacube, weightscube, map);
  HCG_CHECK_LAUNCH("k_normalize");
  return HCG_OK;
}

namespace hcg {
__global__ void __launch_bounds__(64) k_eval_exp_neg(uint32_t n, const double* __restrict__ x, double* __restrict__ out) {
  __shared__ double s_exp[64];
  exp_table_load(s_exp);
  __syncthreads();
  const uint32_t i = blockIdx.x * 64 + threadIdx.x;
  if (i < n) out[i] = exp_neg(x[i], s_exp);
}
}  // namespace hcg

extern "C" int hcg_eval_exp_neg(uint32_t n, const double* x, double* out, void* stream) {
  if (n == 0) return HCG_OK;
  HCG_REQUIRE(x && out, "hcg_eval_exp_neg: NULL buffer");
  k_eval_exp_neg<<<ceil_div_u32(n, 64), 64, 0, as_stream(stream)>>>(n, x, out);
  HCG_CHECK_LAUNCH("k_eval_exp_neg");
  return HCG_OK;
}
