// plain_tile.hpp -- one tile of the single-channel gather-convolution, the
// body of k_grid_tiles (grid_plain.hip), shared with the one- and
// few-channel jobs of the multi-channel entry points (grid_plain.hip's
// k_grid_tiles_1ch / k_grid_tiles_few, and k_batch_tiles for the jobs of a
// batch).
//
// A tile is kTileCols x kTileRows (16 x 4) map cells worked by one wave, in
// three steps:
//   1. lane = cell (column lane / 4, row lane % 4): the cell's window and
//      unit vector;
//   2. lane = ring: the sorted range of each of the tile's rings (up to 64
//      at once), a superset of the union of its cells' windows, by a binary
//      search per lane.  One such round of dependent loads per tile replaces
//      two cooperative searches per ring;
//   3. the ranges are staged in LDS (as many rings as fit at a time), and
//      ring by ring the four lanes of a column take the samples between the
//      column's window edges four at a time (lane phase p: samples p, p + 4,
//      ...) and test each against the column's four cells: its window (one
//      integer compare in half-pixel units, belt_window) and the radius.
// A sample is read from LDS once for four cells, and the four rows are
// separate branches: at a given step the sixteen columns stand at the same
// place of their bands, so a row whose disc does not reach the ring, or no
// longer reaches this far along it, is skipped by the whole wave.  The loop
// is bound by FP64 issue (a candidate costs three FMAs and the compares, a
// selected pair thirteen more), so what counts is that the lanes of a weight
// evaluation are nearly all selected: with lane = cell and one band per lane
// 44% of the lane slots did selected pairs on the 20M-sample raster (rows
// outside a ring's reach and the window's corners outside the disc idled
// through the weight): 1.97e9 vector instructions and 4.40 ms then, 1.39e9
// and 3.49 ms now.  On sparse maps the per-ring chain of searches, loads and
// window arithmetic is what counts (160k samples onto 1024^2: 199 us).
//
// The selection, distance and weight are the ones described in
// grid_plain.hip; a cell's sum is the sum of its four phases' partial sums
// (and of its ring streams'), each in ring and sorted order.
// Instantiations:
//  * BATCH false (k_grid_tiles): FP64 values from the sample records, sums
//    added to the FP64 data and weight cubes (the reference's
//    datacube/weightscube);
//  * BATCH true (a one-channel job of the multi-channel entry points): the
//    job's sorted 16-bit values; the caller adds the streams in stream order
//    and writes the FP32 cube (divided by the weight sum when the job
//    normalises; NaN where no sample contributes) and FP32 weight sum
//    (tile_write);
//  * NC > 0 (few-channel jobs): as BATCH true, with one FP32 sum per channel.
// All synchronisation is within the wave, so the waves of a workgroup may
// work other tiles or streams.
#pragma once

#include <hip/hip_runtime.h>

#include "common.hpp"
#include "expneg.hpp"
#include "healpix.hpp"

namespace hcg {

// Sorted channel values (multi-channel jobs) are blocked by kVB samples:
// block b holds the [nchan][kVB] values of sorted samples kVB b .. kVB b +
// kVB - 1, so a lane's 16-byte MFMA operand (8 samples of one channel) is
// one block row, and the MFMA path packs ring ranges at this granularity.
constexpr uint32_t kVB = 8;

constexpr int kTileCols = 16;
constexpr int kTileRows = 4;
constexpr uint32_t kPhases = 4;      // lanes that share a column's band
constexpr uint32_t kStageCap = 256;  // staged samples
constexpr uint32_t kShortRing = 12;  // a ring's staged samples up to which every column takes them all
static_assert(kTileCols * kTileRows == 64 && kTileCols * kPhases == 64, "one wave per tile");

}  // namespace hcg

#include "gridcore.hpp"

namespace hcg {

// LDS ordering among the lanes of one wave: its LDS instructions execute in
// issue order, so a compiler fence at wavefront scope is enough.
__device__ inline void tile_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// A one-channel job's values and outputs (BATCH true).
struct TileOut {
  const uint16_t* vs;  // sorted values, BF16 or FP16: [n_pad] (one channel), or 8-sample blocked
                       // [n_pad / 8][nchan][8] (few channels)
  float* cube;         // [nchan][side * side]
  float* wsum;         // [side * side] or NULL
  uint32_t bf16;       // vs holds BF16 (else FP16)
  uint32_t normalize;  // cube = sums / weight sums
  uint32_t nchan;      // channels (few-channel tiles)
};

// The part of a tile's non-empty rings one call of grid_tile walks: the
// phase-th, the phase + stride-th, ... in ascending order (all of them:
// phase 0, stride 1; stride a power of two).
struct RingStream {
  uint32_t phase, stride;
};

// Per-wave LDS of a one-channel tile: staged x, y, z, value columns and keys
// (of a size that lets four four-wave workgroups share a CU).
constexpr uint32_t kOneCap = 192;
constexpr size_t kTileLdsBytes = (size_t)kOneCap * (4 * sizeof(double) + sizeof(uint32_t));

// Tiles of the kTileCols x kTileRows tiling of a side x side map.
inline uint32_t tile_cols_of(uint32_t side) { return (side + kTileCols - 1) / kTileCols; }
inline uint32_t tile_count_of(uint32_t side) { return tile_cols_of(side) * ((side + kTileRows - 1) / kTileRows); }

// One-channel jobs of the multi-channel entry points (hcg_grid_mfma*, batch
// jobs) that take the FP64 tile path instead of the MFMA contraction:
// GAUSS1D, no per-sample weights, a radius small enough for the three-term
// weight series.  The result is closer to FP64 (unrounded weights), and with
// one channel the weight is all the work: here and in the contraction 1M
// samples onto 512^2 227 and 304 us, 300k onto 2048^2 631 and 934, 5k onto 20^2
// 68 and 79; 2M onto 128^2, on few tiles, 1374 and 1090.
inline bool one_channel_tiles(const GridParams& P, uint32_t kernel_type, bool weighted, uint32_t nchan) {
  return nchan == 1 && kernel_type == HCG_GAUSS1D && !weighted && gauss_tiny_radius(P);
}

// Partial streams per tile of a one-channel job, fixed by the map alone (so
// a job's sums do not depend on the launch shape): maps of fewer than
// kOneChannelMinTiles tiles (four per SIMD of the 256-CU chip) split each
// tile's rings over kOneChannelStreams waves, ring r to stream
// (r - first ring) % streams; larger maps take one wave per tile.  (A
// 5M-sample 128^2 map, 256 tiles, took 25 ms on one wave per tile.)
constexpr uint32_t kOneChannelMinTiles = 4096;
constexpr uint32_t kOneChannelStreams = 4;
inline uint32_t one_channel_streams(uint32_t side) {
  return tile_count_of(side) < kOneChannelMinTiles ? kOneChannelStreams : 1u;
}

// Few-channel jobs (2..kFewChannels channels on sparse maps, at most one
// sample per kFewCellsPerSample cells, otherwise as one_channel_tiles, at
// dot_distance_ok radii (their tile loop tests candidates on p.q), on maps
// of at least kOneChannelMinTiles tiles) also take the tile loop: FP64
// weights, FP32 accumulation per channel, one wave per tile.  On sparse maps a
// set-up per 64 cells and no value blocks outweigh the matrix products: 300k
// samples x 2 onto 2048^2 (0.07 samples per cell) 655 us here and 935 in the
// contraction, x 8 692 and 947; 400k x 8 onto 2048^2 (0.095) 775 and 994; 20k x
// 8 onto 512^2 48 and 65.  On denser maps the contraction is the faster one
// (195k x 3 onto 500^2: 190 us a pass, and 382 with this loop before it had
// its registers).
constexpr int kFewChannels = 8;
constexpr uint32_t kFewCellsPerSample = 10;
constexpr uint32_t kFewCap = 128;  // staged samples per round
constexpr size_t kFewTileLdsBytes = (size_t)kFewCap * (3 * sizeof(double) + sizeof(uint32_t) + kFewChannels * 2);

inline bool few_channel_tiles(const GridParams& P, uint32_t kernel_type, bool weighted, uint32_t nchan, uint32_t n) {
  return nchan >= 2 && nchan <= (uint32_t)kFewChannels &&
         (uint64_t)n * kFewCellsPerSample <= (uint64_t)P.side * P.side && kernel_type == HCG_GAUSS1D && !weighted &&
         gauss_tiny_radius(P) && dot_distance_ok(P) && tile_count_of(P.side) >= kOneChannelMinTiles;
}

// Launches the tile path for one one-channel job: one workgroup per tile,
// one_channel_streams(side) waves.
int launch_tiles_one_channel(const GridParams& P, const GridBuffers& B, const TileOut& O, hipStream_t s);

// Launches the tile path for one few-channel job: one wave per tile.
int launch_tiles_few_channels(const GridParams& P, const GridBuffers& B, const TileOut& O, hipStream_t s);

// ---- the quad of lanes that share a column (DPP, no LDS traffic) ----

template <int CTRL>
__device__ inline uint32_t quad_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ inline double quad_f64(double v) {
  const uint64_t u = __builtin_bit_cast(uint64_t, v);
  return __builtin_bit_cast(double, (uint64_t)quad_u32<CTRL>((uint32_t)u) |
                                        ((uint64_t)quad_u32<CTRL>((uint32_t)(u >> 32)) << 32));
}
template <int CTRL>
__device__ inline float quad_f32(float v) {
  return __builtin_bit_cast(float, quad_u32<CTRL>(__builtin_bit_cast(uint32_t, v)));
}
constexpr int kQuadXor1 = 0xB1, kQuadXor2 = 0x4E;  // quad_perm [1,0,3,2], [2,3,0,1]
constexpr int quad_bcast(int r) { return r * 0x55; }
// v[r] = x of the quad's lane r, r < ROWS
template <int ROWS>
__device__ inline void quad_all(uint32_t x, uint32_t (&v)[ROWS]) {
  v[0] = ROWS == 1 ? x : quad_u32<quad_bcast(0)>(x);
  if constexpr (ROWS > 1) v[1] = quad_u32<quad_bcast(1)>(x);
  if constexpr (ROWS > 2) {
    v[2] = quad_u32<quad_bcast(2)>(x);
    v[3] = quad_u32<quad_bcast(3)>(x);
  }
}
template <int ROWS>
__device__ inline void quad_all(double x, double (&v)[ROWS]) {
  v[0] = ROWS == 1 ? x : quad_f64<quad_bcast(0)>(x);
  if constexpr (ROWS > 1) v[1] = quad_f64<quad_bcast(1)>(x);
  if constexpr (ROWS > 2) {
    v[2] = quad_f64<quad_bcast(2)>(x);
    v[3] = quad_f64<quad_bcast(3)>(x);
  }
}
// row `row`'s sum over the quad
template <int ROWS>
__device__ inline double quad_rows_sum(const double (&v)[ROWS], uint32_t row) {
  double out = 0.0;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    double t = v[r] + quad_f64<kQuadXor1>(v[r]);
    t += quad_f64<kQuadXor2>(t);
    if (r == 0 || row == (uint32_t)r) out = t;
  }
  return out;
}
template <int ROWS>
__device__ inline float quad_rows_sum(const float (&v)[ROWS], uint32_t row) {
  float out = 0.f;
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    float t = v[r] + quad_f32<kQuadXor1>(v[r]);
    t += quad_f32<kQuadXor2>(t);
    if (r == 0 || row == (uint32_t)r) out = t;
  }
  return out;
}

// The windows of a tile taken together, for the ring ranges: the span of the
// longitudes (compat) and of the longitude ranges (polar, disc) of its cells.
struct TileSpan {
  uint32_t r_begin, r_end;     // rings (r_begin > r_end: none)
  bool any_compat, any_range;  // some cell has a window of that kind
  bool whole;                  // some cell takes whole rings, or longitudes are not in [0, 2 pi)
  double tl, tr;               // the outermost compat window edges (units of pi/2, not reduced)
  float tlo, thi;              // outermost ranges
  bool disc;                   // HCG_SELECT_DISC
  // the cells themselves: sin of the latitudes, relative to zref, the least
  // cos, and the longitudes in units of pi/2 (ring_chord)
  double zref;
  float zmin, zmax, cmin, tmin, tmax;
};

// (pz, coslat, tt: sin and cos of the lane's cell's latitude, its longitude in units of pi/2 in [0, 4))
__device__ inline TileSpan tile_span(const GridParams& P, const Window& w, uint32_t firstring, double pz,
                                     double coslat, double tt) {
  TileSpan t;
  const bool has = w.uring <= w.dring;
  t.r_begin = wave_min_u32(has ? w.uring : 0xFFFFFFFFu);
  t.r_end = wave_max_u32(has ? w.dring : 0u);
  if (t.r_begin == firstring && skips_first_ring(P)) ++t.r_begin;  // the first used ring contributes nothing
  const bool compat = has && w.mode == kWinCompat, range = has && w.mode != kWinCompat;
  t.any_compat = __ballot(compat) != 0;
  t.any_range = __ballot(range) != 0;
  t.disc = P.selection == HCG_SELECT_DISC;
  t.whole = false;
  t.tl = t.tr = 0.0;
  t.tlo = 1.f;
  t.thi = 0.f;
  if (t.any_compat) {
    const double lo = wave_min_f64(compat ? w.phi : 1e300);
    const double hi = -wave_min_f64(compat ? -w.phi : 1e300);
    t.whole = !(lo >= 0.0 && hi < 2.0 * kPi);
    t.tl = (lo - P.disc_size) * kInvHalfPi;
    t.tr = (hi + P.disc_size) * kInvHalfPi;
  }
  if (t.any_range) {
    t.whole = t.whole || __ballot(range && !(w.range.tlo <= w.range.thi)) != 0;
    t.tlo = (float)wave_min_f64(range ? (double)w.range.tlo : 1e300);
    t.thi = (float)-wave_min_f64(range ? -(double)w.range.thi : 1e300);
  }
  t.zref = wave_min_f64(has ? pz : 1e300);
  t.zmin = 0.f;
  t.zmax = wave_max_f32(has ? (float)(pz - t.zref) : 0.f) * (1.f + 1e-6f);
  t.cmin = -wave_max_f32(has ? -(float)coslat : -2.f) * (1.f - 1e-6f);
  t.tmin = -wave_max_f32(has ? -(float)tt : -8.f) - 1e-6f;
  t.tmax = wave_max_f32(has ? (float)tt : -8.f) + 1e-6f;
  return t;
}

// What the radius reaches of a ring.  A sample at latitude bs within R of a
// cell at bc has hav R > hav(bs - bc) + cos bs cos bc hav(dl); the pixels of a
// ring lie between the centre latitudes of its neighbours, so
// |sin(bs) - sin(bc)| >= dz, the gap between that band and the cell, and with
// |sin bs - sin bc| <= 2 sin(|bs - bc| / 2) max cos,
//   sin^2(dl / 2) <= (sin^2(R / 2) - (dz / (2 max cos))^2) / (min cos bs min cos bc).
// In half pixels of the ring a sample within reach of a cell at x = q2 tt has
// its position within k sqrt(h2 - dz^2) of x, and none is where h2 <= dz^2.
// Single precision, relative to the tile's zref: R is widened by 1e-5, which
// covers what is relative to dz, and the band by what rounding leaves of its
// edges and of the cells' places (tiles may be far larger than the radius) and
// by what the keys' own rounding does (pixel edges move by ~1e-15).  The
// position of a sample at longitude x is within [x - 2, x + 3].
struct RingChord {
  float zu, zd;  // the band, sin of latitude relative to the tile's zref
  float h2, k, q2;
};
// (half2d: sin^2(R / 2))
__host__ __device__ inline RingChord ring_chord(double half2d, const TileSpan& T, uint32_t npr, uint32_t kr,
                                       uint32_t usedrings, const double* __restrict__ ring_z) {
  RingChord c;
  c.q2 = 0.5f * (float)npr;
  if (kr == 0 || kr + 1 >= usedrings) {  // the neighbours' latitudes are not at hand: no narrowing
    c.zu = 1e9f;
    c.zd = -1e9f;
    c.h2 = c.k = 1e30f;
    return c;
  }
  const double zu = ring_z[kr - 1], zd = ring_z[kr + 1];
  c.zu = (float)(zu - T.zref);
  c.zd = (float)(zd - T.zref);
  constexpr float kEps = 1.2e-7f;  // 2^-23: half an ulp of an edge and of a cell each, twice over
  c.zu += fmaf(kEps, fabsf(c.zu) + T.zmax, 4e-15f);
  c.zd -= fmaf(kEps, fabsf(c.zd) + T.zmax, 4e-15f);
  const float cu = (float)((1.0 - zu) * (1.0 + zu)), cd = (float)((1.0 - zd) * (1.0 + zd));  // cos^2
  const double zlo = T.zref, zhi = T.zref + (double)T.zmax;
  // the largest cos^2 between the band and the cells: 1 if they straddle the equator
  float cmax2 = fmaxf(fmaxf(cu, cd), (float)(zlo > 0.0 ? (1.0 - zlo) * (1.0 + zlo) : (1.0 - zhi) * (1.0 + zhi)));
  if (!((zd > 0.0 && zlo > 0.0) || (zu < 0.0 && zhi < 0.0))) cmax2 = 1.f;
  cmax2 = 4.00004f * cmax2;
  const float half2 = (float)half2d * (1.f + 1e-5f);
  const float cc = sqrtf(fminf(cu, cd)) * T.cmin * (1.f - 1e-5f);
  const float s2 = half2 / cc;
  c.h2 = half2 * cmax2;
  // asin s <= s / sqrt(1 - s^2)
  c.k = cc > 0.f && s2 < 0.25f ? c.q2 * (float)(4.0 / kPi) * 1.00001f / sqrtf(cc * (1.f - s2) * cmax2) : 1e30f;
  return c;
}
// Narrows the keys lp..rp of a ring (first pixel sp, npr pixels) to what the
// radius reaches from the tile; false: nothing.
__host__ __device__ inline bool chord_pixels(const TileSpan& T, const RingChord& c, uint32_t sp, uint32_t npr,
                                             uint32_t& lp, uint32_t& rp) {
  const float dz = fmaxf(fmaxf(c.zd - T.zmax, T.zmin - c.zu), 0.f);
  const float num = fmaf(-dz, dz, c.h2);
  if (!(num > 0.f)) return false;
  const float hc = fmaf(c.k, sqrtf(num), 0.1f);
  const float xl = fmaf(T.tmin, c.q2, -hc), xh = fmaf(T.tmax, c.q2, hc);
  if (T.tmax - T.tmin < 1.f && xl >= 0.f && xh < 2.f * (float)npr - 4.f) {
    lp = max(lp, sp + ((uint32_t)xl >> 1));
    rp = min(rp, sp + ((uint32_t)xh >> 1) + 1u);
  }
  return lp <= rp;
}

// What the radius reaches of a ring from one cell (zf: sin of its latitude
// relative to zref, ttf: its longitude in units of pi/2): half-pixel positions
// xl to xh, all of them if not narrow.
struct CellReach {
  bool any, narrow;
  float xl, xh;
};
// (chord(&RingChord::m): the ring's m, read where it is used: read together, one
// after the other, 20M samples take 1% longer)
template <class F>
__host__ __device__ inline CellReach chord_cell(const F& chord, float zf, float ttf) {
  CellReach r;
  const float q2 = chord(&RingChord::q2);
  const float dz = fmaxf(fmaxf(chord(&RingChord::zd) - zf, zf - chord(&RingChord::zu)), 0.f);
  const float num = fmaf(-dz, dz, chord(&RingChord::h2));
#if defined(__HIP_DEVICE_COMPILE__)
  const float root = __builtin_amdgcn_sqrtf(fmaxf(num, 0.f));
#else
  const float root = sqrtf(fmaxf(num, 0.f));
#endif
  const float hc = fmaf(chord(&RingChord::k), root, 2.2f);
  r.xl = fmaf(ttf, q2, -hc);
  r.xh = fmaf(ttf, q2, hc + 2.f);
  r.any = !(num <= 0.f);
  r.narrow = r.xl >= 0.f && r.xh < 4.f * q2 - 4.f;
  return r;
}

// A pixel range of ring r that holds every cell's window in it (ring_window):
// a ring's pixel index grows with the longitude, so the outermost edges bound
// the others; two pixels of margin.  Within three pixels of longitude 0 an
// edge opens to the ring's end (a cell whose own window wraps through 0
// selects nothing, since its lpix is then past its rpix), and whole rings
// are taken where the reasoning ends.
__device__ inline void span_pixels(const Hpx32& hx, const TileSpan& t, uint32_t ring, double rz, double rs,
                                   uint32_t& lp, uint32_t& rp) {
  uint32_t sp, npr;
  ring_info32(hx, ring, sp, npr);
  const uint32_t last = sp + npr - 1;
  lp = sp;
  rp = last;
  const bool cap = ring < hx.nside || ring > 3 * hx.nside;
  if (t.whole || (t.any_range && !cap && !t.disc)) return;
  uint32_t a = last, b = sp;
  if (t.any_compat) {
    const bool have = rs >= 0.0;
    const double q = (double)(npr >> 2);
    a = sp;
    b = last;
    if (t.tl * q > 3.0) {
      const uint32_t l = loc2pix32(hx, rz, t.tl, have ? rs : 0., have);
      if (l - sp >= npr) return;
      a = l - sp < 2 ? sp : l - 2;
    }
    if (t.tr * q < (double)npr - 3.0) {
      const uint32_t r = loc2pix32(hx, rz, t.tr, have ? rs : 0., have);
      if (r - sp >= npr) return;
      b = last - r < 2 ? last : r + 2;
    }
  }
  if (t.any_range) {
    const float q = (float)(npr >> 2);
    const int32_t m = t.disc ? 4 : 3;
    const int32_t lo = (int32_t)floorf(t.tlo * q) - m;
    const int32_t hi = (int32_t)floorf(t.thi * q) + m;
    if (lo < 0 || hi >= (int32_t)npr) return;
    a = min(a, sp + (uint32_t)lo);
    b = max(b, sp + (uint32_t)hi);
  }
  lp = a;
  rp = b;
}

// The sorted range [lo, hi) of the keys lp..rp within [start, end) (start < end).
// Both bounds in one loop, three probes each a step: a step is one round of
// dependent loads, and the range falls to a quarter.
__device__ inline void key_range(const uint32_t* __restrict__ keys, uint32_t start, uint32_t end, uint32_t lp,
                                 uint32_t rp, uint32_t& lo, uint32_t& hi) {
  uint32_t a0 = start, a1 = end, b0 = start, b1 = end;
  while (a0 < a1 || b0 < b1) {
    const uint32_t da = (a1 - a0) >> 2, db = (b1 - b0) >> 2;
    // a0 <= pa0 <= pa1 <= pa2 < a1 while the range is not empty; index
    // `end` of an empty one can be read (keys[n] is the sentinel)
    const uint32_t pa0 = a0 + da, pa1 = a0 + ((a1 - a0) >> 1), pa2 = pa1 + da;
    const uint32_t pb0 = b0 + db, pb1 = b0 + ((b1 - b0) >> 1), pb2 = pb1 + db;
    const uint32_t ka0 = keys[pa0], ka1 = keys[pa1], ka2 = keys[min(pa2, end)];
    const uint32_t kb0 = keys[pb0], kb1 = keys[pb1], kb2 = keys[min(pb2, end)];
    if (a0 < a1) {
      if (pa2 < a1 && ka2 < lp)
        a0 = pa2 + 1;
      else if (ka1 < lp)
        a0 = pa1 + 1, a1 = min(a1, pa2);
      else if (ka0 < lp)
        a0 = pa0 + 1, a1 = pa1;
      else
        a1 = pa0;
    }
    if (b0 < b1) {
      if (pb2 < b1 && kb2 <= rp)
        b0 = pb2 + 1;
      else if (kb1 <= rp)
        b0 = pb1 + 1, b1 = min(b1, pb2);
      else if (kb0 <= rp)
        b0 = pb0 + 1, b1 = pb1;
      else
        b1 = pb0;
    }
  }
  lo = a0;
  hi = b0;
}

// The sorted range of a ring's part of the tile (lo >= hi: none), and its
// chord.  Out of line, as the windows of general rings are: both run next to
// the sample loop, and inline their temporaries and constants take its
// registers (270k samples onto 300^2 with GAUSS2D: a pass 481 -> 278 us).
struct RingRange {
  uint32_t lo, hi;
  RingChord c;
};
[[maybe_unused]] static __device__ __noinline__ RingRange ring_range_call(Hpx32 hx, TileSpan T, double half2,
                                                                          uint32_t firstring, uint32_t usedrings,
                                                                          const uint32_t* lut, const double* ring_z,
                                                                          const double* ring_s, const uint32_t* keys,
                                                                          uint32_t ring) {
  RingRange r{};
  if (T.r_begin > T.r_end || ring > T.r_end) return r;
  const uint32_t kr = ring - firstring;
  const uint32_t start = lut[kr], end = lut[kr + 1];
  if (start >= end) return r;
  uint32_t lp, rp, sp, npr;
  span_pixels(hx, T, ring, ring_z[kr], ring_s[kr], lp, rp);
  ring_info32(hx, ring, sp, npr);
  r.c = ring_chord(half2, T, npr, kr, usedrings, ring_z);
  if (chord_pixels(T, r.c, sp, npr, lp, rp)) key_range(keys, start, end, lp, rp, r.lo, r.hi);
  return r;
}
__device__ inline RingRange ring_range(const GridParams& P, const GridBuffers& B, const TileSpan& T,
                                       const hcg_ring_meta& m, uint32_t ring) {
  return ring_range_call(hpx32(P.hp), T, P.polar_half * P.polar_half, m.firstring, m.usedrings, B.lut, B.ring_z,
                         B.ring_s, B.keys, ring);
}

// lpix | rpix << 32 of ring_window_at; 1 | 0 for none
[[maybe_unused]] static __device__ __noinline__ uint64_t ring_window_call(Hpx32 hx, Window w, double tl, double tr,
                                                                          uint32_t ring, double rz, double rs) {
  uint32_t a = 1, b = 0;
  if (!ring_window_at(hx, w, tl, tr, ring, rz, rs, a, b)) return 1;
  return (uint64_t)b << 32 | a;
}

// First index in [from, from + cnt) with g >= x (from + cnt if none), in
// halving steps that are uniform over the wave (cnt > 0).
__device__ inline uint32_t band_search(const uint32_t* __restrict__ g, uint32_t from, uint32_t cnt, uint32_t x) {
  uint32_t a = 0;
  for (uint32_t s = 1u << (31 - __builtin_clz(cnt)); s; s >>= 1) {
    const uint32_t i = a + s;
    const uint32_t v = g[from + min(i, cnt) - 1];
    if (i <= cnt && v < x) a = i;
  }
  return from + a;
}

// Inclusive maximum over the lanes up to this one.
__device__ inline uint32_t wave_scan_max_u32(uint32_t v) {
  v = max(v, dpp_u32<kRowShr1, 0xF>(0u, v));
  v = max(v, dpp_u32<kRowShr2, 0xF>(0u, v));
  v = max(v, dpp_u32<kRowShr4, 0xF>(0u, v));
  v = max(v, dpp_u32<kRowShr8, 0xF>(0u, v));
  v = max(v, dpp_u32<kRowBcast15, 0xA>(0u, v));
  return max(v, dpp_u32<kRowBcast31, 0xC>(0u, v));
}

// A cell's window in a ring, in half pixels: sample (pixel p of ring r, p
// counted from the ring's first) is in it when g - lo <= hi - lo (unsigned),
// g = 2 p + 1 - (r odd).
//
// In a belt ring (nside < r < 3 nside) pixel boundaries lie at longitudes tt
// (units of pi/2) whose nside tt is an integer for even r and a half-integer
// for odd r: the formulas of HCGrid/healpix.cu:126-205 at the ring's centre
// give p = floor(nside tt) and floor(nside tt + 1/2).  With h = floor(2 nside
// tt), an edge at tt lies in pixel floor(h / 2) or floor((h + 1) / 2), and a
// window from tl to tr holds the samples with hl <= g <= hr + 1 whatever the
// ring's parity.  So a compat window is one pair of numbers for every belt
// ring.  Exact unless an edge is within rounding of a boundary (2 nside tt
// within 1e-6 of an integer; the formulas' own error is below 1e-10), or the
// window meets longitude 0: then (returns false) the tile evaluates its
// windows ring by ring.
constexpr uint32_t kNoWindow = 0x80000001u;  // lo of a cell outside the ring's range: no g reaches it
__device__ inline bool belt_window(const GridParams& P, double tl, double tr, uint32_t& lo, uint32_t& hi) {
  const uint32_t ns = (uint32_t)P.hp.nside;
  const double xl = 2.0 * (double)ns * tl, xr = 2.0 * (double)ns * tr;
  const double fl = floor(xl), fr = floor(xr);
  lo = (uint32_t)fl;
  hi = (uint32_t)fr + 1;
  const double gl = xl - fl, gr = xr - fr;
  return ns >= 2 && gl > 1e-6 && gl < 1.0 - 1e-6 && gr > 1e-6 && gr < 1.0 - 1e-6 && xl < xr &&
         xr < 8.0 * (double)ns - 2.0;
}

__device__ inline float high_f32(double x) {
  return __builtin_bit_cast(float, (uint32_t)(__builtin_bit_cast(uint64_t, x) >> 32));
}

// A tile's sums, one cell per lane (column lane / 4, row lane % 4).
template <int NC>
struct TileSums {
  double d, w;
  float c[NC > 0 ? NC : 1];
};

// Step 1 and 2 of a tile, for the other waves of its workgroup.
struct TileShared {
  Window win[64];
  double tl[64], tr[64], p[3][64];
  RingRange rings[64];
  float tt[64];
  TileSpan T;
};

// WMODE (GAUSS1D): 0 general exponent and exp; 1 gauss_small_radius; 2
// gauss_tiny_radius; 3 also lean_weight_ok (the candidate test on p.q and
// the lean weight).  The other kernels: 0 general, 4 frame_weight_ok (5:
// GAUSS2D and not frame_weight_short).
// lds: CAP x (x, y, z, v doubles, key), with HAS_W then CAP weights; with NC
// > 0 CAP x (x, y, z doubles, key, NC 16-bit values).
// s_exp: the 64-entry exponential table (exp_table_load), visible to the wave.
// ROWS: map rows of the tile (4; fewer on small maps, for more tiles).
// SHARED: the waves of the workgroup walk streams of the same tile; wave 0
// works out the windows and ring ranges and the others take them from `sh`
// (holds a workgroup barrier).
template <int KT, bool HAS_W, int WMODE, bool BATCH, int NC, uint32_t CAP, int ROWS = kTileRows, bool SHARED = false>
__device__ __forceinline__ void grid_tile(const GridParams& P, const GridBuffers& B, uint32_t tile, uint32_t tiles_x,
                                          char* __restrict__ lds, const double* __restrict__ s_exp, const TileOut& O,
                                          RingStream S, TileSums<NC>& out, TileShared* sh = nullptr) {
  static_assert(NC == 0 || (BATCH && NC % 2 == 0 && WMODE == 3), "few-channel tiles: even counts, the lean weight");
  static_assert(WMODE != 3 || KT == HCG_GAUSS1D, "the lean weight is GAUSS1D's");
  static_assert(!(HAS_W && BATCH), "batch jobs carry no sample weights");
  double* const s_x = reinterpret_cast<double*>(lds);
  double* const s_y = s_x + CAP;
  double* const s_z = s_y + CAP;
  double* const s_v = s_z + CAP;                                   // NC == 0
  double* const s_w = s_v + CAP;                                   // HAS_W
  uint32_t* const s_g = reinterpret_cast<uint32_t*>(NC > 0 ? s_v : HAS_W ? s_w + CAP : s_w);
  uint16_t* const s_c = reinterpret_cast<uint16_t*>(s_g + CAP);  // NC > 0

  const hcg_ring_meta m = *B.meta;
  const uint32_t lane = __lane_id();
  const uint32_t row = lane & (ROWS - 1u);  // this lane's row as a cell
  const uint32_t phase = lane & 3u;         // and its phase in the sample loop
  const uint32_t col = (tile % tiles_x) * kTileCols + (lane >> 2);
  const uint32_t row0 = (tile / tiles_x) * ROWS;

  double npx[ROWS], npy[ROWS], npz[ROWS], acc_d[ROWS], acc_w[ROWS];
  float acc_c[ROWS][NC > 0 ? NC : 1];
#pragma unroll
  for (int r = 0; r < ROWS; ++r) {
    acc_d[r] = acc_w[r] = 0.0;
#pragma unroll
    for (int c = 0; c < (NC > 0 ? NC : 1); ++c) acc_c[r][c] = 0.f;
  }
  // GAUSS2D's tangent frames (WMODE 4): east and north turned by the position angle
  constexpr bool kFrame = (WMODE == 4 || WMODE == 5) && KT == HCG_GAUSS2D;
  double fu[kFrame ? ROWS : 1][3], fv[kFrame ? ROWS : 1][3];
  Window win;
  double tl = 0.0, tr = 0.0;  // compat: the window's edges, fmodulo4 in units of pi/2
  // the span waits in LDS: past the set-up only a tile of more than 64 rings
  // wants it (in registers it took 25 to 70 more spills in the sample loop's
  // surroundings; with the shared tiles' windows, passes 331 -> 296 us on the
  // disc at dec 80, 279 -> 252 with GAUSS2D, 85 -> 79 on the 20^2 map)
  __shared__ TileSpan spans[SHARED ? 1 : kOneChannelStreams];
  TileSpan& far_span = SHARED ? sh->T : spans[threadIdx.x >> 6];
  uint32_t r_begin, r_end;
  RingRange ring_r;  // lane = ring: the ranges of 64 rings
  float zf, ttf;  // the cell's place, as ring_chord wants it
  {
    double px, py, pz;
    TileSpan T;
    if (!SHARED || threadIdx.x < 64) {
      const bool live = col < P.side && row0 + row < P.side;
      const uint32_t rr = live ? row0 + row : 0, cc = live ? col : 0;
      const uint32_t cell = rr * P.side + cc;
      const uint32_t anchor = rr * P.side + (cc / P.factor) * P.factor;
      win = window_of(P, m.firstring, m.usedrings, B.xwcs[anchor], B.ywcs[anchor]);
      if (!live || m.usedrings == 0) {  // an empty ring range: never active
        win.uring = 1;
        win.dring = 0;
      }
      if (win.mode == kWinCompat) compat_edges(P, win, tl, tr);
      double sb, cb, sl, cl;
      sincos(B.ywcs[cell] * kDeg2Rad, &sb, &cb);
      sincos(B.xwcs[cell] * kDeg2Rad, &sl, &cl);
      px = cb * cl;
      py = cb * sl;
      pz = sb;
      const double tt = fmodulo4(B.xwcs[cell] * kDeg2Rad * kInvHalfPi);
      ttf = (float)tt;
      T = tile_span(P, win, m.firstring, pz, cb, tt);
      ring_r = ring_range(P, B, T, m, T.r_begin + lane);
    }
    if constexpr (SHARED) {
      TileShared& H = *sh;
      if (threadIdx.x < 64) {
        H.win[lane] = win;
        H.tl[lane] = tl;
        H.tr[lane] = tr;
        H.p[0][lane] = px;
        H.p[1][lane] = py;
        H.p[2][lane] = pz;
        H.rings[lane] = ring_r;
        H.tt[lane] = ttf;
        if (lane == 0) H.T = T;
      }
      __syncthreads();
      if (threadIdx.x >= 64) {
        win = H.win[lane];
        tl = H.tl[lane];
        tr = H.tr[lane];
        px = H.p[0][lane];
        py = H.p[1][lane];
        pz = H.p[2][lane];
        ring_r = H.rings[lane];
        ttf = H.tt[lane];
        T = H.T;
      }
    }
    if constexpr (kFrame) {
      const uint32_t rr = min(row0 + row, P.side - 1), cc = min(col, P.side - 1);
      double sl, cl;
      sincos(B.xwcs[rr * P.side + cc] * kDeg2Rad, &sl, &cl);
      const double cb = cos(B.ywcs[rr * P.side + cc] * kDeg2Rad);
      const double e[3] = {-sl, cl, 0.0}, nn[3] = {-pz * cl, -pz * sl, cb};
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        double u[ROWS], v[ROWS];
        quad_all(fma(e[i], P.f[2], -(nn[i] * P.f[3])), u);
        quad_all(fma(nn[i], P.f[2], e[i] * P.f[3]), v);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) {
          fu[r][i] = u[r];
          fv[r][i] = v[r];
        }
      }
    }
    zf = (float)(pz - T.zref);
    r_begin = __builtin_amdgcn_readfirstlane(T.r_begin);
    r_end = __builtin_amdgcn_readfirstlane(T.r_end);
    if (!SHARED && lane == 0) far_span = T;
    // -p: h = 1 - p.q is three FMAs from 1
    quad_all(-px, npx);
    quad_all(-py, npy);
    quad_all(-pz, npz);
  }
  uint32_t hl0 = 0, hh0 = 0;  // the cell's window in every belt ring (belt_window)
  const bool has = win.uring <= win.dring;
  const bool belt_ok = __ballot(has && !(win.mode == kWinCompat && belt_window(P, tl, tr, hl0, hh0))) == 0;
  const uint32_t ns = (uint32_t)P.hp.nside;
  // WMODE 3: the tests on h = 1 - p.q = c2 / 2 (halving is exact, so
  // h < c_hi / 2 <=> c2 < c_hi)
  const double t_hi = WMODE == 3 ? 0.5 * P.c_hi : P.c_hi, t_lo = WMODE == 3 ? 0.5 * P.c_lo : P.c_lo;
  // With sample weights the pairs are tested on the high words of the
  // distances, compared as floats (a double's high word is its order, NaN
  // included): below t_lo32 selected, above t_hi32 not, and a lane between the
  // two (a relative 1e-6 of the radius around the guard band) is decided
  // exactly.  The 347^2 map with weights took 1160 us with these compares and
  // 1282 us with 64-bit ones; without weights the 64-bit ones are the faster
  // (20M samples: 3421 against 3527 us).
  constexpr bool kHigh = HAS_W;
  const float t_lo32 = high_f32(t_lo), t_hi32 = high_f32(t_hi);
  // the lean weight's constants for y = h (2 k0 + 4 k1 h), which equals
  // c2 (k0 + k1 c2); k1 and kExpE3 in vector registers (hoisted out of the loops)
  const double k0h = 2.0 * P.k0;
  const double k1v = WMODE == 3 ? in_vgprs(4.0 * P.k1) : 0.0, e3v = WMODE == 3 ? in_vgprs(kExpE3) : 0.0;
  uint32_t seen = 0;  // non-empty rings before this round

  for (uint32_t rb = r_begin; rb <= r_end && r_begin <= r_end; rb += 64) {
    // lane = ring
    if (rb != r_begin) {  // (more than 64 rings)
      tile_sync();
      ring_r = ring_range(P, B, far_span, m, rb + lane);
    }
    uint32_t lo_l = ring_r.lo;
    const uint32_t hi_l = ring_r.hi;
    const RingChord& chord_r = ring_r.c;
    const uint64_t ne = __ballot(lo_l < hi_l);
    const uint32_t rank = seen + (uint32_t)__popcll(ne & lanemask_lt());
    uint64_t mine = __ballot(lo_l < hi_l && (rank & (S.stride - 1u)) == S.phase);
    seen += (uint32_t)__popcll(ne);
    // of this lane's ring: g = 2 key + gc
    uint32_t gc;
    {
      uint32_t sp, npr;
      ring_info32(hpx32(P.hp), rb + lane, sp, npr);
      gc = 1u - ((rb + lane) & 1u) - 2u * sp;
    }
    while (mine) {  // uniform
      // A chunk: whole rings while they fit in CAP, or a piece of a longer
      // one.  On sparse maps it holds many rings, and one round of loads
      // serves them all.
      uint32_t cnt = 0, first = 0;
      uint32_t seg_off = 0, seg_len = 0, seg_src = 0;  // this lane's ring in the chunk
      uint64_t in = 0;                                 // the chunk's rings
      while (mine) {
        const uint32_t k = (uint32_t)__ffsll((unsigned long long)mine) - 1u;
        const uint32_t lo_u = __builtin_amdgcn_readlane(lo_l, k), hi_u = __builtin_amdgcn_readlane(hi_l, k);
        if (cnt != 0 && hi_u - lo_u > CAP - cnt) break;
        const uint32_t take = min(hi_u - lo_u, CAP);
        if (lane == k) {
          seg_off = cnt;
          seg_len = take;
          seg_src = lo_u;
          lo_l = lo_u + take;
        }
        if (cnt == 0) first = k;
        in |= 1ull << k;
        cnt += take;
        if (take < hi_u - lo_u) break;
        mine &= mine - 1;
      }
      const bool one_ring = (in & (in - 1)) == 0;
      tile_sync();  // previous chunk fully consumed
      if (!one_ring) {
        // each ring marks its first position; a position's ring is the last mark at or before it
        for (uint32_t p = lane; p < cnt; p += 64) s_g[p] = 0;
        tile_sync();
        if (in >> lane & 1u) s_g[seg_off] = lane + 1;
        tile_sync();
      }
      const uint32_t base1 = __builtin_amdgcn_readlane(seg_src, first), gc1 = __builtin_amdgcn_readlane(gc, first);
      uint32_t carry = 0;
      for (uint32_t p0 = 0; p0 < cnt; p0 += 128) {  // uniform; two positions per lane in flight
        uint32_t src[2], sgc[2];
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
          const uint32_t p = p0 + 64 * i + lane;
          src[i] = base1 + min(p, cnt - 1);
          sgc[i] = gc1;
          if (!one_ring && p0 + 64 * i < cnt) {  // uniform
            const uint32_t k1 = max(carry, wave_scan_max_u32(p < cnt ? s_g[p] : 0u));
            carry = (uint32_t)__builtin_amdgcn_readlane((int)k1, 63);
            const int from = (int)((k1 - 1) * 4);
            src[i] = min(p, cnt - 1) + (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)(seg_src - seg_off));
            sgc[i] = (uint32_t)__builtin_amdgcn_ds_bpermute(from, (int)gc);
          }
        }
        hcg_sample q[2];
        uint32_t key[2];
        double ws[2];
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i)
          if (p0 + 64 * i < cnt) {  // uniform
            q[i] = B.rec[src[i]];
            key[i] = B.keys[src[i]];
            if constexpr (BATCH && NC == 0) q[i].v = (double)widen16(O.vs[src[i]], O.bf16 != 0);
            if constexpr (HAS_W) ws[i] = B.w_s[src[i]];
          }
#pragma unroll
        for (uint32_t i = 0; i < 2; ++i) {
          const uint32_t j = p0 + 64 * i + lane;
          if (j < cnt) {
            s_x[j] = q[i].x;
            s_y[j] = q[i].y;
            s_z[j] = q[i].z;
            if constexpr (HAS_W) {  // the value times its weight, and the weight: one FMA each per pair
              s_v[j] = q[i].v * ws[i];
              s_w[j] = ws[i];
            } else if constexpr (NC == 0) {
              s_v[j] = q[i].v;
            }
            s_g[j] = 2 * key[i] + sgc[i];
            if constexpr (NC > 0) {
              // a sample's channels are kVB values apart; slots past nchan hold 0
              const uint16_t* v = O.vs + (size_t)(src[i] / kVB) * O.nchan * kVB + (src[i] % kVB);
#pragma unroll
              for (uint32_t ch = 0; ch < (uint32_t)NC; ++ch) s_c[j * NC + ch] = ch < O.nchan ? v[ch * kVB] : (uint16_t)0;
            }
          }
        }
      }
      tile_sync();
      for (; in; in &= in - 1) {  // the chunk's rings, uniform
        const uint32_t k = (uint32_t)__ffsll((unsigned long long)in) - 1u;
        const uint32_t r = rb + k;
        const uint32_t off = __builtin_amdgcn_readlane(seg_off, k), n_r = __builtin_amdgcn_readlane(seg_len, k);
        // this lane's cell's window in the ring
        bool act = r >= win.uring && r <= win.dring;
        uint32_t wl = hl0, wh = hh0;
        if (!(belt_ok && r > ns && r < 3 * ns)) {  // uniform
          const uint32_t kr = r - m.firstring;
          uint64_t ab;
          if constexpr (SHARED)  // (held there, not in registers through the sample loop)
            ab = ring_window_call(hpx32(P.hp), sh->win[lane], sh->tl[lane], sh->tr[lane], r, B.ring_z[kr], B.ring_s[kr]);
          else
            ab = ring_window_call(hpx32(P.hp), win, tl, tr, r, B.ring_z[kr], B.ring_s[kr]);
          const uint32_t a = (uint32_t)ab, b = (uint32_t)(ab >> 32);
          act = act && a <= b;
          wl = 2 * a + (uint32_t)__builtin_amdgcn_readlane(gc, k);
          wh = 2 * b + (uint32_t)__builtin_amdgcn_readlane(gc, k);
        }
        // narrowed to what the radius reaches (the windows are as wide as the
        // disc in every ring): the pass of 20M samples onto 2048^2 4.45 ->
        // 4.32 ms, a 5 sigma beam with weights onto 347^2 1.27 -> 1.19
        {
          const auto of_ring = [&](float RingChord::*m) {
            return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, chord_r.*m), k));
          };
          const CellReach reach = chord_cell(of_ring, zf, ttf);
          act = act && reach.any;
          if (reach.narrow) {
            wl = max(wl, (uint32_t)reach.xl);
            wh = min(wh, (uint32_t)reach.xh);
          }
          act = act && wl <= wh;
        }
        const uint64_t live = __ballot(act);
        if (live == 0) continue;  // uniform
        uint32_t hl[ROWS], hw[ROWS];
        quad_all(act ? wl : kNoWindow, hl);
        quad_all(act ? wh - wl : 0u, hw);
        // the column's samples: all of a short segment, else from the first
        // lower edge to the last upper edge of its four cells (lanes 0 and 1
        // of the quad search the one, 2 and 3 the other)
        uint32_t jb = off, je = off + n_r;
        if (n_r > kShortRing) {
          uint32_t lo = act ? wl : 0xFFFFFFFFu, hi = act ? wh + 1 : 0u;
          lo = min(lo, quad_u32<kQuadXor1>(lo));
          lo = min(lo, quad_u32<kQuadXor2>(lo));
          hi = max(hi, quad_u32<kQuadXor1>(hi));
          hi = max(hi, quad_u32<kQuadXor2>(hi));
          const uint32_t at = band_search(s_g, off, n_r, phase < 2 ? lo : hi);
          jb = quad_u32<quad_bcast(0)>(at);
          je = quad_u32<quad_bcast(2)>(at);
        }
        constexpr uint64_t kRow = ROWS == 1 ? ~0ull : ROWS == 2 ? 0x5555555555555555ull : 0x1111111111111111ull;
        const uint32_t src0 = (uint32_t)__builtin_amdgcn_readlane(seg_src, k) - off;  // sorted index of position 0
        for (uint32_t j = jb + phase; j < je; j += kPhases) {
          const double qx = s_x[j], qy = s_y[j], qz = s_z[j];
          const uint32_t qg = s_g[j];
          double qv = 0.0, qw = 1.0;
          if constexpr (NC == 0) qv = s_v[j];
          if constexpr (HAS_W) qw = s_w[j];
          float cv[NC > 0 ? NC : 1];
          if constexpr (NC > 0) {
            // two channels per 32-bit LDS word; the value type is the job's (a uniform branch)
            const uint32_t* w2 = reinterpret_cast<const uint32_t*>(s_c + j * NC);
#pragma unroll
            for (int h = 0; h < NC / 2; ++h) {
              const uint32_t u = w2[h];
              if (O.bf16) {
                cv[2 * h] = __uint_as_float(u << 16);
                cv[2 * h + 1] = __uint_as_float(u & 0xFFFF0000u);
              } else {
                cv[2 * h] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u & 0xFFFFu));
                cv[2 * h + 1] = (float)__builtin_bit_cast(_Float16, (uint16_t)(u >> 16));
              }
            }
          }
#pragma unroll
          for (int k = 0; k < ROWS; ++k) {
            if ((live & (kRow << k)) == 0) continue;  // uniform: the ring is out of this row's reach
            double t;  // the tested distance: h = 1 - p.q (WMODE 3) or c2 = |p - q|^2
            double dx = 0.0, dy = 0.0, dz = 0.0;
            if constexpr (WMODE == 3) {
              t = fma(npx[k], qx, fma(npy[k], qy, fma(npz[k], qz, 1.0)));
            } else {
              dx = npx[k] + qx, dy = npy[k] + qy, dz = npz[k] + qz;
              t = fma(dx, dx, fma(dy, dy, dz * dz));
            }
            if (qg - hl[k] <= hw[k] && (kHigh ? high_f32(t) <= t_hi32 : t < t_hi)) {
              const uint32_t cell = (row0 + (uint32_t)k) * P.side + col, isrc = src0 + j;
              double wt;
              if constexpr (WMODE == 3)
                wt = gauss_weight_lean(t, k0h, k1v, e3v, s_exp);
              else if constexpr (kFrame)
                wt = gauss2d_frame_weight<WMODE == 5>(
                    P, t, fma(dx, fu[k][0], fma(dy, fu[k][1], dz * fu[k][2])),
                    fma(dx, fv[k][0], fma(dy, fv[k][1], dz * fv[k][2])), s_exp);
              else if constexpr (WMODE == 4)
                wt = sinc_frame_weight(P, t, s_exp);
              else if constexpr (KT == HCG_GAUSS1D && WMODE > 0)
                wt = gauss_weight_series<WMODE>(P, t, s_exp);
              else if constexpr (KT == HCG_GAUSS1D)
                wt = exp_scaled_neg(gauss_exponent_scaled(P, t), s_exp);
              else
                wt = weight_general<KT>(P.params[0], P.params[1], P.params[2], B.xwcs, B.ywcs, B.lon_s, B.lat_s,
                                        0.25 * t, cell, isrc);
              // lanes near the radius (rare, and wave-uniformly skipped): the
              // reference's test decides, and a pair that it rejects adds
              // nothing, whatever its value and sample weight are
              const bool near =
                  __builtin_amdgcn_ballot_w64(!(kHigh ? high_f32(t) < t_lo32 : t < t_lo)) != 0;  // uniform
              const auto inside = [&]() {
                return t < t_lo ||
                       (t < t_hi && radius_test_ref(B.xwcs, B.ywcs, B.lon_s, B.lat_s, cell, isrc, P.sphere_radius));
              };
              if constexpr (NC > 0) {
                // (zeroed copies of the channels' values would take registers)
                bool in = true;
                if (near) {
                  asm volatile("; guard band" ::);
                  in = inside();
                }
                if (in) {
                  const float wf = (float)wt;
#pragma unroll
                  for (int c = 0; c < NC; ++c) acc_c[k][c] = fmaf(wf, cv[c], acc_c[k][c]);
                  acc_w[k] += wt;
                }
              } else {
                // a rejected lane adds zero: one compare and no lane mask in
                // the common case (sums under a mask, as above, cost 6% on
                // 20M samples; the weight's copy 1.5% on weighted maps)
                double vv = qv, ww = qw;
                if (near) {
                  // (a block of its own, so the branch above stays a scalar one)
                  asm volatile("; guard band" ::);
                  if (!inside()) wt = vv = ww = 0.0;
                }
                acc_d[k] = fma(vv, wt, acc_d[k]);
                if constexpr (HAS_W)
                  acc_w[k] = fma(ww, wt, acc_w[k]);
                else
                  acc_w[k] += wt;
              }
            }
          }
        }
      }
    }
  }
  out.w = quad_rows_sum(acc_w, row);
  if constexpr (NC > 0) {
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      float v[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) v[r] = acc_c[r][c];
      out.c[c] = quad_rows_sum(v, row);
    }
  } else {
    out.d = quad_rows_sum(acc_d, row);
  }
}

// The map cell whose sums this lane holds; false for none.
template <int ROWS = kTileRows>
__device__ inline bool tile_cell(uint32_t side, uint32_t tile, uint32_t tiles_x, uint32_t& cell) {
  const uint32_t lane = __lane_id();
  const uint32_t col = (tile % tiles_x) * kTileCols + (lane >> 2);
  const uint32_t row = (tile / tiles_x) * ROWS + (lane & 3u);
  cell = row * side + col;
  return col < side && row < side && (lane & 3u) < (uint32_t)ROWS;
}

// The FP32 outputs of one one-channel tile cell (lane) from its sums.
__device__ inline void tile_write(const GridParams& P, uint32_t tile, uint32_t tiles_x, const TileOut& O, double d,
                                  double w) {
  uint32_t cell;
  if (tile_cell(P.side, tile, tiles_x, cell)) {
    O.cube[cell] = O.normalize ? (float)(d / w) : (float)d;
    if (O.wsum) O.wsum[cell] = (float)w;
  }
}

// LDS of one_channel_tile: `active` staging slices, then the streams' sums
// when there are several.
constexpr size_t one_channel_lds_bytes(uint32_t active, uint32_t streams) {
  return active * kTileLdsBytes + (streams > 1 ? (size_t)streams * 64 * 2 * sizeof(double) : 0);
}

// One one-channel tile over `streams` partial streams: waves w < active of
// the workgroup walk streams w, w + active, ... in their own kTileLdsBytes
// slice of `lds`; the streams' sums meet after the slices and wave 0 adds
// them in stream order and writes the cells.  Every wave of the workgroup
// calls this (it holds a workgroup barrier when streams > 1).
template <int WMODE>
__device__ __forceinline__ void one_channel_tile(const GridParams& P, const GridBuffers& B, const TileOut& O,
                                                 uint32_t tile, uint32_t tiles_x, uint32_t streams, uint32_t active,
                                                 char* lds, const double* s_exp) {
  const uint32_t wave = threadIdx.x >> 6, lane = __lane_id();
  double* red = reinterpret_cast<double*>(lds + active * kTileLdsBytes);
  TileSums<0> s{};
  if (wave < active) {
    for (uint32_t q = wave; q < streams; q += active) {
      grid_tile<HCG_GAUSS1D, false, WMODE, true, 0, kOneCap>(P, B, tile, tiles_x, lds + wave * kTileLdsBytes, s_exp,
                                                               O, RingStream{q, streams}, s);
      if (streams > 1) {
        red[(q * 64 + lane) * 2] = s.d;
        red[(q * 64 + lane) * 2 + 1] = s.w;
      }
    }
  }
  if (streams > 1) {
    __syncthreads();
    if (wave == 0) {
      s.d = red[lane * 2];
      s.w = red[lane * 2 + 1];
      for (uint32_t q = 1; q < streams; ++q) {
        s.d += red[(q * 64 + lane) * 2];
        s.w += red[(q * 64 + lane) * 2 + 1];
      }
    }
  }
  if (wave == 0) tile_write(P, tile, tiles_x, O, s.d, s.w);
}

// One few-channel tile in a kFewTileLdsBytes slice of LDS (one wave).
__device__ __forceinline__ void few_channel_tile_body(const GridParams& P, const GridBuffers& B, const TileOut& O,
                                                      uint32_t tile, uint32_t tiles_x, char* lds,
                                                      const double* s_exp) {
  TileSums<kFewChannels> s;
  grid_tile<HCG_GAUSS1D, false, 3, true, kFewChannels, kFewCap>(P, B, tile, tiles_x, lds, s_exp, O, RingStream{0, 1},
                                                                s);
  uint32_t cell;
  if (tile_cell(P.side, tile, tiles_x, cell)) {
    const size_t M = (size_t)P.side * P.side;
#pragma unroll
    for (int ch = 0; ch < kFewChannels; ++ch)
      if ((uint32_t)ch < O.nchan)
        O.cube[(size_t)ch * M + cell] = O.normalize ? (float)((double)s.c[ch] / s.w) : s.c[ch];
    if (O.wsum) O.wsum[cell] = (float)s.w;
  }
}

}  // namespace hcg
