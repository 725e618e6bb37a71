// mfma_kernels.hpp -- multi-channel gridding as a dense MFMA contraction.  The
// kernel's instances are built in one file for each group of weight kinds
// (grid_mfma.hip, mfma_gauss.hip, mfma_gauss2d_sinc.hip): in parallel, and a
// process loads those that it uses.
//
// The reference grids a spectral cube one channel at a time, rerunning the
// full single-channel kernel per channel on its own stream
// (HCGrid+/gridding-omp.cu:552-678, kernel HCGrid+/gridding-omp.cu:294-420).
// The selection and weights do not depend on the channel, so here they are
// computed once per (cell, sample) pair in FP64 and the channel sums become
//     cube[ch][cell] = sum_s W[cell][s] * V[ch][s]   (FP32 accumulation)
// evaluated with v_mfma_f32_16x16x32_{bf16,f16}.  Each FP64 weight is carried
// as hi + lo, two values of the channel type (hi = round(w), lo = round(w -
// hi)), and both are contracted: the weight keeps ~2x the type's significand
// (relative error ~2^-17 for BF16) at twice the MFMA count.
//
// A workgroup owns a block of 64 cells, four squares of 16.  A square's
// samples are the 8-sample blocks of its rings' sorted ranges, each ring
// narrowed to its windows and to what the radius reaches; 32 at a time
// (a k-block) they are staged in LDS, and lane l evaluates the weights of
// cell l % 16 and samples 8 (l / 16) .. + 7: exactly its A operand, in
// registers, every pair of the 16 x 32 (45% of them selected on rasters of
// two and more samples per cell).  mfma_tile is a wave per square, without
// barriers, for up to 256 channels; mfma_wide shares a block's weights over
// 512 channels through LDS.  Both come for each kind of weight
// (mfma_weight_kind).
//
// What counts is vector instructions (FP64 weights), then the latency of the
// LDS reads and weight chains at two to four waves per SIMD.  Before, weights
// went through a row-major LDS tile (cleared, each cell's band searched and
// filled by lane = cell, 44% of the lanes on selected pairs) between four
// workgroup barriers per 128-512 samples, one wave contracting while the
// rest waited on small jobs.  A pass before and now: 195k samples x 3
// channels onto 500^2 911 -> 190 us; 482k x 67 onto 511^2 1316 -> 413 us;
// 300k x 16 onto 2048^2 3337 -> 1370 us; 1.2M x 64 onto 512^2 (new
// coordinates) 2697 -> 1522 us; 2M x 1024 onto 1024^2 9526 -> 8200 us (this
// kernel 7.40 -> 6.0 ms: 1.34e9 vector and 1.9e8 MFMA instructions at two
// waves per SIMD).
//
// Selection, FP64 distance and weight follow the single-channel kernel
// exactly; only the products with channel values run in BF16/FP16.
#pragma once

#include <hip/hip_runtime.h>

#include "gridcore.hpp"
#include "mfma_job.hpp"

namespace hcg {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2_t __attribute__((ext_vector_type(2)));


typedef short s16x8_t __attribute__((ext_vector_type(8)));  // a raw 16-byte MFMA operand

// Channel type of a kernel instance.  Values and weights are kept as raw
// 16-bit words; the type matters only where a weight is rounded and where
// the MFMA issues.
enum : int { kDtBf16 = 0, kDtF16 = 1 };

__device__ inline f32x4_t mfma16(bool bf, s16x8_t a, s16x8_t b, f32x4_t c) {
  if (bf)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b),
                                                   c, 0, 0, 0);
  return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c,
                                                0, 0, 0);
}

// FP64 weight of a selected pair by calls (the single-channel kernel's general evaluation).
__device__ inline double pair_weight_call(const GridParams& P, const GridBuffers& B, uint32_t kt, double c2,
                                          const double* s_exp, uint32_t cell, uint32_t i) {
  if (kt == HCG_GAUSS1D) return exp_scaled_neg(gauss_exponent_scaled(P, c2), s_exp);
  if (kt == HCG_GAUSS2D)
    return weight_general<HCG_GAUSS2D>(P.params[0], P.params[1], P.params[2], B.xwcs, B.ywcs, B.lon_s, B.lat_s,
                                       0.25 * c2, cell, i);
  return weight_general<HCG_TAPERED_SINC>(P.params[0], P.params[1], P.params[2], B.xwcs, B.ywcs, B.lon_s,
                                          B.lat_s, 0.25 * c2, cell, i);
}

// FP64 weights of two pairs from series (garbage where a pair is not selected):
// (dx, dy, dz) = q - p, fu and fv the cell's tangent frame (kWeight2d).
template <uint32_t WK>
__device__ __forceinline__ void pair_weights_series(const GridParams& P, const double (&c2)[2], const double (&dx)[2],
                                                    const double (&dy)[2], const double (&dz)[2],
                                                    const double (&fu)[3], const double (&fv)[3],
                                                    const double* s_exp, double (&wt)[2]) {
  double y[2], amp[2] = {1.0, 1.0};
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    if constexpr (WK == kWeightSmall) {
      y[e] = gauss_exponent_series(P, c2[e]);
    } else if constexpr (WK == kWeight2d) {
      const double U = fma(dx[e], fu[0], fma(dy[e], fu[1], dz[e] * fu[2]));
      const double V = fma(dx[e], fv[0], fma(dy[e], fv[1], dz[e] * fv[2]));
      y[e] = distance_series<true>(c2[e]) * fma(P.f[0] * U, U, (P.f[1] * V) * V);
    } else {
      const double d2 = c2[e] * distance_series<false>(c2[e]);
      y[e] = (WK == kWeightSinc ? P.f[1] : P.k0) * d2;
      if constexpr (WK == kWeightSinc) amp[e] = sinc_triple(P.f[0] * d2);
    }
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    // (kWeightSmall's exponents are above the clamp)
    wt[e] = WK == kWeightSmall ? exp_scaled_neg_fold(y[e], s_exp) : exp_scaled_neg(y[e], s_exp);
    if constexpr (WK == kWeightSinc) wt[e] *= amp[e];
  }
}

// The tested distance of a pair: h = 1 - p.q (LEAN), or c2 = |p - q|^2 (np = -p).
template <bool LEAN>
__device__ inline double pair_distance(double npx, double npy, double npz, double x, double y, double z) {
  if constexpr (LEAN) return fma(npx, x, fma(npy, y, fma(npz, z, 1.0)));
  const double dx = npx + x, dy = npy + y, dz = npz + z;
  return fma(dx, dx, fma(dy, dy, dz * dz));
}

// Four consecutive doubles (32-byte aligned), two 16-byte reads.
__device__ inline void lds_read4(const double* p, double (&v)[4]) {
  const double2 a = *reinterpret_cast<const double2*>(p), b = *reinterpret_cast<const double2*>(p + 2);
  v[0] = a.x;
  v[1] = a.y;
  v[2] = b.x;
  v[3] = b.y;
}

// Two FP32 values rounded to 16 bits (nearest even) in one word, and back.
template <bool BF>
__device__ inline uint32_t round16x2(f32x2_t v) {
  if constexpr (BF)
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
  else
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, f16x2_t));
}
template <bool BF>
__device__ inline f32x2_t widen16x2(uint32_t w) {
  if constexpr (BF)
    return f32x2_t{__uint_as_float(w << 16), __uint_as_float(w & 0xFFFF0000u)};
  else
    return __builtin_convertvector(__builtin_bit_cast(f16x2_t, w), f32x2_t);
}

// A set of cells taken together (block_ring_range).
struct BlockSpan {
  TileSpan T;
  bool simple;          // every window is one pair of half-pixel numbers (belt_window), every ring a belt ring
  uint32_t hlo, hhi;    // simple: the outermost of them
};

constexpr uint32_t kNoRingLane = 255;        // the ring lane of a block list's padding
constexpr uint32_t kNoSample = 0x40000000u;  // half-pixel position that no window holds

// NS staged samples.
template <uint32_t NS, uint32_t WK>
struct Staged {
  __attribute__((aligned(16))) double x[NS], y[NS], z[NS];
  __attribute__((aligned(16))) double w[WK == kWeightLean ? 2 : NS];  // sample weights
  __attribute__((aligned(16))) uint32_t g[NS];  // half-pixel positions
};

// The value blocks that a set of cells looks at, for 64 rings (lane = ring),
// listed NL (a multiple of 4) at a time.
template <uint32_t NL>
struct BlockList {
  uint32_t lb[NL];         // listed block: its index among the sorted 8-sample blocks
  double rz[64], rs[64];   // ring_z, ring_s
  uint32_t gc[64];         // half-pixel position of a sample: 2 key + gc
  uint32_t b0[64], ex[64], nb[64];  // the ring's first value block, their place in the sequence, their number
  BlockSpan span;
  uint8_t lr[NL];          // listed block: its ring's lane
};

// A block's 64 cells, row by row.
struct MfmaCells {
  Window win[kMcCols];
  double tl[kMcCols], tr[kMcCols];  // compat: the window's edges (compat_edges)
  double p[3][kMcCols];
  double coslat[kMcCols], tt[kMcCols];
  uint32_t wlo[kMcCols], wwid[kMcCols];           // the window in every belt ring (belt_window)
  uint8_t belt[kMcCols];                          // it holds
};

// The cells' tangent frames (kWeight2d): east and north turned by the position angle.
template <uint32_t WK>
struct MfmaFrames {
  double u[3][WK == kWeight2d ? kMcCols : 1], v[3][WK == kWeight2d ? kMcCols : 1];
};

// One wave's LDS: a staged k-block and its list.
template <uint32_t WK>
struct MfmaWave {
  Staged<32, WK> st;
  BlockList<128> bl;
};
template <uint32_t WK>
union MfmaLds {
  struct {
    MfmaWave<WK> w[kMcWaves];
    MfmaCells c;
    MfmaFrames<WK> f;
  } s;
  float t[kMcCols * 64];  // the epilogue's 64 channels x 64 cells
};

// The square's set-up runs once per 64 rings and the windows of general rings
// once per k-block, both next to the sample loop: out of line, so that their
// constants and temporaries do not live in its registers (230 of them inline
// against 100).  Ranges come back as first | last << 32, 1 | 0 for none.
constexpr uint64_t kNoRange = 1;
__device__ inline uint64_t pack_range(uint32_t lp, uint32_t rp) { return (uint64_t)rp << 32 | lp; }

static __device__ __noinline__ uint64_t span_pixels_call(Hpx32 hx, TileSpan t, uint32_t ring, double rz, double rs) {
  uint32_t lp, rp;
  span_pixels(hx, t, ring, rz, rs, lp, rp);
  return pack_range(lp, rp);
}

static __device__ __noinline__ uint64_t cell_window_call(Hpx32 hx, const MfmaCells* C, uint32_t cb, uint32_t ring,
                                                         double rz, double rs) {
  uint32_t a = 1, b = 0;
  if (!ring_window_at(hx, C->win[cb], C->tl[cb], C->tr[cb], ring, rz, rs, a, b)) return kNoRange;
  return pack_range(a, b);
}

// The keys of ring `ring` that a square's cells can take samples from: a
// superset of the samples both in a cell's window and within its radius.
__device__ inline uint64_t block_ring_range(const GridParams& P, const GridBuffers& B, const BlockSpan& S,
                                            const hcg_ring_meta& m, uint32_t ring) {
  const uint32_t kr = ring - m.firstring;
  const Hpx32 hx = hpx32(P.hp);
  uint32_t sp, npr;
  ring_info32(hx, ring, sp, npr);
  uint32_t lp, rp;
  if (S.simple) {  // g = 2 p + 1 - odd in [hlo, hhi]
    const uint32_t odd = ring & 1u;
    lp = sp + ((S.hlo + odd) >> 1);
    rp = sp + ((S.hhi - 1u + odd) >> 1);
  } else {
    const uint64_t range = span_pixels_call(hx, S.T, ring, B.ring_z[kr], B.ring_s[kr]);
    lp = (uint32_t)range;
    rp = (uint32_t)(range >> 32);
  }
  return chord_pixels(S.T, ring_chord(P.polar_half * P.polar_half, S.T, npr, kr, m.usedrings, B.ring_z), sp, npr, lp, rp) ? pack_range(lp, rp)
                                                                                              : kNoRange;
}

// A cell (a lane's) of a block.
struct CellGeom {
  Window win;
  double tl, tr;              // compat: the window's edges (compat_edges)
  double px, py, pz;          // unit vector
  double coslat, tt;          // cos of the latitude; longitude (units of pi/2)
  uint32_t wlo, wwid;         // the window in every belt ring (belt_window)
  bool belt;                  // it holds
};

// Lane = cell of the block at (y0, x0), row by row.
__device__ __forceinline__ CellGeom block_cell(const GridParams& P, const GridBuffers& B, const hcg_ring_meta& m,
                                               uint32_t y0, uint32_t x0, uint32_t tc_shift, bool& live) {
  const uint32_t lane = __lane_id();
  const uint32_t row = y0 + (lane >> tc_shift), col = x0 + (lane & ((1u << tc_shift) - 1u));
  live = row < P.side && col < P.side;
  const uint32_t cell = live ? row * P.side + col : 0;
  const uint32_t anchor = live ? row * P.side + (col / P.factor) * P.factor : 0;
  const double xc = B.xwcs[cell] * kDeg2Rad, yc = B.ywcs[cell] * kDeg2Rad;
  CellGeom g;
  g.win = window_of(P, m.firstring, m.usedrings, B.xwcs[anchor], B.ywcs[anchor]);
  if (!live || m.usedrings == 0) {
    g.win.uring = 1;
    g.win.dring = 0;
  }
  double cb, sl, cl;
  sincos(yc, &g.pz, &cb);
  sincos(xc, &sl, &cl);
  g.px = cb * cl;
  g.py = cb * sl;
  g.tl = g.tr = 0.0;
  uint32_t whi = 0;
  g.wlo = 0;
  g.belt = false;
  if (g.win.mode == kWinCompat) {
    compat_edges(P, g.win, g.tl, g.tr);
    g.belt = belt_window(P, g.tl, g.tr, g.wlo, whi);
  }
  g.wwid = whi - g.wlo;
  g.coslat = cb;
  g.tt = fmodulo4(xc * kInvHalfPi);
  return g;
}

__device__ __forceinline__ void put_cell(MfmaCells& C, uint32_t i, const CellGeom& g) {
  C.win[i] = g.win;
  C.tl[i] = g.tl;
  C.tr[i] = g.tr;
  C.p[0][i] = g.px;
  C.p[1][i] = g.py;
  C.p[2][i] = g.pz;
  C.coslat[i] = g.coslat;
  C.tt[i] = g.tt;
  C.wlo[i] = g.wlo;
  C.wwid[i] = g.wwid;
  C.belt[i] = g.belt;
}

// Lane = cell of the block, as block_cell.
template <uint32_t WK>
__device__ __forceinline__ void put_frames(const MfmaJob& J, MfmaFrames<WK>& F, uint32_t y0, uint32_t x0) {
  if constexpr (WK == kWeight2d) {
    const GridParams& P = J.P;
    const uint32_t lane = __lane_id();
    const uint32_t row = min(y0 + (lane >> J.tc_shift), P.side - 1);
    const uint32_t col = min(x0 + (lane & ((1u << J.tc_shift) - 1u)), P.side - 1);
    double sl, cl, sb, cb;
    sincos(J.B.xwcs[row * P.side + col] * kDeg2Rad, &sl, &cl);
    sincos(J.B.ywcs[row * P.side + col] * kDeg2Rad, &sb, &cb);
    const double e[3] = {-sl, cl, 0.0}, nn[3] = {-sb * cl, -sb * sl, cb};
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      F.u[i][lane] = fma(e[i], P.f[2], -(nn[i] * P.f[3]));
      F.v[i][lane] = fma(nn[i], P.f[2], e[i] * P.f[3]);
    }
  }
}

// The span of the wave's cells.
__device__ __forceinline__ BlockSpan cells_span(const GridParams& P, const hcg_ring_meta& m, const CellGeom& g) {
  BlockSpan S;
  S.T = tile_span(P, g.win, m.firstring, g.pz, g.coslat, g.tt);
  const bool has = g.win.uring <= g.win.dring;
  const uint32_t ns = (uint32_t)P.hp.nside;
  const bool belt_ok = __ballot(has && !g.belt) == 0;
  S.simple = belt_ok && S.T.r_begin > ns && S.T.r_end < 3 * ns;  // uniform
  S.hlo = wave_min_u32(has ? g.wlo : 0xFFFFFFFFu);
  S.hhi = wave_max_u32(has ? g.wlo + g.wwid : 1u);
  return S;
}

// The value blocks [b0, b0 + nblk) of ring r of a span (lane = ring).
__device__ __forceinline__ void ring_block_range(const GridParams& P, const GridBuffers& B, const hcg_ring_meta& m,
                                                 const BlockSpan& S, uint32_t r, uint32_t& b0, uint32_t& nblk) {
  b0 = nblk = 0;
  if (r > S.T.r_end) return;
  const uint32_t kr = r - m.firstring;
  const uint32_t start = B.lut[kr], end = B.lut[kr + 1];
  if (start >= end) return;
  const uint64_t range = block_ring_range(P, B, S, m, r);
  const uint32_t lp = (uint32_t)range, rp = (uint32_t)(range >> 32);
  uint32_t lo = 0, hi = 0;
  if (lp <= rp) key_range(B.keys, start, end, lp, rp, lo, hi);
  if (lo < hi) {
    b0 = lo / kVB;
    nblk = (hi + kVB - 1) / kVB - b0;
  }
}

__device__ __forceinline__ uint32_t wave_scan_sum_u32(uint32_t v) {  // inclusive
  const uint32_t lane = __lane_id();
#pragma unroll
  for (uint32_t off = 1; off < 64; off <<= 1) {
    const uint32_t t = __shfl_up(v, off, 64);
    if (lane >= off) v += t;
  }
  return v;
}

// Rings rb .. rb + 63 of the list's span (lane = ring, one wave) with their
// value blocks; the blocks' number.
template <uint32_t NL>
__device__ __forceinline__ uint32_t put_rings(const GridParams& P, BlockList<NL>& L, uint32_t rb, uint32_t b0,
                                              uint32_t nblk) {
  const uint32_t lane = __lane_id(), r = rb + lane;
  uint32_t sp, npr;
  ring_info32(hpx32(P.hp), r, sp, npr);
  L.gc[lane] = 1u - (r & 1u) - 2u * sp;
  const uint32_t in = wave_scan_sum_u32(nblk);
  L.b0[lane] = b0;
  L.ex[lane] = in - nblk;
  L.nb[lane] = nblk;
  return (uint32_t)__builtin_amdgcn_readlane((int)in, 63);
}
template <uint32_t NL>
__device__ __forceinline__ uint32_t ring_blocks(const GridParams& P, const GridBuffers& B, const hcg_ring_meta& m,
                                                uint32_t rb, BlockList<NL>& L) {
  const uint32_t lane = __lane_id(), r = rb + lane;
  uint32_t b0, nblk;
  ring_block_range(P, B, m, L.span, r, b0, nblk);
  if (r <= L.span.T.r_end) {
    L.rz[lane] = B.ring_z[r - m.firstring];
    L.rs[lane] = B.ring_s[r - m.firstring];
  }
  return put_rings(P, L, rb, b0, nblk);
}

// The plan of a block for mfma_wide: what its set-up works out, in one
// coalesced read (set up in the kernel, one wave at work and seven waiting,
// the 2M x 1024 cube's 32768 blocks took 0.8 ms more).  ok: the span is
// simple and has at most 64 rings; otherwise the kernel does the set-up.
struct MfmaPlan {
  double p[3][kMcCols];
  uint32_t uring[kMcCols], dring[kMcCols], wlo[kMcCols], wwid[kMcCols];  // cell by cell
  uint32_t b0[64], nb[64];                                              // ring by ring
  uint32_t ok, r_begin, r_end, pad;
};
static_assert(sizeof(MfmaPlan) <= kPlanBytes && kPlanBytes % 8 == 0, "plan layout");
__device__ __forceinline__ void plan_tile(const MfmaJob& J, uint32_t tile) {  // one wave
  const uint32_t lane = __lane_id();
  const hcg_ring_meta m = *J.B.meta;
  bool live;
  const CellGeom g = block_cell(J.P, J.B, m, (tile / J.tiles_x) << (6u - J.tc_shift),
                                (tile % J.tiles_x) << J.tc_shift, J.tc_shift, live);
  const BlockSpan S = cells_span(J.P, m, g);
  MfmaPlan& L = *reinterpret_cast<MfmaPlan*>(static_cast<char*>(J.plan) + tile * kPlanBytes);
  const bool none = S.T.r_begin > S.T.r_end, ok = none || (S.simple && S.T.r_end - S.T.r_begin < 64);
  if (lane == 0) {
    L.ok = ok;
    L.r_begin = none ? 1 : S.T.r_begin;
    L.r_end = none ? 0 : S.T.r_end;
  }
  if (!ok) return;  // uniform
  L.p[0][lane] = g.px;
  L.p[1][lane] = g.py;
  L.p[2][lane] = g.pz;
  L.uring[lane] = g.win.uring;
  L.dring[lane] = g.win.dring;
  L.wlo[lane] = g.wlo;
  L.wwid[lane] = g.wwid;
  uint32_t b0 = 0, nblk = 0;
  if (!none) ring_block_range(J.P, J.B, m, S, S.T.r_begin + lane, b0, nblk);
  L.b0[lane] = b0;
  L.nb[lane] = nblk;
}

// Lists blocks q0 .. q0 + cnt - 1 (one wave), then the last one again up to
// the k-block boundary, as padding without samples.
template <uint32_t NL>
__device__ __forceinline__ void list_blocks(BlockList<NL>& L, uint32_t q0, uint32_t cnt) {
  const uint32_t lane = __lane_id();
  const uint32_t ex = L.ex[lane], in = ex + L.nb[lane], b = L.b0[lane] - ex;
  for (uint32_t t = max(ex, q0); t < min(in, q0 + cnt); ++t) {
    L.lb[t - q0] = b + t;
    L.lr[t - q0] = (uint8_t)lane;
    if (t - q0 == cnt - 1)
      for (uint32_t p = cnt; p < (cnt + 3) / 4 * 4; ++p) {
        L.lb[p] = b + t;
        L.lr[p] = (uint8_t)kNoRingLane;
      }
  }
}

// Sample s of k-block u of the list, half of it a lane: half 0 its x, y and
// sample weight (if there are any), half 1 its z and position; in flight from
// fetch to store.
template <uint32_t WK>
struct StageRegs {
  double v0, v1, w;
  uint32_t pos;
  template <uint32_t NL>
  __device__ __forceinline__ void fetch(const GridBuffers& B, const hcg_ring_meta& m, const BlockList<NL>& L,
                                        uint32_t u, uint32_t s, uint32_t half) {
    const uint32_t q = u * 4 + (s >> 3);
    const uint32_t i = L.lb[q] * kVB + (s & 7u), rl = L.lr[q];
    v0 = v1 = w = 0.0;
    pos = kNoSample;
    if (rl != kNoRingLane && i < m.n) {
      const double* r = &B.rec[i].x + 2 * half;
      v0 = r[0];
      v1 = r[1];
      if (half) pos = 2u * B.keys[i] + L.gc[rl];
      if constexpr (WK != kWeightLean)
        if (B.w_s && !half) w = B.w_s[i];
    }
  }
  template <uint32_t NS>
  __device__ __forceinline__ void store(Staged<NS, WK>& S, uint32_t p, uint32_t half) const {
    if (half) {
      S.z[p] = v0;
      S.g[p] = pos;
    } else {
      S.x[p] = v0;
      S.y[p] = v1;
      if constexpr (WK != kWeightLean) S.w[p] = w;
    }
  }
};

// One lane's cell of a square, and the constants of the weights.
template <uint32_t WK>
struct SquareCell {
  static constexpr bool LEAN = WK == kWeightLean;
  double npx, npy, npz;
  uint32_t uring, dring, wlo, wwid;
  double h_hi, h_lo, k0h, k1v, e3v;
  double wsum;
  uint32_t cb;  // its place in the block
  bool simple;
  __device__ __forceinline__ void init(const GridParams& P, const MfmaCells& C, uint32_t cell_in_block, bool smp) {
    cb = cell_in_block;
    simple = smp;
    npx = -C.p[0][cb];
    npy = -C.p[1][cb];
    npz = -C.p[2][cb];
    uring = C.win[cb].uring;
    dring = C.win[cb].dring;
    wlo = C.wlo[cb];
    wwid = C.wwid[cb];
    h_hi = LEAN ? 0.5 * P.c_hi : P.c_hi;
    h_lo = LEAN ? 0.5 * P.c_lo : P.c_lo;
    k0h = 2.0 * P.k0;
    k1v = LEAN ? in_vgprs(4.0 * P.k1) : 0.0;
    e3v = LEAN ? in_vgprs(kExpE3) : 0.0;
    wsum = 0.0;
  }
  // the window in ring lane rl of the list, in half pixels
  template <uint32_t NL>
  __device__ __forceinline__ void window(const GridParams& P, const MfmaCells& C, const BlockList<NL>& L, uint32_t rb,
                                         uint32_t rl, uint32_t& wl, uint32_t& ww) const {
    const uint32_t r = rb + rl;
    bool act = rl != kNoRingLane && r >= uring && r <= dring;
    wl = wlo;
    ww = wwid;
    if (!simple) {  // uniform
      const uint64_t range = cell_window_call(hpx32(P.hp), &C, cb, r, L.rz[rl & 63u], L.rs[rl & 63u]);
      const uint32_t a = (uint32_t)range, b = (uint32_t)(range >> 32);
      act = act && a <= b;
      wl = 2u * a + L.gc[rl & 63u];
      ww = 2u * (b - a);
    }
    if (!act) {
      wl = kNoWindow;
      ww = 0;
    }
  }
};

// One lane's A operand: the weights of 8 samples, hi and lo.
struct WeightOperand {
  union {
    uint32_t d[4];
    s16x8_t v;
  } h, l;
};

// The weights of a wave's 16 cells and the 32 samples at S[at ..]: lane l
// takes cell l % 16 and samples 8 (l / 16) .. + 7 (of value block blk), which
// is the layout of an MFMA operand.  Returns the lanes with a selected pair;
// guard: those with one within rounding of the radius (kept here).
template <int DT, uint32_t WK, uint32_t NS>
__device__ __forceinline__ uint64_t weigh_kblock(const MfmaJob& J, SquareCell<WK>& Q, const Staged<NS, WK>& S,
                                                 const MfmaFrames<WK>& F, uint32_t at, uint32_t wl, uint32_t ww,
                                                 uint32_t cell, uint32_t blk, const double* s_exp, WeightOperand& A,
                                                 uint64_t& guard) {
  constexpr bool bf = DT == kDtBf16, LEAN = WK == kWeightLean;
  uint64_t any = 0;
  guard = 0;
  double fu[3] = {0.0, 0.0, 0.0}, fv[3] = {0.0, 0.0, 0.0};
  if constexpr (WK == kWeight2d) {
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      fu[i] = F.u[i][Q.cb];
      fv[i] = F.v[i][Q.cb];
    }
  }
#pragma unroll
  for (uint32_t hf = 0; hf < 2; ++hf) {  // four samples at a time
    const uint32_t j0 = at + (__lane_id() >> 4) * 8 + hf * 4;
    double qx[4], qy[4], qz[4], t[4];
    uint32_t qg[4];
    lds_read4(&S.x[j0], qx);
    lds_read4(&S.y[j0], qy);
    lds_read4(&S.z[j0], qz);
    *reinterpret_cast<uint4*>(qg) = *reinterpret_cast<const uint4*>(&S.g[j0]);
    uint64_t sel[4];
#pragma unroll
    for (uint32_t e = 0; e < 4; ++e) {
      t[e] = pair_distance<LEAN>(Q.npx, Q.npy, Q.npz, qx[e], qy[e], qz[e]);
      sel[e] = __builtin_amdgcn_ballot_w64(t[e] < Q.h_hi) & __builtin_amdgcn_ballot_w64(qg[e] - wl <= ww);
      guard |= sel[e] & __builtin_amdgcn_ballot_w64(!(t[e] < Q.h_lo));
    }
    any |= (sel[0] | sel[1]) | (sel[2] | sel[3]);
    double qw[4] = {1.0, 1.0, 1.0, 1.0};
    if constexpr (!LEAN)
      if (J.B.w_s) lds_read4(&S.w[j0], qw);  // uniform
#pragma unroll
    for (uint32_t k = 0; k < 2; ++k) {
      const uint32_t jj = hf * 2 + k;
      A.h.d[jj] = A.l.d[jj] = 0;
      if ((sel[2 * k] | sel[2 * k + 1]) == 0) continue;  // uniform
      // both weights at once, every lane's (two chains of FP64 steps and
      // table reads hide each other's latency), then the selected ones
      double wt[2] = {0.0, 0.0};
      if constexpr (LEAN) {
        gauss_weight_lean2(t[2 * k], t[2 * k + 1], Q.k0h, Q.k1v, Q.e3v, s_exp, wt);
      } else if constexpr (WK != kWeightCall) {
        const double c2[2] = {t[2 * k], t[2 * k + 1]};
        const double dx[2] = {Q.npx + qx[2 * k], Q.npx + qx[2 * k + 1]};
        const double dy[2] = {Q.npy + qy[2 * k], Q.npy + qy[2 * k + 1]};
        const double dz[2] = {Q.npz + qz[2 * k], Q.npz + qz[2 * k + 1]};
        pair_weights_series<WK>(J.P, c2, dx, dy, dz, fu, fv, s_exp, wt);
        if (J.B.w_s) {  // uniform
          wt[0] *= qw[2 * k];
          wt[1] *= qw[2 * k + 1];
        }
      } else {
#pragma unroll
        for (uint32_t e = 0; e < 2; ++e)
          if (__builtin_amdgcn_inverse_ballot_w64(sel[2 * k + e])) {
            wt[e] = pair_weight_call(J.P, J.B, J.kt, t[2 * k + e], s_exp, cell, blk * kVB + jj * 2 + e);
            if (J.B.w_s) wt[e] *= qw[2 * k + e];
          }
      }
      const f32x2_t wf = {__builtin_amdgcn_inverse_ballot_w64(sel[2 * k]) ? (float)wt[0] : 0.f,
                          __builtin_amdgcn_inverse_ballot_w64(sel[2 * k + 1]) ? (float)wt[1] : 0.f};
      // the weight as hi + lo in the value type (~2x its significand): wf -
      // hi is exact (Sterbenz), and hi + lo is exact in FP32 (at most 2 x 11
      // significant bits, the second ~2^-8 below the first)
      A.h.d[jj] = round16x2<bf>(wf);
      const f32x2_t fh = widen16x2<bf>(A.h.d[jj]);
      A.l.d[jj] = round16x2<bf>(f32x2_t{wf.x - fh.x, wf.y - fh.y});
      const f32x2_t fl = widen16x2<bf>(A.l.d[jj]);
      Q.wsum += (double)(fh.x + fl.x);
      Q.wsum += (double)(fh.y + fl.y);
    }
  }
  return any;
}

// The pairs within rounding of the radius: the reference's test decides, and
// a pair that it rejects is taken out again.  A lean weight is subtracted from
// the sum, exactly; with the general weights, which may be infinite or NaN by
// the sample's, the sum starts again from wsum0, its value before the k-block.
template <int DT, uint32_t WK, uint32_t NS>
__device__ __forceinline__ void guard_kblock(const MfmaJob& J, SquareCell<WK>& Q, const Staged<NS, WK>& S,
                                             uint32_t at, uint32_t wl, uint32_t ww, uint32_t cell, uint32_t blk, double wsum0,
                                             WeightOperand& A) {
  constexpr bool bf = DT == kDtBf16, LEAN = WK == kWeightLean;
#pragma unroll 1
  for (uint32_t e = 0; e < 8; ++e) {
    const uint32_t j = at + (__lane_id() >> 4) * 8 + e;
    const double t = pair_distance<LEAN>(Q.npx, Q.npy, Q.npz, S.x[j], S.y[j], S.z[j]);
    if (t < Q.h_hi && S.g[j] - wl <= ww && !(t < Q.h_lo) &&
        !radius_test_ref(J.B.xwcs, J.B.ywcs, J.B.lon_s, J.B.lat_s, cell, blk * kVB + e, J.P.sphere_radius)) {
      const uint32_t sh = (e & 1u) * 16u, keep = 0xFFFF0000u >> sh;
      uint32_t hw = 0, lw = 0;
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i)
        if (i == e >> 1) {
          hw = A.h.d[i] >> sh;
          lw = A.l.d[i] >> sh;
          A.h.d[i] &= keep;
          A.l.d[i] &= keep;
        }
      if constexpr (LEAN) Q.wsum -= (double)(widen16((uint16_t)hw, bf) + widen16((uint16_t)lw, bf));
    }
  }
  if constexpr (!LEAN) {
    Q.wsum = wsum0;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {  // as weigh_kblock adds them
      const f32x2_t fh = widen16x2<bf>(A.h.d[i]), fl = widen16x2<bf>(A.l.d[i]);
      Q.wsum += (double)(fh.x + fl.x);
      Q.wsum += (double)(fh.y + fl.y);
    }
  }
}

// The squares of a block: 4 x 4 cells (2 x 8 and 1 x 16 in blocks of 32 and
// 64 columns); MFMA row i of square mb is cell (i / width, i % width) of it.
struct Squares {
  uint32_t w_shift, x_shift, tc_shift;  // a square's width; squares side by side; the block's width
  __device__ __forceinline__ explicit Squares(uint32_t tc)
      : w_shift(tc <= 4 ? 2u : tc - 2u), x_shift(tc - (tc <= 4 ? 2u : tc - 2u)), tc_shift(tc) {}
  __device__ __forceinline__ uint32_t cell(uint32_t mb, uint32_t i) const {  // its place in the block
    const uint32_t mx = (mb & ((1u << x_shift) - 1u)) << w_shift, my = (mb >> x_shift) << (4u - w_shift);
    return ((my + (i >> w_shift)) << tc_shift) + mx + (i & ((1u << w_shift) - 1u));
  }
};

// Four cells of a map row (quad q of the block at (y0, x0)) of channel ch.
__device__ __forceinline__ void store_quad(const MfmaJob& J, uint32_t y0, uint32_t x0, uint32_t q, uint32_t ch,
                                           const float4& v) {
  const uint32_t side = J.P.side, c0 = q * 4;
  const uint32_t row = y0 + (c0 >> J.tc_shift), col = x0 + (c0 & ((1u << J.tc_shift) - 1u));
  if (row >= side || col >= side || ch >= J.nchan) return;
  float* dst = J.cube + (size_t)ch * side * side + (size_t)row * side + col;
  if ((side & 3u) == 0) {  // uniform; aligned then
    *reinterpret_cast<float4*>(dst) = v;
  } else {
    dst[0] = v.x;
    if (col + 1 < side) dst[1] = v.y;
    if (col + 2 < side) dst[2] = v.z;
    if (col + 3 < side) dst[3] = v.w;
  }
}

// The lane's row of the channel values (MFMA B operand): row ch_base + l % 16
// of a value block, 16 bytes; the 16 lanes of a k-group read one contiguous
// 256-byte piece.  Rows past the last channel fill columns that nothing
// reads: they are the following blocks' (value_rows_read; with one channel
// every lane reads row 0).
__device__ __forceinline__ const char* value_rows(const MfmaJob& J, uint32_t ch_base) {
  return static_cast<const char*>(J.vs) +
         (size_t)(ch_base + (J.nchan > 1 ? __lane_id() & 15u : 0u)) * (kVB * 2u);
}

// One block of 64 cells and up to 16 NB channels (group `group` of them): a
// wave takes a square of 16 cells, on its own but for the set-up and the
// stores.  WK: the kind of weight (mfma_weight_kind).
template <int DT, int NB, uint32_t WK>
__device__ __forceinline__ void mfma_tile(const MfmaJob& J, uint32_t tile, uint32_t group, MfmaLds<WK>& lds,
                                          const double* s_exp) {
  constexpr bool bf = DT == kDtBf16;
  const GridParams& P = J.P;
  const GridBuffers& B = J.B;
  const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6, kg = lane >> 4;
  const hcg_ring_meta m = *B.meta;
  const uint32_t y0 = (tile / J.tiles_x) << (6u - J.tc_shift), x0 = (tile % J.tiles_x) << J.tc_shift;
  MfmaCells& C = lds.s.c;
  MfmaWave<WK>& W = lds.s.w[wave];
  const Squares sq(J.tc_shift);

  if (wave == 0) {
    bool lv;
    const CellGeom g = block_cell(P, B, m, y0, x0, J.tc_shift, lv);
    put_cell(C, lane, g);
  } else if (wave == 1) {
    put_frames(J, lds.s.f, y0, x0);
  }
  __syncthreads();
  const uint32_t cb = sq.cell(wave, lane & 15u);
  const uint32_t crow = y0 + (cb >> J.tc_shift), ccol = x0 + (cb & ((1u << J.tc_shift) - 1u));
  const bool live = crow < P.side && ccol < P.side;
  const uint32_t cell = live ? crow * P.side + ccol : 0;
  uint32_t r_begin, r_end;
  SquareCell<WK> Q;
  {
    CellGeom g;
    g.win = C.win[cb];
    g.pz = C.p[2][cb];
    g.coslat = C.coslat[cb];
    g.tt = C.tt[cb];
    g.wlo = C.wlo[cb];
    g.wwid = C.wwid[cb];
    g.belt = C.belt[cb] != 0;
    const BlockSpan S = cells_span(P, m, g);
    r_begin = S.T.r_begin;
    r_end = S.T.r_end;
    Q.init(P, C, cb, S.simple);
    if (lane == 0) W.bl.span = S;
  }
  const uint32_t ch_base = group * (NB * 16u);
  const char* const vs = value_rows(J, ch_base);
  const size_t blk_bytes = (size_t)J.nchan * kVB * 2u;
  f32x4_t acc[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  for (uint32_t rb = r_begin; r_begin <= r_end && rb <= r_end; rb += 64) {
    tile_sync();
    const uint32_t total = ring_blocks(P, B, m, rb, W.bl);
    for (uint32_t q0 = 0; q0 < total; q0 += 128) {  // uniform
      const uint32_t cnt = min(total - q0, 128u), nkb = (cnt + 3) / 4;
      tile_sync();
      list_blocks(W.bl, q0, cnt);
      tile_sync();
      StageRegs<WK> st;
      st.fetch(B, m, W.bl, 0, lane & 31u, lane >> 5);
      for (uint32_t u = 0; u < nkb; ++u) {
        tile_sync();  // the previous k-block is consumed
        st.store(W.st, lane & 31u, lane >> 5);
        const uint32_t blk = W.bl.lb[u * 4 + kg];
        uint32_t wl, ww;
        Q.window(P, C, W.bl, rb, W.bl.lr[u * 4 + kg], wl, ww);
        s16x8_t bn[NB];
        auto load_b = [&]() {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            bn[nb] = *reinterpret_cast<const s16x8_t*>(vs + blk * blk_bytes + nb * (16 * kVB * 2));
        };
        load_b();
        if (u + 1 < nkb) st.fetch(B, m, W.bl, u + 1, lane & 31u, lane >> 5);
        tile_sync();
        WeightOperand A;
        uint64_t guard;
        const double wsum0 = Q.wsum;
        const uint64_t any = weigh_kblock<DT>(J, Q, W.st, lds.s.f, 0, wl, ww, cell, blk, s_exp, A, guard);
        if (guard) {  // uniform, rare
          // the sums wait in scratch memory meanwhile (volatile: here and only
          // here), and the channel values are read again: across the call they
          // would not fit the registers that it preserves, and would be
          // spilled in every k-block
          volatile float keep[NB * 4];
#pragma unroll
          for (int i = 0; i < NB * 4; ++i) keep[i] = acc[i / 4][i % 4];
          guard_kblock<DT>(J, Q, W.st, 0, wl, ww, cell, blk, wsum0, A);
#pragma unroll
          for (int i = 0; i < NB * 4; ++i) acc[i / 4][i % 4] = keep[i];
          load_b();
        }
        if (any) {  // uniform
#pragma unroll
          for (int nb = 0; nb < NB; ++nb) {
            acc[nb] = mfma16(bf, A.h.v, bn[nb], acc[nb]);
            acc[nb] = mfma16(bf, A.l.v, bn[nb], acc[nb]);
          }
        }
      }
    }
  }

  // per-cell weight sums over the k-groups (exact in FP64 in any order: every
  // weight is hi + lo of two 16-bit values).  The normalisation is one
  // multiply per value: v * (1 / t) is within an FP64 ulp or two of v / t, so
  // the FP32 result is the quotient's except where it lies that close to an
  // FP32 rounding boundary (1 ulp then); t = 0 gives inf, so an empty cell is
  // 0 * inf = NaN as 0 / 0 is.
  double wsum = Q.wsum;
  wsum += __shfl_xor(wsum, 16, 64);
  wsum += __shfl_xor(wsum, 32, 64);
  if (group == 0 && J.wsum && live && lane < 16) J.wsum[cell] = (float)wsum;
  const double inv = J.normalize ? 1.0 / wsum : 1.0;
  double iv[4];  // of the lane's MFMA rows 4 kg .. 4 kg + 3
#pragma unroll
  for (uint32_t j = 0; j < 4; ++j) iv[j] = __shfl(inv, kg * 4 + j, 64);
  // Stores through LDS, 64 channels of the block at a time: the 16-byte quads
  // (four cells of a map row) of a channel's 64 cells, XOR-swizzled by the
  // channel, so that the 16 channels of a write and the 16 quads of a read
  // fall in distinct bank groups; a store instruction then writes four
  // channels' whole rows of the block instead of 64 scattered pieces.
  const uint32_t q_own = sq.cell(wave, kg * 4) >> 2;
#pragma unroll
  for (int s = 0; s < (NB + 3) / 4; ++s) {
    if (ch_base + s * 64 >= J.nchan) break;  // uniform
    __syncthreads();  // the samples, or the previous channels, are done with
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int nb = s * 4 + k;
      if (nb < NB) {
        const uint32_t cr = k * 16 + (lane & 15u);
        *reinterpret_cast<float4*>(&lds.t[cr * 64 + ((q_own ^ (cr & 15u)) << 2)]) =
            make_float4((float)((double)acc[nb][0] * iv[0]), (float)((double)acc[nb][1] * iv[1]),
                        (float)((double)acc[nb][2] * iv[2]), (float)((double)acc[nb][3] * iv[3]));
      }
    }
    __syncthreads();
    constexpr uint32_t kSteps = NB >= 4 ? 4 : NB;  // 16 channels a step of the four waves
    const uint32_t q = lane & 15u;
#pragma unroll
    for (uint32_t k = 0; k < kSteps; ++k) {
      const uint32_t cr = k * 16 + wave * 4 + kg;
      store_quad(J, y0, x0, q, ch_base + s * 64 + cr,
                 *reinterpret_cast<const float4*>(&lds.t[cr * 64 + ((q ^ (cr & 15u)) << 2)]));
    }
  }
}

// Many channels: a workgroup of eight waves takes a block of 64 cells and 512
// channels, a wave all four squares of 64 channels, and the weights, once per
// workgroup, go through LDS.  Four k-blocks a round, one barrier: wave w
// evaluates the weights of square w % 4 in k-blocks w / 4 and w / 4 + 2 of the
// round to come and contracts all squares of the present one, two k-blocks
// after each.  Half of the waves (one on each SIMD) start with the weights and
// half with the products, so that matrix and vector instructions overlap.  The
// channel values of two k-blocks are read when the two before are done with,
// and arrive while weights are evaluated.
constexpr uint32_t kWideList = 256;
template <uint32_t WK>
union MfmaWideLds {
  struct {
    s16x8_t a[2][4][4][2][64];  // [round parity][k-block][square][hi, lo][lane]
    uint32_t any[2][4][4];      // the operand holds a weight
    Staged<128, WK> st[2];
    BlockList<kWideList> bl;
    MfmaCells c;
    MfmaFrames<WK> f;
    double wsum[kWideWaves][16];
    double inv[kMcCols];
    uint32_t total;
  } s;
  float t[kWideWaves][16 * 64];  // the epilogue's 16 channels x 64 cells of a wave
};

template <int DT, uint32_t WK>
__device__ __forceinline__ void mfma_wide(const MfmaJob& J, uint32_t tile, uint32_t group, MfmaWideLds<WK>& lds,
                                          const double* s_exp) {
  constexpr bool bf = DT == kDtBf16;
  const GridParams& P = J.P;
  const GridBuffers& B = J.B;
  const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6, kg = lane >> 4;
  const hcg_ring_meta m = *B.meta;
  const uint32_t y0 = (tile / J.tiles_x) << (6u - J.tc_shift), x0 = (tile % J.tiles_x) << J.tc_shift;
  MfmaCells& C = lds.s.c;
  BlockList<kWideList>& L = lds.s.bl;
  const Squares sq(J.tc_shift);
  const uint32_t mb_own = wave & 3u, kb_own = wave >> 2;  // whose weights this wave evaluates

  const MfmaPlan* const plan =
      J.plan ? reinterpret_cast<const MfmaPlan*>(static_cast<const char*>(J.plan) + tile * kPlanBytes) : nullptr;
  const bool planned = plan && __builtin_amdgcn_readfirstlane(plan->ok) != 0;  // uniform
  if (planned) {
    if (wave < 3) {
      C.p[wave][lane] = plan->p[wave][lane];
    } else if (wave == 3) {
      C.win[lane].uring = plan->uring[lane];
      C.win[lane].dring = plan->dring[lane];
    } else if (wave == 4) {
      C.wlo[lane] = plan->wlo[lane];
      C.wwid[lane] = plan->wwid[lane];
    } else if (wave == 5 && lane == 0) {
      L.span.T.r_begin = plan->r_begin;
      L.span.T.r_end = plan->r_end;
      L.span.simple = true;
    }
  } else if (wave == 0) {
    bool lv;
    const CellGeom g = block_cell(P, B, m, y0, x0, J.tc_shift, lv);
    put_cell(C, lane, g);
    const BlockSpan S = cells_span(P, m, g);
    if (lane == 0) L.span = S;
  }
  if (wave == 6) put_frames(J, lds.s.f, y0, x0);
  __syncthreads();
  const uint32_t cb = sq.cell(mb_own, lane & 15u);
  const uint32_t crow = y0 + (cb >> J.tc_shift), ccol = x0 + (cb & ((1u << J.tc_shift) - 1u));
  const bool live = crow < P.side && ccol < P.side;
  const uint32_t cell = live ? crow * P.side + ccol : 0;
  const uint32_t r_begin = __builtin_amdgcn_readfirstlane(L.span.T.r_begin);
  const uint32_t r_end = __builtin_amdgcn_readfirstlane(L.span.T.r_end);
  SquareCell<WK> Q;
  Q.init(P, C, cb, __builtin_amdgcn_readfirstlane((uint32_t)L.span.simple) != 0);
  const uint32_t ch_base = (group * kWideWaves + wave) * 64u;
  const bool mine = ch_base < J.nchan;  // uniform: the wave has channels
  const char* const vs = value_rows(J, mine ? ch_base : 0);
  const size_t blk_bytes = (size_t)J.nchan * kVB * 2u;
  f32x4_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i / 4][i % 4] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  s16x8_t bn[2][4];

  for (uint32_t rb = r_begin; r_begin <= r_end && rb <= r_end; rb += 64) {
    __syncthreads();
    if (wave == 0) {
      const uint32_t t =
          planned ? put_rings(P, L, rb, plan->b0[lane], plan->nb[lane]) : ring_blocks(P, B, m, rb, L);
      if (lane == 0) lds.s.total = t;
    }
    __syncthreads();
    const uint32_t total = __builtin_amdgcn_readfirstlane(lds.s.total);
    for (uint32_t q0 = 0; q0 < total; q0 += kWideList) {  // uniform
      const uint32_t cnt = min(total - q0, kWideList), nkb = (cnt + 3) / 4, nr = (nkb + 3) / 4;
      __syncthreads();
      if (wave == 0) list_blocks(L, q0, cnt);
      __syncthreads();
      // waves 0 to 3 stage the 128 samples of round r (a k-block past the
      // last is neither staged nor weighed)
      StageRegs<WK> st;
      const uint32_t ssp = (wave & 1u) * 64 + lane;  // sample of a round
      auto fetch = [&](uint32_t r) {
        if (wave < 4 && 4 * r + (ssp >> 5) < nkb) st.fetch(B, m, L, 4 * r + (ssp >> 5), ssp & 31u, wave >> 1);
      };
      auto stage = [&](uint32_t r) {
        if (wave < 4 && 4 * r + (ssp >> 5) < nkb) st.store(lds.s.st[r & 1u], ssp, wave >> 1);
      };
      auto load_b = [&](uint32_t u) {  // of k-blocks u and u + 1
        if (!mine) return;
#pragma unroll
        for (uint32_t kb = 0; kb < 2; ++kb) {
          const uint32_t blk = L.lb[min(u + kb, nkb - 1) * 4 + kg];
#pragma unroll
          for (int nb = 0; nb < 4; ++nb)
            bn[kb][nb] = *reinterpret_cast<const s16x8_t*>(vs + blk * blk_bytes + nb * (16 * kVB * 2));
        }
      };
      auto weigh = [&](uint32_t r, uint32_t h) {  // k-block kb_own + 2 h of round r
        const uint32_t k = kb_own + 2 * h, u = 4 * r + k, par = r & 1u;
        uint64_t any = 0;
        if (u < nkb) {  // uniform
          const uint32_t blk = L.lb[u * 4 + kg];
          uint32_t wl, ww;
          Q.window(P, C, L, rb, L.lr[u * 4 + kg], wl, ww);
          WeightOperand A;
          uint64_t guard;
          const double wsum0 = Q.wsum;
          any = weigh_kblock<DT>(J, Q, lds.s.st[par], lds.s.f, k * 32, wl, ww, cell, blk, s_exp, A, guard);
          if (guard) {  // uniform, rare; the sums wait in scratch memory (see mfma_tile)
            volatile float keep[64];
#pragma unroll
            for (int i = 0; i < 64; ++i) keep[i] = acc[i / 16][i / 4 % 4][i % 4];
            guard_kblock<DT>(J, Q, lds.s.st[par], k * 32, wl, ww, cell, blk, wsum0, A);
#pragma unroll
            for (int i = 0; i < 64; ++i) acc[i / 16][i / 4 % 4][i % 4] = keep[i];
          }
          if (any) {
            lds.s.a[par][k][mb_own][0][lane] = A.h.v;
            lds.s.a[par][k][mb_own][1][lane] = A.l.v;
          }
        }
        if (lane == 0) lds.s.any[par][k][mb_own] = any != 0;
      };
      auto contract = [&](uint32_t r, uint32_t h) {  // k-blocks 2 h and 2 h + 1 of round r
        if (!mine) return;
        const uint32_t par = r & 1u;
        uint32_t some[2][4];
#pragma unroll
        for (int i = 0; i < 8; ++i) some[i / 4][i % 4] = lds.s.any[par][2 * h + i / 4][i % 4];
#pragma unroll
        for (uint32_t kb = 0; kb < 2; ++kb) {
          s16x8_t ah[4], al[4];  // (stale where a square has no weight, and unused)
#pragma unroll
          for (uint32_t mb = 0; mb < 4; ++mb) {
            ah[mb] = lds.s.a[par][2 * h + kb][mb][0][lane];
            al[mb] = lds.s.a[par][2 * h + kb][mb][1][lane];
          }
#pragma unroll
          for (uint32_t mb = 0; mb < 4; ++mb) {
            if (!__builtin_amdgcn_readfirstlane(some[kb][mb])) continue;  // uniform
#pragma unroll
            for (int nb = 0; nb < 4; ++nb) {
              acc[mb][nb] = mfma16(bf, ah[mb], bn[kb][nb], acc[mb][nb]);
              acc[mb][nb] = mfma16(bf, al[mb], bn[kb][nb], acc[mb][nb]);
            }
          }
        }
      };
      fetch(0);
      stage(0);
      load_b(0);
      fetch(1);
      __syncthreads();
      weigh(0, 0);
      weigh(0, 1);
      stage(1);
      __syncthreads();
      for (uint32_t r = 0; r < nr; ++r) {
        fetch(r + 2);
        const bool more = r + 1 < nr;
#pragma unroll 1
        for (uint32_t h = 0; h < 2; ++h) {
          if (wave < kWideWaves / 2 && more) weigh(r + 1, h);
          contract(r, h);
          load_b(4 * r + 2 * h + 2);
          if (wave >= kWideWaves / 2 && more) weigh(r + 1, h);
        }
        stage(r + 2);
        __syncthreads();
      }
    }
  }

  // the weight sums of a square's two waves (see mfma_tile)
  double wsum = Q.wsum;
  wsum += __shfl_xor(wsum, 16, 64);
  wsum += __shfl_xor(wsum, 32, 64);
  if (lane < 16) lds.s.wsum[wave][lane] = wsum;
  __syncthreads();
  if (wave < 4 && lane < 16) {
    const double t = lds.s.wsum[wave][lane] + lds.s.wsum[wave + 4][lane];
    if (group == 0 && J.wsum && live) J.wsum[cell] = (float)t;
    lds.s.inv[cb] = J.normalize ? 1.0 / t : 1.0;
  }
  __syncthreads();
  double iv[4][4];
#pragma unroll
  for (uint32_t mb = 0; mb < 4; ++mb)
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) iv[mb][j] = lds.s.inv[sq.cell(mb, kg * 4 + j)];
  __syncthreads();
  // stores as in mfma_tile, 16 channels of the wave's own at a time
  float* const T = lds.t[wave];
#pragma unroll
  for (int nb = 0; nb < 4; ++nb) {
    tile_sync();
#pragma unroll
    for (uint32_t mb = 0; mb < 4; ++mb)
      *reinterpret_cast<float4*>(&T[(lane & 15u) * 64 + (((sq.cell(mb, kg * 4) >> 2) ^ (lane & 15u)) << 2)]) =
          make_float4((float)((double)acc[mb][nb][0] * iv[mb][0]), (float)((double)acc[mb][nb][1] * iv[mb][1]),
                      (float)((double)acc[mb][nb][2] * iv[mb][2]), (float)((double)acc[mb][nb][3] * iv[mb][3]));
    tile_sync();
    const uint32_t q = lane & 15u;
#pragma unroll
    for (uint32_t k = 0; k < 4; ++k) {
      const uint32_t cr = k * 4 + kg;
      store_quad(J, y0, x0, q, ch_base + nb * 16 + cr,
                 *reinterpret_cast<const float4*>(&T[cr * 64 + ((q ^ cr) << 2)]));
    }
  }
}

// The tile of workgroup b of a job.  Workgroup b runs on XCD b % 8: an XCD
// takes a contiguous run of tiles, so neighbouring tiles share an L2.  The
// many-channel kernel, one workgroup per CU, takes maps of 1024 tiles and more
// in patches of 8 x 4 tiles, so that the rows of samples that vertical
// neighbours share are read a quarter of a tile's time apart and not a row of
// the map later: 2M x 1024 a pass 8.46 -> 8.14-8.26 ms (4 x 8 8.33, 2 x 16 8.33,
// 2 x 8 8.28).  With fewer channels a CU holds several workgroups and patches
// change nothing (1.2M x 64 onto 512^2 1.531 and 1.540 ms).
constexpr uint32_t kPatchW = 8, kPatchH = 4, kPatchTiles = kPatchW * kPatchH, kPatchMinTiles = 1024;
__host__ __device__ inline uint32_t patches_per_xcd(uint32_t ntiles, uint32_t tiles_x) {
  return ((tiles_x + kPatchW - 1) / kPatchW * ((ntiles / tiles_x + kPatchH - 1) / kPatchH) + 7u) / 8u;
}
__host__ __device__ inline uint32_t tile_blocks(uint32_t ntiles, uint32_t tiles_x, bool wide) {
  if (!wide || ntiles < kPatchMinTiles) return (ntiles + 7u) / 8u * 8u;
  return 8u * patches_per_xcd(ntiles, tiles_x) * kPatchTiles;
}
// (ntiles or more: none)
__device__ inline uint32_t block_tile(uint32_t b, uint32_t ntiles, uint32_t tiles_x, bool wide) {
  const uint32_t xcd = b & 7u, i = b >> 3;
  if (!wide || ntiles < kPatchMinTiles) return xcd * ((ntiles + 7u) / 8u) + i;
  const uint32_t px = (tiles_x + kPatchW - 1) / kPatchW;
  const uint32_t patch = xcd * patches_per_xcd(ntiles, tiles_x) + i / kPatchTiles;
  const uint32_t x = patch % px * kPatchW + i % kPatchW, y = patch / px * kPatchH + i / kPatchW % kPatchH;
  return x < tiles_x ? y * tiles_x + x : ntiles;  // (past the last row: past ntiles)
}

// The kernel instances: NB 16-channel blocks per wave (mfma_tile), or 0: mfma_wide.
constexpr int mfma_waves_per_simd(int nb, uint32_t kind) {
  return kind != kWeightLean || nb == 0 ? 2 : nb <= 2 ? 4 : nb <= 6 ? 3 : 2;
}
constexpr uint32_t mfma_threads(int nb) { return 64 * (nb == 0 ? kWideWaves : (uint32_t)kMcWaves); }
template <int NB, uint32_t WK>
struct InstanceLds {
  typedef MfmaLds<WK> type;
};
template <uint32_t WK>
struct InstanceLds<0, WK> {
  typedef MfmaWideLds<WK> type;
};
template <int DT, int NB, uint32_t WK>
__device__ __forceinline__ void mfma_work(const MfmaJob& J, uint32_t tile, uint32_t group) {
  __shared__ typename InstanceLds<NB, WK>::type lds;
  __shared__ double s_exp[64];
  if (threadIdx.x < 64) exp_table_load(s_exp);
  if constexpr (NB == 0)
    mfma_wide<DT, WK>(J, tile, group, lds, s_exp);
  else
    mfma_tile<DT, NB, WK>(J, tile, group, lds, s_exp);
}

// One job: grid = (tile_blocks, or a run of them from `first` on, channel groups).
template <int DT, int NB, uint32_t WK>
__global__ void __launch_bounds__(mfma_threads(NB)) __attribute__((amdgpu_waves_per_eu(mfma_waves_per_simd(NB, WK))))
    k_grid_mfma(MfmaJob J, uint32_t first) {
  const uint32_t tile = block_tile(first + blockIdx.x, J.ntiles, J.tiles_x, NB == 0);
  if (tile >= J.ntiles) return;  // uniform
  mfma_work<DT, NB, WK>(J, tile, blockIdx.y);
}

// The jobs of a batch that one instance serves, in one launch: a workgroup
// finds its job by binary search over the range starts (multiples of 8).
template <int DT, int NB, uint32_t WK>
__global__ void __launch_bounds__(mfma_threads(NB)) __attribute__((amdgpu_waves_per_eu(mfma_waves_per_simd(NB, WK))))
    k_grid_mfma_batch(const TileRange* __restrict__ ranges, uint32_t nranges, const MfmaJob* __restrict__ jobs,
                      uint32_t first) {
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
  const uint32_t lb = block - ranges[lo].first, per = tile_blocks(J.ntiles, J.tiles_x, NB == 0);
  const uint32_t tile = block_tile(lb % per, J.ntiles, J.tiles_x, NB == 0), group = lb / per;
  if (tile >= J.ntiles) return;  // uniform
  mfma_work<DT, NB, WK>(J, tile, group);
}

// A launch of one instance: a job's workgroups (`count` of them from `first` on,
// times the channel groups), or a batch's over its ranges (job NULL).
template <uint32_t FORM, int DT>
inline void launch_form(const MfmaLaunch& L) {
  constexpr int nb = (int)kFormNb[FORM];
  constexpr uint32_t kind = kind_of_form(FORM);
  if (L.job)
    k_grid_mfma<DT, nb, kind><<<dim3(L.count, L.groups), mfma_threads(nb), 0, L.stream>>>(*L.job, L.first);
  else
    k_grid_mfma_batch<DT, nb, kind>
        <<<L.count, mfma_threads(nb), 0, L.stream>>>(L.ranges, L.nranges, L.jobs, L.first);
}
template <uint32_t FORM, uint32_t END>
inline void launch_forms(uint32_t inst, const MfmaLaunch& L) {
  if constexpr (FORM < END) {
    if (inst == 2 * FORM)
      launch_form<FORM, kDtBf16>(L);
    else if (inst == 2 * FORM + 1)
      launch_form<FORM, kDtF16>(L);
    else
      launch_forms<FORM + 1, END>(inst, L);
  }
}

}  // namespace hcg
