// presort.hip -- device pre-sort of the samples and the ring lookup table.
//
// Replaces init_input_with_cpu / init_input_with_thrust
// (HCGrid/gridding.cu:70-147): the reference computes HEALPix keys on one
// host thread, sorts 16-byte (key, index) records with boost/Thrust on the
// host, gathers lon/lat/data through the permutation and builds the ring
// LUT with a sequential binary-search loop.  Here all of it stays in HBM:
//
//   k_keys         ang2pix per sample -> key, and the first digit's counts per tile
//   k_rs_upsweep   a later digit's counts per tile        } two or three passes of
//   k_rs_scan      per digit, scan over the tiles         } a stable LSD radix sort
//   k_rs_downsweep stable in-tile ranking, scatter        } on up to ten bits each
//   k_gather       permutation gather fused with the unit-vector records
//   k_ring_lut     firstring, usedrings, LUT and per-ring cos/sin
//
// The radix sort is reduce-then-scan (no inter-workgroup waiting) and stable
// by construction: tiles keep input order, a wave of a tile owns a contiguous
// part of it, and within a wave items are ranked in index order with ballots.
// Keys are < npix <= 12 8192^2 < 2^30, or MAX_Y, which sorts as npix: at most
// 30 bits, three digits of ten (two digits up to nside 256).
//
// What it costs: on small inputs the launches (a dependent launch takes about
// 4.5 us whatever it does), on large ones the scatter, whose 4-byte stores of
// a wave go to as many lines as it has digits.  Four 8-bit passes of four
// launches each, ranked with three workgroup barriers per 256 items, took
// 142 us for 250k samples and 760 us for 20M.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <utility>

#include "common.hpp"
#include "healpix.hpp"

namespace hcg {

// Keys per sort tile: small tiles fill the chip's 256 CUs from few samples on,
// large ones have fewer counts to write and scan (1024 digits a tile).
// Presort: 1M samples 111 us with small tiles, 1.2M 123 us with large ones and
// 112 with middle ones, 2M 150 us with middle and 138 with large ones.
constexpr uint32_t kSmallTile = 256 * 4, kMidTile = 256 * 8, kLargeTile = 512 * 16;
constexpr uint32_t kSmallTiles = 512, kMidTiles = 768;
constexpr int kMaxDigitBits = 10;
constexpr uint32_t kMaxDigits = 1u << kMaxDigitBits;

// A pass: digit = (min(key, top) >> shift) & (2^bits - 1).
struct Digit {
  uint32_t top;  // npix: MAX_Y keys sort as it
  int shift, bits;
};

__device__ inline uint32_t digit_of(uint32_t key, const Digit& g) {
  return (min(key, g.top) >> g.shift) & ((1u << g.bits) - 1u);
}

// The tile of this workgroup: neighbouring tiles, whose counts share cache
// lines, on one XCD (block b runs on XCD b % 8).  sort_blocks(tiles)
// workgroups; tile >= tiles has nothing to do.
__device__ inline uint32_t sort_tile(uint32_t tiles) {
  return (blockIdx.x & 7u) * ((tiles + 7u) >> 3) + (blockIdx.x >> 3);
}
inline uint32_t sort_blocks(uint32_t tiles) { return (tiles + 7u) & ~7u; }

// Adds each valid lane's digit to the workgroup's LDS counts: one add for a
// wave whose digits are all equal (nearly sorted input), else one per lane.
__device__ inline void count_digit(uint32_t* h, uint32_t d, bool valid) {
  const uint64_t vm = __ballot(valid);
  if (vm == 0) return;
  const uint32_t first = (uint32_t)__builtin_amdgcn_readlane((int)d, (int)__ffsll((unsigned long long)vm) - 1);
  if (__ballot(valid && d == first) == vm) {
    if (__lane_id() == 0) atomicAdd(&h[first], (uint32_t)__popcll(vm));
  } else if (valid) {
    atomicAdd(&h[d], 1u);
  }
}

// Keys of one tile and its counts of the first digit, hist[d * tiles + tile].
// Workgroup 0 writes the npix sentinel (HCGrid/gridding.cu:100).
template <uint32_t THREADS, uint32_t ITEMS>
__global__ void __launch_bounds__(THREADS) k_keys(hcg_healpix hp, uint32_t n, const double* __restrict__ lon,
                                                  const double* __restrict__ lat, uint32_t* __restrict__ keys,
                                                  uint32_t* __restrict__ sentinel, Digit g, uint32_t tiles,
                                                  uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[kMaxDigits];
  const Hpx32 hx = hpx32(hp);
  const uint32_t digits = 1u << g.bits, tile = sort_tile(tiles);
  if (tile >= tiles) return;
  for (uint32_t d = threadIdx.x; d < digits; d += THREADS) h[d] = 0;
  __syncthreads();
  // 64-bit index: a 32-bit one wraps for n close to 2^32
  const uint64_t base = (uint64_t)tile * (THREADS * ITEMS);
#pragma unroll 2
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const uint64_t i = base + j * THREADS + threadIdx.x;
    uint32_t key = 0;
    if (i < n) {
      // HCGrid/gridding.cu:78-80
      key = ang2pix32(hx, kHalfPi - kDeg2Rad * lat[i], kDeg2Rad * lon[i]);
      keys[i] = key;
    }
    count_digit(h, digit_of(key, g), i < n);
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < digits; d += THREADS) hist[(size_t)d * tiles + tile] = h[d];
  if (blockIdx.x == 0 && threadIdx.x == 0) *sentinel = hx.npix;
}

// Digit counts of one tile, hist[d * tiles + tile].
template <uint32_t THREADS, uint32_t ITEMS>
__global__ void __launch_bounds__(THREADS) k_rs_upsweep(const uint32_t* __restrict__ keys, uint32_t n, Digit g,
                                                        uint32_t tiles, uint32_t* __restrict__ hist) {
  __shared__ uint32_t h[kMaxDigits];
  const uint32_t digits = 1u << g.bits, tile = sort_tile(tiles);
  if (tile >= tiles) return;
  for (uint32_t d = threadIdx.x; d < digits; d += THREADS) h[d] = 0;
  __syncthreads();
  const uint64_t base = (uint64_t)tile * (THREADS * ITEMS);
#pragma unroll 4
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const uint64_t i = base + j * THREADS + threadIdx.x;
    const bool valid = i < n;
    count_digit(h, digit_of(valid ? keys[i] : 0u, g), valid);
  }
  __syncthreads();
  for (uint32_t d = threadIdx.x; d < digits; d += THREADS) hist[(size_t)d * tiles + tile] = h[d];
}

// Orders this wave's LDS operations (they execute in issue order: a fence for
// the compiler).
__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Exclusive scan of one value per thread over the workgroup (a multiple of
// 64 threads, at most 1024); lds holds one word per wave.
__device__ inline uint32_t block_exclusive_scan(uint32_t v, uint32_t* lds, uint32_t& total) {
  const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  uint32_t x = v;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const uint32_t y = __shfl_up(x, off, 64);
    if (lane >= (uint32_t)off) x += y;
  }
  if (lane == 63) lds[wave] = x;
  __syncthreads();
  uint32_t before = 0;
  total = 0;
  for (uint32_t w = 0; w < nw; ++w) {
    const uint32_t s = lds[w];
    if (w < wave) before += s;
    total += s;
  }
  __syncthreads();
  return before + x - v;
}

// One workgroup per digit: exclusive scan of its row of tile counts; the row
// total goes to digit_tot[d].
__global__ void __launch_bounds__(256) k_rs_scan(uint32_t* __restrict__ hist, uint32_t tiles,
                                                 uint32_t* __restrict__ digit_tot) {
  __shared__ uint32_t lds[4];
  uint32_t* row = hist + (size_t)blockIdx.x * tiles;
  uint32_t running = 0;
  for (uint32_t base = 0; base < tiles; base += 256 * 4) {
    uint32_t v[4];
    uint32_t s = 0;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t i = base + threadIdx.x * 4 + q;
      v[q] = (i < tiles) ? row[i] : 0u;
      s += v[q];
    }
    uint32_t total;
    uint32_t pre = block_exclusive_scan(s, lds, total) + running;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const uint32_t i = base + threadIdx.x * 4 + q;
      if (i < tiles) row[i] = pre;
      pre += v[q];
    }
    running += total;
  }
  if (threadIdx.x == 0) digit_tot[blockIdx.x] = running;
}

// Stable scatter of one tile.  Wave w owns the tile's items w * ITEMS * 64 ..
// and ranks them in index order against its own counts in LDS (its LDS
// operations execute in order, so this needs no barrier); the waves' counts
// then become offsets in wave order.  FIRST: the values are the indexes.
template <uint32_t THREADS, uint32_t ITEMS, bool FIRST>
__global__ void __launch_bounds__(THREADS) k_rs_downsweep(const uint32_t* __restrict__ kin,
                                                          const uint32_t* __restrict__ vin,
                                                          uint32_t* __restrict__ kout, uint32_t* __restrict__ vout,
                                                          uint32_t n, Digit g, uint32_t tiles,
                                                          const uint32_t* __restrict__ hist,
                                                          const uint32_t* __restrict__ digit_tot) {
  constexpr uint32_t W = THREADS / 64;
  constexpr uint32_t PER = kMaxDigits / THREADS;  // digits per thread
  __shared__ uint32_t cnt[W][kMaxDigits];
  __shared__ uint32_t lds[W];
  const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
  const uint32_t digits = 1u << g.bits, tile = sort_tile(tiles);
  if (tile >= tiles) return;
  for (uint32_t d = lane; d < digits; d += 64) cnt[wave][d] = 0;  // (its own wave's: no barrier)
  wave_fence();
  // this tile's first position of each digit: the digits before it, and the tiles before it
  uint32_t off[PER];
  {
    uint32_t tot[PER], s = 0;
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      const uint32_t d = threadIdx.x * PER + q;
      tot[q] = d < digits ? digit_tot[d] : 0u;
      off[q] = d < digits ? hist[(size_t)d * tiles + tile] : 0u;
      s += tot[q];
    }
    uint32_t total;
    uint32_t pre = block_exclusive_scan(s, lds, total);
#pragma unroll
    for (uint32_t q = 0; q < PER; ++q) {
      off[q] += pre;
      pre += tot[q];
    }
  }
  const uint64_t base = (uint64_t)tile * (THREADS * ITEMS) + (uint64_t)wave * (ITEMS * 64) + lane;
  uint32_t key[ITEMS], val[ITEMS];
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const uint64_t i = base + j * 64;
    key[j] = i < n ? kin[i] : 0u;
    val[j] = FIRST ? (uint32_t)i : (i < n ? vin[i] : 0u);
  }
  const uint64_t lt = lanemask_lt();
  uint32_t rank[ITEMS];
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j) {
    const bool valid = base + j * 64 < n;
    const uint32_t d = digit_of(key[j], g);
    uint64_t peers = __ballot(valid);
    for (int b = 0; b < g.bits; ++b) {  // uniform
      const uint64_t vote = __ballot((d >> b) & 1u);
      peers &= ((d >> b) & 1u) ? vote : ~vote;
    }
    const uint32_t before = valid ? cnt[wave][d] : 0u;
    rank[j] = before + (uint32_t)__popcll(peers & lt);
    wave_fence();
    if (valid && (peers & lt) == 0) cnt[wave][d] = before + (uint32_t)__popcll(peers);
    wave_fence();
  }
  __syncthreads();
#pragma unroll
  for (uint32_t q = 0; q < PER; ++q) {
    const uint32_t d = threadIdx.x * PER + q;
    if (d < digits) {
      uint32_t at = off[q];
#pragma unroll
      for (uint32_t w = 0; w < W; ++w) {
        const uint32_t c = cnt[w][d];
        cnt[w][d] = at;
        at += c;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (uint32_t j = 0; j < ITEMS; ++j)
    if (base + j * 64 < n) {
      const uint32_t pos = cnt[wave][digit_of(key[j], g)] + rank[j];
      kout[pos] = key[j];
      vout[pos] = val[j];
    }
}

__global__ void __launch_bounds__(64) k_set_sentinel(uint32_t* keys, uint32_t n, uint32_t npix) {
  if (threadIdx.x == 0 && blockIdx.x == 0) keys[n] = npix;  // HCGrid/gridding.cu:100
}

// Permutation gather (HCGrid/gridding.cu:101-114) fused with the records the
// gridding kernel reads.
__global__ void __launch_bounds__(256) k_gather(uint32_t n, const uint32_t* __restrict__ perm,
                                                const double* __restrict__ lon, const double* __restrict__ lat,
                                                const void* __restrict__ data, int dtype,
                                                const double* __restrict__ w, hcg_sample* __restrict__ rec,
                                                double* __restrict__ lon_s, double* __restrict__ lat_s,
                                                double* __restrict__ data_s, double* __restrict__ w_s) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint32_t j = perm[i];
    if (j >= n) j = (uint32_t)i;  // a permutation never holds this; keeps every read in bounds regardless
    const double lo = lon[j], la = lat[j];
    const double v = !data                      ? 0.0  // multi-channel jobs carry values separately
                     : (dtype == HCG_DTYPE_F64) ? static_cast<const double*>(data)[j]
                                                : (double)static_cast<const float*>(data)[j];
    double sb, cb, sl, cl;
    sincos(la * kDeg2Rad, &sb, &cb);
    sincos(lo * kDeg2Rad, &sl, &cl);
    hcg_sample r;
    r.x = cb * cl;
    r.y = cb * sl;
    r.z = sb;
    r.v = v;
    rec[i] = r;
    if (lon_s) lon_s[i] = lo;
    if (lat_s) lat_s[i] = la;
    if (data_s) data_s[i] = v;
    if (w_s) w_s[i] = w ? w[j] : 1.0;
  }
}

// First index of n keys with key >= x (n if none), three probes a step: a
// step is one round of dependent loads and quarters the range.
__device__ inline uint32_t lower_bound_4(const uint32_t* __restrict__ keys, uint32_t n, uint32_t x) {
  uint32_t a = 0, b = n;
  while (a < b) {
    const uint32_t d = (b - a) >> 2, p0 = a + d, p1 = a + ((b - a) >> 1), p2 = min(p1 + d, b - 1);
    const uint32_t k0 = keys[p0], k1 = keys[p1], k2 = keys[p2];
    if (k2 < x)
      a = p2 + 1;
    else if (k1 < x)
      a = p1 + 1, b = p2;
    else if (k0 < x)
      a = p0 + 1, b = p1;
    else
      b = p0;
  }
  return a;
}

// firstring / usedrings / n_valid (HCGrid/gridding.cu:118-121).  Samples
// whose key is >= npix (theta outside [0, pi]) sort last and are left out of
// the ring span; the reference would take pix2ring of MAX_Y there.
__device__ inline hcg_ring_meta ring_meta(const hcg_healpix& hp, uint32_t n, const uint32_t* __restrict__ keys) {
  const Hpx32 hx = hpx32(hp);
  hcg_ring_meta m;
  m.n = n;
  m.firstring = m.usedrings = 0;
  m.n_valid = n == 0 || keys[n - 1] < hx.npix ? n : lower_bound_4(keys, n, hx.npix);
  if (m.n_valid) {
    m.firstring = pix2ring32(hx, keys[0]);
    m.usedrings = 1 + pix2ring32(hx, keys[m.n_valid - 1]) - m.firstring;
  }
  return m;
}

// Level-1 LUT (HCGrid/gridding.cu:122-136): lut[k] = first index with key >=
// startpix(firstring + k).  The reference's incremental searchLastPosLessThan
// walk returns exactly this lower bound.  Also the per-ring cos/sin of the
// ring-centre colatitude (HCGrid/gridding.cu:332-334); ring_s < 0 marks rings
// where the reference's ang2pix takes the cos-only branch.  Every thread
// works out the ring span (three loads) rather than wait for a launch that
// does; the first writes it.
__global__ void __launch_bounds__(256) k_ring_lut(hcg_healpix hp, uint32_t n, const uint32_t* __restrict__ keys,
                                                  hcg_ring_meta* __restrict__ meta, uint32_t* __restrict__ lut,
                                                  double* __restrict__ ring_z, double* __restrict__ ring_s) {
  const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
  const hcg_ring_meta m = ring_meta(hp, n, keys);
  if (k == 0) *meta = m;
  if (k > m.usedrings) return;
  if (k == 0) {
    lut[0] = 0;
  } else if (k == m.usedrings) {
    lut[k] = m.n;
  } else {
    uint64_t sp, npr;
    ring_info(hp, (uint64_t)m.firstring + k, sp, npr);
    lut[k] = lower_bound_4(keys, m.n, (uint32_t)sp);
  }
  if (k < m.usedrings) {
    const RingGeom g = ring_geom(hp, (uint64_t)m.firstring + k);
    ring_z[k] = g.z;
    ring_s[k] = g.have_sin ? g.s : -1.0;
  }
}

}  // namespace hcg

using namespace hcg;

namespace {
struct SortWorkspace {
  uint32_t* keys_b;
  uint32_t* vals_b;
  uint32_t* hist;
  uint32_t* digit;
  uint32_t tiles;
};

constexpr size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

constexpr uint32_t sort_tile_of(uint32_t n) {
  return n <= kSmallTile * kSmallTiles ? kSmallTile : n <= kMidTile * kMidTiles ? kMidTile : kLargeTile;
}
constexpr uint32_t sort_tiles_of(uint32_t n) {
  return n ? (uint32_t)(((uint64_t)n + sort_tile_of(n) - 1) / sort_tile_of(n)) : 1u;
}

// Sort scratch for n keys: ping-pong keys and values, per-tile digit
// counts, per-digit totals.  Every byte of it is written before it is read.
constexpr size_t sort_ws_bytes(uint32_t n) {
  return 2 * align256((size_t)n * 4) + align256((size_t)sort_tiles_of(n) * kMaxDigits * 4) +
         align256(kMaxDigits * 4);
}

// The largest need of up to n keys: the small tiles' counts take more than
// those of somewhat more keys in larger tiles.
constexpr size_t sort_ws_bytes_up_to(uint32_t n) {
  return std::max({sort_ws_bytes(n), sort_ws_bytes(std::min(n, kSmallTile * kSmallTiles)),
                   sort_ws_bytes(std::min(n, kMidTile * kMidTiles))});
}

void sort_ws_layout(uint32_t n, void* base, SortWorkspace& ws) {
  const uint32_t tiles = sort_tiles_of(n);
  const size_t kb = align256((size_t)n * 4), hb = align256((size_t)tiles * kMaxDigits * 4);
  char* p = static_cast<char*>(base);
  ws.keys_b = reinterpret_cast<uint32_t*>(p);
  ws.vals_b = reinterpret_cast<uint32_t*>(p + kb);
  ws.hist = reinterpret_cast<uint32_t*>(p + 2 * kb);
  ws.digit = reinterpret_cast<uint32_t*>(p + 2 * kb + hb);
  ws.tiles = tiles;
}

// Argument checks shared by hcg_presort and hcg_presort_noalloc.
int presort_args(const hcg_healpix* hp, uint32_t n, const double* lon_deg, const double* lat_deg,
                 const uint32_t* keys_sorted, const uint32_t* perm, const char* who) {
  if (hp == nullptr) return set_error(HCG_ERR_INVALID, std::string(who) + ": hp is NULL");
  if (keys_sorted == nullptr || perm == nullptr) return set_error(HCG_ERR_INVALID, std::string(who) + ": NULL output");
  if (hp->nside == 0 || hp->nside > HCG_MAX_NSIDE || (hp->nside & (hp->nside - 1)))
    return set_error(HCG_ERR_UNSUPPORTED, std::string(who) + ": nside must be a power of two <= 8192");
  if (n >= 0xFFFFFFFFu) return set_error(HCG_ERR_INVALID, std::string(who) + ": n must be < 2^32-1");
  if (n && (lon_deg == nullptr || lat_deg == nullptr))
    return set_error(HCG_ERR_INVALID, std::string(who) + ": NULL input");
  return HCG_OK;
}

// Keys, the radix passes and the sentinel, on workspace `ws` (n > 0).
template <uint32_t THREADS, uint32_t ITEMS>
int presort_enqueue_as(const hcg_healpix* hp, uint32_t n, const double* lon_deg, const double* lat_deg,
                       uint32_t* keys_sorted, uint32_t* perm, const SortWorkspace& ws, hipStream_t s) {
  const uint32_t npix = (uint32_t)hp->npix, tiles = ws.tiles;
  int bits = 1;
  while ((npix >> bits) != 0) ++bits;  // keys sort as 0 .. npix
  const int passes = bits <= 2 * kMaxDigitBits ? 2 : 3;
  // the last pass writes keys_sorted and perm
  uint32_t *kin = passes == 2 ? keys_sorted : ws.keys_b, *vin = passes == 2 ? perm : ws.vals_b;
  uint32_t *kout = passes == 2 ? ws.keys_b : keys_sorted, *vout = passes == 2 ? ws.vals_b : perm;
  Digit g{npix, 0, 0};
  for (int pass = 0; pass < passes; ++pass) {
    g.shift += g.bits;
    g.bits = (bits - g.shift + passes - pass - 1) / (passes - pass);
    if (pass == 0) {
      k_keys<THREADS, ITEMS>
          <<<sort_blocks(tiles), THREADS, 0, s>>>(*hp, n, lon_deg, lat_deg, kin, keys_sorted + n, g, tiles, ws.hist);
      HCG_CHECK_LAUNCH("k_keys");
    } else {
      k_rs_upsweep<THREADS, ITEMS><<<sort_blocks(tiles), THREADS, 0, s>>>(kin, n, g, tiles, ws.hist);
      HCG_CHECK_LAUNCH("k_rs_upsweep");
    }
    k_rs_scan<<<1u << g.bits, 256, 0, s>>>(ws.hist, tiles, ws.digit);
    HCG_CHECK_LAUNCH("k_rs_scan");
    if (pass == 0)
      k_rs_downsweep<THREADS, ITEMS, true>
          <<<sort_blocks(tiles), THREADS, 0, s>>>(kin, vin, kout, vout, n, g, tiles, ws.hist, ws.digit);
    else
      k_rs_downsweep<THREADS, ITEMS, false>
          <<<sort_blocks(tiles), THREADS, 0, s>>>(kin, vin, kout, vout, n, g, tiles, ws.hist, ws.digit);
    HCG_CHECK_LAUNCH("k_rs_downsweep");
    std::swap(kin, kout);
    std::swap(vin, vout);
  }
  return HCG_OK;
}

int presort_enqueue(const hcg_healpix* hp, uint32_t n, const double* lon_deg, const double* lat_deg,
                    uint32_t* keys_sorted, uint32_t* perm, const SortWorkspace& ws, hipStream_t s) {
  switch (sort_tile_of(n)) {
    case kSmallTile: return presort_enqueue_as<256, 4>(hp, n, lon_deg, lat_deg, keys_sorted, perm, ws, s);
    case kMidTile: return presort_enqueue_as<256, 8>(hp, n, lon_deg, lat_deg, keys_sorted, perm, ws, s);
    default: return presort_enqueue_as<512, 16>(hp, n, lon_deg, lat_deg, keys_sorted, perm, ws, s);
  }
}

// The no-allocation variant's scratch: one sort workspace for up to
// HCG_PRESORT_NOALLOC_MAX_N keys in a file-scope device array.  In host code
// `scratch` names a host-side stand-in, not a device address: its device
// address comes from hipGetSymbolAddress, once per device (each device
// holds its own copy of the array, at its own address).
constexpr size_t kNoAllocScratchBytes = sort_ws_bytes_up_to(HCG_PRESORT_NOALLOC_MAX_N);
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
void* g_scratch_ptr[kMaxDevices] = {};

// The current device's address of `scratch` (resolved on the first call on
// that device).
int scratch_address(void** out) {
  int dev = 0;
  HCG_CHECK_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) return set_error(HCG_ERR_UNSUPPORTED, "hcg_presort_noalloc: device index");
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* ptr = nullptr;
    HCG_CHECK_HIP(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) return set_error(HCG_ERR_HIP, "hcg_presort_noalloc: no device address for the scratch array");
    g_scratch_ptr[dev] = ptr;
  }
  *out = g_scratch_ptr[dev];
  return HCG_OK;
}
}  // namespace

extern "C" size_t hcg_presort_workspace_size(uint32_t n) { return sort_ws_bytes_up_to(n); }

extern "C" int hcg_presort(const hcg_healpix* hp, uint32_t n, const double* lon_deg, const double* lat_deg,
                           uint32_t* keys_sorted, uint32_t* perm, void* workspace, size_t workspace_bytes,
                           void* stream) {
  int rc = presort_args(hp, n, lon_deg, lat_deg, keys_sorted, perm, "hcg_presort");
  if (rc != HCG_OK) return rc;
  hipStream_t s = as_stream(stream);
  if (n == 0) {
    k_set_sentinel<<<1, 64, 0, s>>>(keys_sorted, 0, (uint32_t)hp->npix);
    HCG_CHECK_LAUNCH("k_set_sentinel");
    return HCG_OK;
  }
  if (workspace == nullptr || workspace_bytes < sort_ws_bytes(n))
    return set_error(HCG_ERR_WORKSPACE, "hcg_presort: workspace smaller than hcg_presort_workspace_size(n)");
  SortWorkspace ws;
  sort_ws_layout(n, workspace, ws);
  return presort_enqueue(hp, n, lon_deg, lat_deg, keys_sorted, perm, ws, s);
}

extern "C" int hcg_presort_noalloc(const hcg_healpix* hp, uint32_t n, const double* lon_deg, const double* lat_deg,
                                   uint32_t* keys_sorted, uint32_t* perm, void* stream) {
  int rc = presort_args(hp, n, lon_deg, lat_deg, keys_sorted, perm, "hcg_presort_noalloc");
  if (rc != HCG_OK) return rc;
  if (n > HCG_PRESORT_NOALLOC_MAX_N)
    return set_error(HCG_ERR_UNSUPPORTED, "hcg_presort_noalloc: n exceeds HCG_PRESORT_NOALLOC_MAX_N (8388608); "
                                          "use hcg_presort with a workspace");
  hipStream_t s = as_stream(stream);
  if (n == 0) {
    k_set_sentinel<<<1, 64, 0, s>>>(keys_sorted, 0, (uint32_t)hp->npix);
    HCG_CHECK_LAUNCH("k_set_sentinel");
    return HCG_OK;
  }
  void* base = nullptr;
  rc = scratch_address(&base);
  if (rc != HCG_OK) return rc;
  SortWorkspace ws;
  sort_ws_layout(n, base, ws);
  return presort_enqueue(hp, n, lon_deg, lat_deg, keys_sorted, perm, ws, s);
}

extern "C" int hcg_gather_samples(uint32_t n, const uint32_t* perm, const double* lon_deg, const double* lat_deg,
                                  const void* data, int data_dtype, const double* weights, hcg_sample* records,
                                  double* lon_sorted, double* lat_sorted, double* data_sorted,
                                  double* weights_sorted, void* stream) {
  if (n == 0) return HCG_OK;
  HCG_REQUIRE(perm && lon_deg && lat_deg && records, "hcg_gather_samples: NULL argument");
  HCG_REQUIRE(data_dtype == HCG_DTYPE_F64 || data_dtype == HCG_DTYPE_F32,
              "hcg_gather_samples: data_dtype must be HCG_DTYPE_F64 or HCG_DTYPE_F32");
  const uint32_t blocks = std::min<uint32_t>(ceil_div_u32(n, 256), 8192);
  k_gather<<<blocks, 256, 0, as_stream(stream)>>>(n, perm, lon_deg, lat_deg, data, data_dtype, weights, records,
                                                  lon_sorted, lat_sorted, data_sorted, weights_sorted);
  HCG_CHECK_LAUNCH("k_gather");
  return HCG_OK;
}

extern "C" int hcg_ring_lut(const hcg_healpix* hp, uint32_t n, const uint32_t* keys_sorted, uint32_t* lut,
                            double* ring_z, double* ring_s, hcg_ring_meta* meta, void* stream) {
  HCG_REQUIRE(hp && keys_sorted && lut && ring_z && ring_s && meta, "hcg_ring_lut: NULL argument");
  if (hp->nside == 0 || hp->nside > HCG_MAX_NSIDE)
    return set_error(HCG_ERR_UNSUPPORTED, "hcg_ring_lut: nside must be <= 8192");
  hipStream_t s = as_stream(stream);
  const uint32_t threads = (uint32_t)hp->nrings + 1;
  k_ring_lut<<<ceil_div_u32(threads, 256), 256, 0, s>>>(*hp, n, keys_sorted, meta, lut, ring_z, ring_s);
  HCG_CHECK_LAUNCH("k_ring_lut");
  return HCG_OK;
}
