// grid_mfma.hip -- the multi-channel entry points: the contraction's launches
// (mfma_kernels.hpp) and its lean instances, block plans, and the channel gather.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "gridcore.hpp"
#include "mfma_job.hpp"
#include "mfma_kernels.hpp"

namespace hcg {

__global__ void __launch_bounds__(64) k_mfma_plan(MfmaJob J, uint32_t first) { plan_tile(J, first + blockIdx.x); }

// The instance of a job: its form (mfma_form) and value type.
static uint32_t nb_of_instance(uint32_t inst) { return kFormNb[inst / 2]; }
bool mfma_uses_plan(uint32_t inst) { return nb_of_instance(inst) == 0; }
uint32_t mfma_instance(const MfmaJob& J) {
  return 2 * mfma_form(J.nchan, mfma_weight_kind(J.kt, J.B.w_s != nullptr)) + (J.dtype == HCG_DTYPE_BF16 ? 0u : 1u);
}
static uint32_t mfma_groups(const MfmaJob& J, uint32_t inst) {
  const uint32_t nb = nb_of_instance(inst);
  return ceil_div_u32(J.nchan, nb ? 16u * nb : 64u * kWideWaves);
}
uint64_t mfma_blocks(const MfmaJob& J) {
  const uint32_t inst = mfma_instance(J);
  return (uint64_t)tile_blocks(J.ntiles, J.tiles_x, nb_of_instance(inst) == 0) * mfma_groups(J, inst);
}

static void launch_instance(uint32_t inst, const MfmaLaunch& L) {
  const uint32_t form = inst / 2;
  if (form < kFormFirst[kWeightSmall])
    launch_forms<kFormFirst[kWeightLean], kFormFirst[kWeightSmall]>(inst, L);
  else if (form < kFormFirst[kWeight2d])
    launch_gauss_forms(inst, L);
  else
    launch_gauss2d_sinc_forms(inst, L);
}

static int launch_mfma_job(const MfmaJob& J, hipStream_t s) {
  const uint32_t inst = mfma_instance(J);
  const uint32_t nb = nb_of_instance(inst), groups = mfma_groups(J, inst);
  if (J.plan) {
    launch_runs(J.ntiles, 64, [&](uint32_t first, uint32_t count) { k_mfma_plan<<<count, 64, 0, s>>>(J, first); });
    HCG_CHECK_LAUNCH("k_mfma_plan");
  }
  launch_runs(tile_blocks(J.ntiles, J.tiles_x, nb == 0), mfma_threads(nb), [&](uint32_t first, uint32_t count) {
    launch_instance(inst, MfmaLaunch{&J, groups, nullptr, 0, nullptr, first, count, s});
  });
  HCG_CHECK_LAUNCH("k_grid_mfma");
  return HCG_OK;
}

int launch_mfma_batch(uint32_t inst, const TileRange* ranges, uint32_t nranges, uint32_t blocks, const MfmaJob* jobs,
                      hipStream_t s) {
  if (nranges == 0 || blocks == 0) return HCG_OK;
  launch_runs(blocks, mfma_threads(nb_of_instance(inst)), [&](uint32_t first, uint32_t count) {
    launch_instance(inst, MfmaLaunch{nullptr, 0, ranges, nranges, jobs, first, count, s});
  });
  HCG_CHECK_LAUNCH("k_grid_mfma_batch");
  return HCG_OK;
}

// Channel gather into the blocked layout: sorted slot i of channel ch goes
// to block i / 8, row ch, column i % 8 ([nblk][nchan][8], kVB = 8 slots per
// block, zero-padded to nblk = hcg_channels_padded_len(n) / 8 blocks).  A
// workgroup takes kGatherSlots sorted slots x kGatherChans channels through
// LDS: thread t gathers slot t of each channel (consecutive lanes read the
// caller's values at consecutive permuted positions, 2 bytes each), and then
// writes block rows (16 bytes each), consecutive threads the consecutive
// channel rows of one block.
constexpr uint32_t kGatherChans = 32;
constexpr uint32_t kGatherSlots = 256;
constexpr uint32_t kGatherRow = kGatherSlots + 8;  // LDS row stride (16-byte pad against bank conflicts)

template <typename T>
__device__ inline void gather_cm_block(uint32_t bx, uint32_t by, uint32_t n, uint32_t n_pad, uint32_t nchan,
                                       const uint32_t* __restrict__ perm, const T* __restrict__ in,
                                       T* __restrict__ out, uint32_t* __restrict__ nonfinite,
                                       uint16_t* __restrict__ lds /* [kGatherChans][kGatherRow] */) {
  static_assert(sizeof(T) == 2, "16-bit values");
  const uint32_t t = threadIdx.x;
  const uint32_t i0 = bx * kGatherSlots;
  const uint32_t ch0 = by * kGatherChans;
  const uint32_t nc = min(kGatherChans, nchan - ch0);
  const uint32_t i = i0 + t;
  uint32_t j = 0;
  if (i < n) {
    j = perm[i];
    if (j >= n) j = i;  // a permutation never holds this; keeps every read in bounds regardless
  }
  // all of the thread's loads first (up to kGatherChans in flight), then
  // the LDS stores
  uint16_t x[kGatherChans];
  const bool live = i < n;
  const T* src = in + (size_t)ch0 * n + j;
#pragma unroll
  for (uint32_t c = 0; c < kGatherChans; ++c)
    x[c] = (live && c < nc) ? __builtin_bit_cast(uint16_t, src[(size_t)c * n]) : (uint16_t)0;
  uint32_t bad = 0;
#pragma unroll
  for (uint32_t c = 0; c < kGatherChans; ++c) {
    if (c < nc) {
      bad += isfinite((float)__builtin_bit_cast(T, x[c])) ? 0u : 1u;
      lds[c * kGatherRow + t] = x[c];
    }
  }
  if (nonfinite && bad) atomicAdd(nonfinite, bad);
  __syncthreads();
  // pieces: (block b of the workgroup's slots, channel c) -> one block row
  // of kVB values; the output is 16-byte aligned when the buffer is (a row
  // is 16 bytes)
  static_assert(kVB == 8 && kGatherSlots % kVB == 0, "a block row is one 16-byte piece");
  const bool vec = (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
  const uint32_t npieces = (kGatherSlots / kVB) * nc;
  for (uint32_t p = t; p < npieces; p += 256) {
    const uint32_t b = p / nc, c = p % nc;
    const uint32_t blk = i0 / kVB + b;
    if (blk * kVB >= n_pad) continue;
    const uint16_t* src = lds + c * kGatherRow + b * kVB;
    T* dst = out + ((size_t)blk * nchan + ch0 + c) * kVB;
    if (vec) {
      *reinterpret_cast<uint4*>(dst) = *reinterpret_cast<const uint4*>(src);
    } else {
#pragma unroll
      for (uint32_t e = 0; e < 8; ++e) dst[e] = __builtin_bit_cast(T, src[e]);
    }
  }
}

template <typename T>
__global__ void __launch_bounds__(256) k_gather_channels_cm(uint32_t n, uint32_t n_pad, uint32_t nchan,
                                                            const uint32_t* __restrict__ perm,
                                                            const T* __restrict__ in, T* __restrict__ out,
                                                            uint32_t* __restrict__ nonfinite) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[kGatherChans * kGatherRow];
  gather_cm_block<T>(blockIdx.x, blockIdx.y, n, n_pad, nchan, perm, in, out, nonfinite, lds);
}

// Sample-major input ([n][nchan]): a lane makes whole block rows (8 samples of
// a channel, 16 bytes) from eight 2-byte loads; consecutive lanes take the
// rows in output order, so that they read a sample's channels and write a
// block's rows side by side, kGatherRows rows a lane with all loads in
// flight.  Memory bound: 2M x 1024 values (8.2 GB moved) 1.58 ms, and 4.86
// with 64 x 64 tiles transposed in LDS; 482k x 67 values 25 us, then 100.
constexpr uint32_t kGatherRows = 2;
inline uint32_t gather_sm_gx(uint32_t n_pad, uint32_t nchan) {
  return ceil_div_u32((uint64_t)(n_pad / kVB) * nchan, 256u * kGatherRows);
}
template <typename T>
__device__ inline void gather_sm_block(uint32_t bx, uint32_t n, uint32_t n_pad, uint32_t nchan,
                                       const uint32_t* __restrict__ perm, const T* __restrict__ in,
                                       T* __restrict__ out, uint32_t* __restrict__ nonfinite) {
  static_assert(sizeof(T) == 2 && kVB == 8, "a block row is one 16-byte piece");
  const uint64_t rows = (uint64_t)(n_pad / kVB) * nchan;
  uint16_t x[kGatherRows][kVB];
#pragma unroll
  for (uint32_t k = 0; k < kGatherRows; ++k) {
    const uint64_t row = ((uint64_t)bx * kGatherRows + k) * 256u + threadIdx.x;
    const uint32_t i0 = (uint32_t)(row / nchan) * kVB, ch = (uint32_t)(row % nchan);
#pragma unroll
    for (uint32_t e = 0; e < kVB; ++e) {
      const uint32_t i = i0 + e;
      x[k][e] = 0;
      if (row < rows && i < n) {
        uint32_t j = perm[i];
        if (j >= n) j = i;  // a permutation never holds this; keeps every read in bounds regardless
        x[k][e] = __builtin_bit_cast(uint16_t, in[(size_t)j * nchan + ch]);
      }
    }
  }
  uint32_t bad = 0;
#pragma unroll
  for (uint32_t k = 0; k < kGatherRows; ++k) {
    const uint64_t row = ((uint64_t)bx * kGatherRows + k) * 256u + threadIdx.x;
    if (row < rows) {
#pragma unroll
      for (uint32_t e = 0; e < kVB; ++e) bad += isfinite((float)__builtin_bit_cast(T, x[k][e])) ? 0u : 1u;
      __builtin_memcpy(out + row * kVB, x[k], 16);
    }
  }
  if (nonfinite && bad) atomicAdd(nonfinite, bad);
}

template <typename T>
__global__ void __launch_bounds__(256) k_gather_channels_sm(uint32_t n, uint32_t n_pad, uint32_t nchan,
                                                            const uint32_t* __restrict__ perm,
                                                            const T* __restrict__ in, T* __restrict__ out,
                                                            uint32_t* __restrict__ nonfinite, uint32_t first) {
  gather_sm_block<T>(first + blockIdx.x, n, n_pad, nchan, perm, in, out, nonfinite);
}

// Every job's channel gather and block plan (mfma_wide) of a batch in one
// launch (prep_ranges): the plans' dependent key searches are latency-bound
// and the gathers bandwidth-bound, so sharing the chip lets each hide the
// other.  A range is a run of workgroups of one kind for one job; each
// workgroup finds its range by binary search over the range starts.
__global__ void __launch_bounds__(256) k_batch_prep(const PrepRange* __restrict__ ranges, uint32_t nranges,
                                                    const PrepJob* __restrict__ pj,
                                                    const MfmaJob* __restrict__ jobs, uint32_t first) {
  __shared__ __attribute__((aligned(16))) uint16_t smem[kGatherChans * kGatherRow];
  const uint32_t block = first + blockIdx.x;
  uint32_t lo = 0, hi = nranges;  // last range with first <= block
  while (hi - lo > 1) {
    const uint32_t mid = (lo + hi) >> 1;
    if (ranges[mid].first <= block)
      lo = mid;
    else
      hi = mid;
  }
  const PrepRange R = ranges[lo];
  const uint32_t lb = block - R.first;
  const PrepJob& G = pj[R.job];
  const MfmaJob& J = jobs[R.job];
  const uint32_t bx = lb % R.gx, by = lb / R.gx;
  switch (R.kind) {
    case kPrepPlan: {
      const uint32_t t = lb * 4 + (threadIdx.x >> 6);  // a wave per block
      if (t < J.ntiles) plan_tile(J, t);
      break;
    }
    case kPrepGatherCm:
      if (J.dtype == HCG_DTYPE_BF16)
        gather_cm_block<__bf16>(bx, by, G.n, J.n_pad, J.nchan, G.perm, static_cast<const __bf16*>(G.in),
                                static_cast<__bf16*>(const_cast<void*>(J.vs)), G.nonfinite, smem);
      else
        gather_cm_block<_Float16>(bx, by, G.n, J.n_pad, J.nchan, G.perm, static_cast<const _Float16*>(G.in),
                                  static_cast<_Float16*>(const_cast<void*>(J.vs)), G.nonfinite, smem);
      break;
    default:  // kPrepGatherSm
      if (J.dtype == HCG_DTYPE_BF16)
        gather_sm_block<__bf16>(lb, G.n, J.n_pad, J.nchan, G.perm, static_cast<const __bf16*>(G.in),
                                static_cast<__bf16*>(const_cast<void*>(J.vs)), G.nonfinite);
      else
        gather_sm_block<_Float16>(lb, G.n, J.n_pad, J.nchan, G.perm, static_cast<const _Float16*>(G.in),
                                  static_cast<_Float16*>(const_cast<void*>(J.vs)), G.nonfinite);
      break;
  }
}

int prep_ranges(uint32_t njobs, const MfmaJob* jobs, const uint32_t* layouts, std::vector<PrepRange>& out,
                uint32_t* blocks) {
  out.clear();
  uint64_t first = 0;
  auto add = [&](uint32_t j, uint32_t kind, uint32_t gx, uint64_t blocks) {
    if (blocks == 0) return;
    out.push_back(PrepRange{(uint32_t)first, j, kind, gx});
    first += blocks;
  };
  // plans first: their workgroups run longest
  for (uint32_t j = 0; j < njobs; ++j)
    if (jobs[j].plan && jobs[j].nchan) add(j, kPrepPlan, 1, ceil_div_u32(jobs[j].ntiles, 4));
  for (uint32_t j = 0; j < njobs; ++j) {
    const MfmaJob& J = jobs[j];
    if (J.nchan == 0 || J.n_pad == 0) continue;
    if (layouts[j] == 0) {
      const uint32_t gx = ceil_div_u32(J.n_pad, kGatherSlots), gy = ceil_div_u32(J.nchan, kGatherChans);
      add(j, kPrepGatherCm, gx, (uint64_t)gx * gy);
    } else {
      const uint32_t gx = gather_sm_gx(J.n_pad, J.nchan);
      add(j, kPrepGatherSm, gx, gx);
    }
  }
  if (first >= 0x7FFFFFFFull) return set_error(HCG_ERR_INVALID, "hcg_batch_create: too many prep workgroups");
  *blocks = (uint32_t)first;
  return HCG_OK;
}

int launch_batch_prep(const PrepRange* ranges, uint32_t nranges, uint32_t blocks, const PrepJob* pj,
                      const MfmaJob* jobs, hipStream_t s) {
  if (nranges == 0 || blocks == 0) return HCG_OK;
  launch_runs(blocks, 256, [&](uint32_t first, uint32_t count) {
    k_batch_prep<<<count, 256, 0, s>>>(ranges, nranges, pj, jobs, first);
  });
  HCG_CHECK_LAUNCH("k_batch_prep");
  return HCG_OK;
}

}  // namespace hcg

using namespace hcg;

extern "C" uint32_t hcg_channels_padded_len(uint32_t n) { return ((n + 31u) & ~31u) + 64u; }

extern "C" int hcg_gather_channels(uint32_t n, uint32_t nchan, const uint32_t* perm, const void* values, int dtype,
                                   int layout, void* values_sorted, uint32_t* nonfinite, void* stream) {
  if (n == 0 || nchan == 0) return HCG_OK;
  HCG_REQUIRE(perm && values && values_sorted, "hcg_gather_channels: NULL buffer");
  HCG_REQUIRE(dtype == HCG_DTYPE_BF16 || dtype == HCG_DTYPE_F16, "hcg_gather_channels: dtype must be BF16 or F16");
  HCG_REQUIRE(layout == 0 || layout == 1, "hcg_gather_channels: layout must be 0 (channel-major) or 1 (sample-major)");
  const uint32_t n_pad = hcg_channels_padded_len(n);
  hipStream_t s = as_stream(stream);
  if (layout == 0) {
    const dim3 grid(ceil_div_u32(n_pad, kGatherSlots), ceil_div_u32(nchan, kGatherChans));
    if (dtype == HCG_DTYPE_BF16)
      k_gather_channels_cm<__bf16><<<grid, 256, 0, s>>>(n, n_pad, nchan, perm, static_cast<const __bf16*>(values),
                                                        static_cast<__bf16*>(values_sorted), nonfinite);
    else
      k_gather_channels_cm<_Float16><<<grid, 256, 0, s>>>(n, n_pad, nchan, perm,
                                                          static_cast<const _Float16*>(values),
                                                          static_cast<_Float16*>(values_sorted), nonfinite);
  } else {
    launch_runs(gather_sm_gx(n_pad, nchan), 256, [&](uint32_t first, uint32_t count) {
      if (dtype == HCG_DTYPE_BF16)
        k_gather_channels_sm<__bf16><<<count, 256, 0, s>>>(n, n_pad, nchan, perm, static_cast<const __bf16*>(values),
                                                           static_cast<__bf16*>(values_sorted), nonfinite, first);
      else
        k_gather_channels_sm<_Float16><<<count, 256, 0, s>>>(n, n_pad, nchan, perm,
                                                             static_cast<const _Float16*>(values),
                                                             static_cast<_Float16*>(values_sorted), nonfinite, first);
    });
  }
  HCG_CHECK_LAUNCH("k_gather_channels");
  return HCG_OK;
}

extern "C" size_t hcg_grid_mfma_workspace_size(uint32_t side, const hcg_mfma_shape* shape) {
  const uint32_t tc = (shape && shape->tile_cols) ? shape->tile_cols : kMcDefaultTileCols;
  if (!(tc == 8 || tc == 16 || tc == 32 || tc == 64)) return 0;
  const size_t ntiles = (size_t)ceil_div_u32(side, tc) * ceil_div_u32(side, 64u / tc);
  return ntiles * kPlanBytes;
}

extern "C" int hcg_grid_mfma_ex(const hcg_healpix* hp, const hcg_kernel* kern, uint32_t side, uint32_t n,
                                uint32_t nchan, int dtype, const hcg_sample* records, const uint32_t* keys_sorted,
                                const double* lon_sorted, const double* lat_sorted, const double* weights_sorted,
                                const void* values_sorted, const uint32_t* lut, const double* ring_z,
                                const double* ring_s, const hcg_ring_meta* meta, const double* xwcs,
                                const double* ywcs, float* cube, float* wsum, int normalize,
                                const hcg_mfma_shape* shape, void* workspace, size_t workspace_bytes,
                                void* stream) {
  HCG_REQUIRE(hp && kern, "hcg_grid_mfma: NULL hp/kern");
  if (hp->nside == 0 || hp->nside > HCG_MAX_NSIDE)
    return set_error(HCG_ERR_UNSUPPORTED, "hcg_grid_mfma: nside must be <= 8192");
  HCG_REQUIRE(kern->kernel_type >= HCG_GAUSS1D && kern->kernel_type <= HCG_TAPERED_SINC,
              "hcg_grid_mfma: unknown kernel type");
  HCG_REQUIRE(kern->factor >= 1, "hcg_grid_mfma: factor must be >= 1");
  HCG_REQUIRE(kern->selection <= HCG_SELECT_DISC,
              "hcg_grid_mfma: selection must be HCG_SELECT_COMPAT or HCG_SELECT_DISC");
  HCG_REQUIRE(dtype == HCG_DTYPE_BF16 || dtype == HCG_DTYPE_F16, "hcg_grid_mfma: dtype must be BF16 or F16");
  HCG_REQUIRE(side <= 65535, "hcg_grid_mfma: side must be <= 65535");
  hcg_mfma_shape sh = shape ? *shape : hcg_mfma_shape{0, 0, 0, 0};
  HCG_REQUIRE(sh.tile_cols == 0 || sh.tile_cols == 8 || sh.tile_cols == 16 || sh.tile_cols == 32 ||
                  sh.tile_cols == 64,
              "hcg_grid_mfma: shape.tile_cols must be 0, 8, 16, 32 or 64");
  HCG_REQUIRE(sh.waves == 0 || sh.waves == 1 || sh.waves == 2 || sh.waves == 4 || sh.waves == 8,
              "hcg_grid_mfma: shape.waves must be 0, 1, 2, 4 or 8");
  HCG_REQUIRE(sh.chunk == 0 || sh.chunk == 128 || sh.chunk == 256 || sh.chunk == 512,
              "hcg_grid_mfma: shape.chunk must be 0, 128, 256 or 512");
  if (side == 0 || nchan == 0) return HCG_OK;
  HCG_REQUIRE(records && keys_sorted && lon_sorted && lat_sorted && values_sorted && lut && ring_z && ring_s && meta &&
                  xwcs && ywcs && cube,
              "hcg_grid_mfma: NULL buffer");
  hipStream_t s = as_stream(stream);
  GridParams P = make_grid_params(hp, kern, side);
  GridBuffers B{records, keys_sorted, lon_sorted, lat_sorted, weights_sorted, lut, ring_z, ring_s, meta,
                xwcs,    ywcs,        nullptr,    nullptr};
  const uint32_t route = route_of(P, kern->kernel_type, weights_sorted != nullptr, nchan, n);
  if (route != kRouteMfma) {
    const TileOut O{static_cast<const uint16_t*>(values_sorted), cube, wsum, dtype == HCG_DTYPE_BF16 ? 1u : 0u,
                    (uint32_t)(normalize ? 1 : 0), nchan};
    return route == kRouteFew ? launch_tiles_few_channels(P, B, O, s) : launch_tiles_one_channel(P, B, O, s);
  }
  const uint32_t tc = sh.tile_cols ? sh.tile_cols : kMcDefaultTileCols;
  const uint32_t tiles_x = ceil_div_u32(side, tc), ntiles = tiles_x * ceil_div_u32(side, 64u / tc);
  if (workspace && workspace_bytes < hcg_grid_mfma_workspace_size(side, &sh))
    return set_error(HCG_ERR_WORKSPACE, "hcg_grid_mfma_ex: workspace smaller than hcg_grid_mfma_workspace_size");
  MfmaJob J{P,     B,    values_sorted,   cube,    wsum,   mfma_weight_form(P, kern->kernel_type),
                  hcg_channels_padded_len(n), nchan, (uint32_t)dtype, tile_shift_of(tc), tiles_x, ntiles,
                  (uint32_t)(normalize ? 1 : 0), nullptr};
  if (workspace && mfma_uses_plan(mfma_instance(J))) J.plan = workspace;
  return launch_mfma_job(J, s);
}

extern "C" int hcg_grid_mfma(const hcg_healpix* hp, const hcg_kernel* kern, uint32_t side, uint32_t n, uint32_t nchan,
                             int dtype, const hcg_sample* records, const uint32_t* keys_sorted,
                             const double* lon_sorted, const double* lat_sorted, const double* weights_sorted,
                             const void* values_sorted, const uint32_t* lut, const double* ring_z,
                             const double* ring_s, const hcg_ring_meta* meta, const double* xwcs, const double* ywcs,
                             float* cube, float* wsum, int normalize, void* stream) {
  return hcg_grid_mfma_ex(hp, kern, side, n, nchan, dtype, records, keys_sorted, lon_sorted, lat_sorted,
                          weights_sorted, values_sorted, lut, ring_z, ring_s, meta, xwcs, ywcs, cube, wsum, normalize,
                          nullptr, nullptr, 0, stream);
}

extern "C" int hcg_grid_mfma_shaped(const hcg_healpix* hp, const hcg_kernel* kern, uint32_t side, uint32_t n,
                                    uint32_t nchan, int dtype, const hcg_sample* records, const uint32_t* keys_sorted,
                                    const double* lon_sorted, const double* lat_sorted, const double* weights_sorted,
                                    const void* values_sorted, const uint32_t* lut, const double* ring_z,
                                    const double* ring_s, const hcg_ring_meta* meta, const double* xwcs,
                                    const double* ywcs, float* cube, float* wsum, int normalize,
                                    const hcg_mfma_shape* shape, void* stream) {
  return hcg_grid_mfma_ex(hp, kern, side, n, nchan, dtype, records, keys_sorted, lon_sorted, lat_sorted,
                          weights_sorted, values_sorted, lut, ring_z, ring_s, meta, xwcs, ywcs, cube, wsum, normalize,
                          shape, nullptr, 0, stream);
}
