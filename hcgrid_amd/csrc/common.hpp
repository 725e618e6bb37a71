// common.hpp -- error plumbing and small device helpers shared by the kernels.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string>

#include "hcgrid_amd.h"

namespace hcg {

// Records the detail of the calling thread's last failure and returns `code`.
int set_error(int code, const std::string& msg);

#define HCG_CHECK_HIP(expr)                                                              \
  do {                                                                                   \
    hipError_t e_ = (expr);                                                              \
    if (e_ != hipSuccess)                                                                \
      return ::hcg::set_error(HCG_ERR_HIP, std::string(#expr ": ") + hipGetErrorString(e_)); \
  } while (0)

#define HCG_CHECK_LAUNCH(name)                                                           \
  do {                                                                                   \
    hipError_t e_ = hipGetLastError();                                                   \
    if (e_ != hipSuccess)                                                                \
      return ::hcg::set_error(HCG_ERR_HIP, std::string(name " launch: ") + hipGetErrorString(e_)); \
  } while (0)

#define HCG_REQUIRE(cond, msg)                                                           \
  do {                                                                                   \
    if (!(cond)) return ::hcg::set_error(HCG_ERR_INVALID, msg);                          \
  } while (0)

inline hipStream_t as_stream(void* s) { return reinterpret_cast<hipStream_t>(s); }

inline uint32_t ceil_div_u32(uint64_t a, uint64_t b) { return (uint32_t)((a + b - 1) / b); }

// A launch counts its threads in 32 bits (HIP refuses more): work of `blocks`
// workgroups goes as launch(first, count) over runs of at most this many, a
// multiple of 8, so that workgroup first + b runs on XCD b % 8 as in one launch.
constexpr uint32_t max_launch_blocks(uint32_t threads) { return 0xFFFFFFFFu / threads & ~7u; }
template <class F>
inline void launch_runs(uint64_t blocks, uint32_t threads, F&& launch) {
  const uint32_t most = max_launch_blocks(threads);
  for (uint64_t first = 0; first < blocks; first += most)
    launch((uint32_t)first, (uint32_t)(blocks - first < most ? blocks - first : most));
}

__device__ inline uint64_t lanemask_lt() {
  const uint32_t lane = __lane_id();
  return lane ? (~0ull >> (64 - lane)) : 0ull;
}

}  // namespace hcg
