// mfma_gauss2d_sinc.hip -- the contraction's GAUSS2D and TAPERED_SINC instances,
// and those that evaluate any weight by calls.
#include <hip/hip_runtime.h>

#include "mfma_job.hpp"
#include "mfma_kernels.hpp"

namespace hcg {

void launch_gauss2d_sinc_forms(uint32_t inst, const MfmaLaunch& L) {
  launch_forms<kFormFirst[kWeight2d], kForms>(inst, L);
}

}  // namespace hcg
