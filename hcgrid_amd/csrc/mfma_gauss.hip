// mfma_gauss.hip -- the contraction's GAUSS1D instances besides the lean ones:
// sample weights, and radii outside the lean weight's.
#include <hip/hip_runtime.h>

#include "mfma_job.hpp"
#include "mfma_kernels.hpp"

namespace hcg {

void launch_gauss_forms(uint32_t inst, const MfmaLaunch& L) {
  launch_forms<kFormFirst[kWeightSmall], kFormFirst[kWeight2d]>(inst, L);
}

}  // namespace hcg
