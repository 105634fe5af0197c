// dpd_gemm_bf16x3.hip -- the packed-panel GEMM kernels of one precision (dpd_gemm_fr.hpp).
#include "dpd_gemm_fr.hpp"

namespace dpd {
hipError_t launch_fr_bf16x3(const GemmLaunch& g, const GroupTab* gt, const void* PA, const void* PB, hipStream_t s) {
  return fr::launch_shape<PREC_BF16X3, 1>(g, gt, PA, PB, s);
}
}  // namespace dpd
