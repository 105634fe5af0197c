// dpd_gemm_f64.hip -- the packed-panel GEMM kernels of one precision (dpd_gemm_fr.hpp).
#include "dpd_gemm_fr.hpp"

namespace dpd {
hipError_t launch_fr_f64(const GemmLaunch& g, const GroupTab* gt, const void* PA, const void* PB, hipStream_t s) {
  return fr::launch_shape<PREC_F64, 1>(g, gt, PA, PB, s);
}
}  // namespace dpd
