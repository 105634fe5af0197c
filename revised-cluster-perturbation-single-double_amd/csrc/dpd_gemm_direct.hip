// dpd_gemm_direct.hip -- FP64 GEMM with one operand in panels and the other read
// where it lies (dpd_gemm_fr.hpp).
#include "dpd_gemm_fr.hpp"

namespace dpd {
hipError_t launch_fr_direct(const GemmLaunch& g, const void* PB, hipStream_t s) {
  if (g.nwg == 0) return hipSuccess;
  return fr::launch_direct<1>(g, PB, s);
}
}  // namespace dpd
