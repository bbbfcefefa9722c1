// The fast GEMM kernels for f16 activations and f16 weights.
#include "gemm_lds.h"

namespace we {
hipError_t gemm_lds_f16_f16(const FastArgs& a, uint32_t splits, int cfg, int reduce_xcd, hipStream_t s) {
  return launch_fast_types<true, F16>(a, splits, cfg, reduce_xcd, s);
}
}  // namespace we
