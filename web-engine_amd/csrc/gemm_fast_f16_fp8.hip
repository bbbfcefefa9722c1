// The fast GEMM kernels for f16 activations and fp8 weights.
#include "gemm_lds.h"

namespace we {
hipError_t gemm_lds_f16_fp8(const FastArgs& a, uint32_t splits, int cfg, int reduce_xcd, hipStream_t s) {
  return launch_fast_types<true, FP8>(a, splits, cfg, reduce_xcd, s);
}
}  // namespace we
