// The fast GEMM kernels for bf16 activations and bf16 weights.
#include "gemm_lds.h"

namespace we {
hipError_t gemm_lds_bf16_bf16(const FastArgs& a, uint32_t splits, int cfg, int reduce_xcd, hipStream_t s) {
  return launch_fast_types<false, BF16>(a, splits, cfg, reduce_xcd, s);
}
}  // namespace we
