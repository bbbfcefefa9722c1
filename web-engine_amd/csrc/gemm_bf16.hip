// The general GEMM kernels for bf16 activations.
#include "gemm_general.h"

namespace we {
hipError_t gemm_general_bf16(int w_dtype, const GemmArgs& a, uint32_t splits, int cfg, hipStream_t s) {
  return launch_w<BF16>(w_dtype, a, splits, cfg, s);
}
}  // namespace we
