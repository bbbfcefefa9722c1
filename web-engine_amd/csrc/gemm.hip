// Host side of the general GEMM (gemm_general.h): the tile shape of a launch, and the fast path before it.
#include "gemm_general.h"

namespace we {

static bool aligned16(const void* p, uint64_t elems_offset, uint64_t stride, int bytes) {
  return (((uintptr_t)p) % 16 == 0) && ((elems_offset * bytes) % 16 == 0) && ((stride * bytes) % 16 == 0);
}

int pick_gemm_cfg(uint32_t m, uint32_t n, uint32_t splits) {
  if (m <= 32) return GEMM_CFG_32x64;
  if (m <= 64) return GEMM_CFG_64x64;
  const uint64_t big = (uint64_t)((m + 255) / 256) * ((n + 255) / 256) * splits;
  if (m >= 256 && n >= 256 && big >= 512) return GEMM_CFG_256x256;
  const uint64_t mid = (uint64_t)((m + 255) / 256) * ((n + 127) / 128) * splits;
  if (m >= 256 && mid >= 256) return GEMM_CFG_256x128;
  return GEMM_CFG_128x128;
}

hipError_t gemm_launch(const GemmLaunch& L, hipStream_t stream) {
  if (!L.generic && !L.conv_width) {
    const hipError_t e = gemm_fast_launch(L, stream);
    if (e != hipErrorNotSupported || L.k_wrap) return e;  // planes of x (k_wrap) exist for the fast path only
  }
  GemmArgs a{};
  a.x = L.x;
  a.w = L.w;
  a.y = L.y;
  a.bias = L.bias;
  a.gate = L.gate;
  a.res = L.res;
  a.m = L.m;
  a.n = L.n;
  a.k = L.k;
  a.scale = L.scale;
  a.x_stride = L.x_stride;
  a.w_stride = L.w_stride;
  a.y_stride = L.y_stride;
  a.x_offset = L.x_offset;
  a.w_offset = L.w_offset;
  a.y_offset = L.y_offset;
  a.flags = L.flags;
  a.y_dtype = (uint32_t)L.y_dtype;
  a.mul = (uint32_t)L.mul;
  a.conv_width = L.conv_width;
  a.conv_cin = L.conv_cin;
  a.only_if = L.only_if;
  const uint32_t splits = L.splits < 1 ? 1 : L.splits;
  a.kc = splits > 1 ? L.kc : L.k;
  const int xb = L.x_dtype == F32 ? 4 : 2;
  const int wb = L.w_dtype == F32 ? 4 : (L.w_dtype == FP8 ? 1 : 2);
  a.aligned = aligned16(L.x, L.x_offset, L.x_stride, xb) && aligned16(L.w, L.w_offset, L.w_stride, wb) &&
              ((uint64_t)a.kc * xb) % 16 == 0 && ((uint64_t)a.kc * wb) % 16 == 0;
  // f32 x against 16-bit or fp8 weights holds three planes of x: a 128 x 128 tile takes 128 KB, one workgroup of 4 waves per
  // CU. 64 x 64 is faster where such tiles leave half of the CUs idle or K is short: 1024 x 32 x 6144 in 24 K slices 29.8 ->
  // 18.2 us, 1024 x 6144 x 32 73 -> 35, 300 x 3072 x 3080 529 -> 274; not at 1024 x 3072 x 3080 (286, 304 with 64 x 64)
  const uint64_t tiles128 = (uint64_t)((L.m + 127) / 128) * ((L.n + 127) / 128) * splits;
  const bool small = L.x_dtype == F32 && L.m > 64 && (tiles128 < 128 || L.k <= 256 || L.n <= 64);
  const int cfg = L.cfg >= 0 ? L.cfg : small ? (int)GEMM_CFG_64x64 : pick_gemm_cfg(L.m, L.n, splits);
  switch (L.x_dtype) {
    case BF16: return gemm_general_bf16(L.w_dtype, a, splits, cfg, stream);
    case F16: return gemm_general_f16(L.w_dtype, a, splits, cfg, stream);
    default: return gemm_general_f32(L.w_dtype, a, splits, cfg, stream);
  }
}

}  // namespace we
