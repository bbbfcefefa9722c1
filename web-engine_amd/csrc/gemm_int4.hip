// int4 weights times 16-bit activations for more rows than the GEMV kernels of gemv_int4.hip share a weight read over:
// the tiles of gemm_lds.h with the weights as stored in LDS (32 bytes per column and 64-k block), unpacked to exact f16
// or bf16 integers in registers. Each 64-k block lies in one scale group: its sums of x q come out of the MFMAs in f32
// and its f16 scale multiplies them there, so the dequantized value q * s is never rounded to 16 bits.
#include <algorithm>

#include "gemm_lds.h"

namespace we {
namespace {

constexpr uint32_t kCUs = 256;

template <bool IS_F16>
hipError_t launch_tile(const FastArgs& a, uint32_t splits, int cfg, int rx, hipStream_t s) {
  if (cfg == GEMM_CFG_128x128) return launch_fast_cfg<128, 128, 1, 4, IS_F16, INT4, 2>(a, splits, rx, s);
  return launch_fast_cfg<64, 64, 2, 2, IS_F16, INT4, 3>(a, splits, rx, s);
}

// 64 x 64 tiles (three workgroups per CU) where 128 x 128 ones (two, of 4 waves of 128 x 32: each weight is unpacked once
// per workgroup) would fill at most a quarter of their slots: 400 x 4096 x 2048 32.9 -> 27.2 us, 2048 x 1024 x 1536 35.2 ->
// 20.8, 128 x 4096 x 4096 25.6 -> 19.4; but 256 x 18944 x 3584 72.5 us with 128 x 128, 89.0 with 64 x 64.
int pick_cfg(const Int4Launch& L) {
  if (L.cfg == GEMM_CFG_128x128 || L.cfg == GEMM_CFG_64x64) return L.cfg;
  const uint64_t tiles128 = (uint64_t)((L.m + 127) / 128) * ((L.n + 127) / 128);
  return L.m <= 64 || tiles128 <= 128 ? GEMM_CFG_64x64 : GEMM_CFG_128x128;
}

}  // namespace

bool int4_gemm_supported(const Int4Launch& L) {
  const uint64_t xb = L.k ? ((uint64_t)(L.m - 1) * L.x_stride + L.k) * 2 : 0;
  // From M 33 on, and where the GEMV kernel's passes over the weights (one per 16 rows) unpack at least 24M values: that
  // kernel takes about 5 us + 0.31 us per million, the tiles (with their reduce pass) no less than 9 us. 17 x 18944 x 3584
  // 34.6 us there against 37.8 us here, 64 x 1024 x 1536 7.2 against 9.6, 100 x 4096 x 4096 43 against 20.
  const uint64_t passes = (L.m + 15) / 16;
  if (L.m <= 32 || passes * L.n * L.k < 24000000ull) return false;
  return (L.x_dtype == F16 || L.x_dtype == BF16) && L.k % 64 == 0 && L.k > 0 && L.path == 0 &&
         (uintptr_t)L.w % 16 == 0 && ((uintptr_t)L.x + (uint64_t)L.x_offset * 2) % 16 == 0 && L.x_stride % 8 == 0 &&
         xb < kInvalid && (uint64_t)L.n * L.k / 2 < kInvalid;
}

GemmReducePlan int4_gemm_plan(const Int4Launch& L) {
  GemmReducePlan p{1, L.k, 0, -1, 1};
  const int cfg = pick_cfg(L);
  const uint32_t bm = cfg == GEMM_CFG_64x64 ? 64 : 128, bn = bm;
  const uint64_t tiles = (uint64_t)((L.m + bm - 1) / bm) * ((L.n + bn - 1) / bn);
  const uint64_t slots = kCUs * (bm == 64 ? 3 : 2);
  if (tiles * 2 > slots) return p;
  uint32_t rs = (uint32_t)((slots + tiles - 1) / tiles);
  rs = std::min(rs, L.k / 256);  // every slice keeps at least 256 of K
  if (rs < 2) return p;
  const uint32_t kc = (L.k + rs * BK - 1) / (rs * BK) * BK;
  const uint32_t slices = (L.k + kc - 1) / kc;
  if (slices < 2) return p;
  return GemmReducePlan{slices, kc, (size_t)slices * L.m * L.n * 4, -1, 1};
}

hipError_t int4_gemm_launch(const Int4Launch& L, hipStream_t stream) {
  const int yb = L.y_dtype == F32 ? 4 : 2;
  FastArgs a{};
  a.x = (const char*)L.x + (uint64_t)L.x_offset * 2;
  a.w = L.w;
  a.y = L.y;
  a.bias = L.bias;
  a.gate = L.gate;
  a.res = L.res;
  a.x_bytes = (uint32_t)(((uint64_t)(L.m - 1) * L.x_stride + L.k) * 2);
  a.w_bytes = (uint32_t)((uint64_t)L.n * L.k / 2);
  a.m = L.m;
  a.n = L.n;
  a.k = L.k;
  a.kwrap = a.kwrap2 = 0xffffffffu;
  a.scale = L.scale;
  a.x_stride = L.x_stride;
  a.w_stride = L.k;
  a.y_stride = L.y_stride;
  a.y_offset = L.y_offset;
  a.kc = L.k;
  a.flags = L.flags;
  a.y_dtype = (uint32_t)L.y_dtype;
  a.vec_store = ((uintptr_t)L.y % (4 * yb) == 0 && (uintptr_t)L.res % (4 * yb) == 0 && (uintptr_t)L.gate % 16 == 0 &&
                 L.y_offset % 4 == 0 && L.y_stride % 4 == 0)
                    ? 1u
                    : 0u;
  a.sc = L.scales;
  a.sc_groups = L.k / L.group;
  a.sc_blocks = L.group / BK;
  uint32_t splits = 1;
  if (L.rsplits > 1) {
    a.part = (float*)L.scratch;
    a.rsplits = splits = L.rsplits;
    a.kc = L.rkc;
  }
  const int cfg = pick_cfg(L);
  return L.x_dtype == F16 ? launch_tile<true>(a, splits, cfg, 1, stream) : launch_tile<false>(a, splits, cfg, 1, stream);
}

}  // namespace we
