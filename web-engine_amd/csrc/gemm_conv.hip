// The 3x3 convolution of an f32 channel-last image (src/kernels/matmul.ts:74-83) on the tiles of gemm_lds.h. The image
// and f32 weights are split into two f16 planes each in scratch (kernels_misc.hip), bf16 weights into one, and one GEMM
// runs over the plane products lo x hi, hi x lo, hi x hi (bf16 weights: lo x w, hi x w) along K, with the pixels of each
// tap gathered by the direct-to-LDS loads' addresses; lo planes carry another 2^12, which the sums lose before hi x hi. 128 x 128 pixels, 384 -> 384 channels: 3 x 43.5 GFLOP of MFMA.
#include <algorithm>

#include "gemm_lds.h"

namespace we {
namespace {

constexpr uint32_t kCUs = 256;

struct Plan {
  int cfg;
  uint32_t rsplits, rkc, kp, segments;
  size_t image, weights, col_scale, misc, part, bytes;  // scratch offsets and size
};

size_t round256(size_t n) { return (n + 255) / 256 * 256; }

// Tile shape and K slices by predicted time: rounds of resident workgroups times a tile's time at the shape's rate, and
// the partial sums' traffic.
void pick(const GemmLaunch& L, uint32_t k, Plan& p) {
  struct Cand {
    int cfg;
    uint32_t bm, bn, per_cu;
    double rate;  // TFLOP/s of the chip full of such tiles
  };
  const Cand cands[] = {{GEMM_CFG_256x192, 256, 192, 1, 1000.0}, {GEMM_CFG_128x128, 128, 128, 2, 800.0},
                        {GEMM_CFG_64x64, 64, 64, 3, 500.0}};
  double best = 1e30;
  p.cfg = GEMM_CFG_64x64;
  p.rsplits = 1;
  p.rkc = k;
  for (const Cand& c : cands) {
    if (L.cfg >= 0 && c.cfg != L.cfg && (L.cfg == GEMM_CFG_256x192 || L.cfg == GEMM_CFG_128x128 || L.cfg == GEMM_CFG_64x64))
      continue;
    const uint64_t tiles = (uint64_t)((L.m + c.bm - 1) / c.bm) * ((L.n + c.bn - 1) / c.bn);
    const uint64_t slots = (uint64_t)kCUs * c.per_cu;
    for (uint32_t rs = 1; rs <= 16 && k / rs >= 512; rs++) {
      const uint32_t kc = (k + rs * BK - 1) / (rs * BK) * BK;
      const uint32_t slices = (k + kc - 1) / kc;
      if (slices != rs) continue;
      const uint64_t rounds = (tiles * rs + slots - 1) / slots;
      const double tile_us = 2.0 * c.bm * c.bn * (kc + 256.0) * c.per_cu * kCUs / (c.rate * 1e6);
      const double reduce_us = rs > 1 ? 3.0 + 4.0 * L.m * L.n * (rs + 1.0) / 3e6 : 0.0;
      const double t = (double)rounds * tile_us + reduce_us;
      if (t < best) {
        best = t;
        p.cfg = c.cfg;
        p.rsplits = rs;
        p.rkc = kc;
      }
    }
  }
}

bool make_plan(const GemmLaunch& L, Plan& p) {
  if (!L.conv_width || L.generic || L.x_dtype != F32 || (L.w_dtype != F32 && L.w_dtype != BF16)) return false;
  if (L.conv_cin % 8 || L.splits > 1 || (L.flags & WE_EPI_SPLIT_K_BIT) || L.m == 0 || L.n == 0) return false;
  const int wb = L.w_dtype == F32 ? 4 : 2;
  if ((uintptr_t)L.x % 16 || ((uintptr_t)L.w + (uint64_t)L.w_offset * wb) % 16 || ((uint64_t)L.w_stride * wb) % 16)
    return false;
  if (L.conv_cin > 4096) return false;  // the tap of a k (below 2^16) by one multiplication
  // The four launches take about 15 us whatever the size; the general kernel's one is faster where K is short. f32 weights,
  // 64 x 64 pixels -> 32 channels: from 8 channels 14.8 us there and 17.1 here, from 16 19.1 and 18.8. bf16 weights -> 32:
  // 4 x 4 pixels of 8 channels 9.1 and 14.8, 8 x 8 of 16 13.7 and 15.8, 8 x 8 of 32 19.0 and 18.2, 16 x 16 of 8 21.9 and
  // 15.3, 2 x 2 of 48 20.0 and 20.1. (A forced tile shape stays.)
  const bool pays = L.w_dtype == F32 ? L.conv_cin >= 16 : L.conv_cin >= 48 || (uint64_t)L.m * L.conv_cin >= 2048;
  if (L.cfg < 0 && !pays) return false;
  p.kp = (9 * L.conv_cin + BK - 1) / BK * BK;
  p.segments = L.w_dtype == F32 ? 3 : 2;
  const uint64_t image = (uint64_t)L.m * L.conv_cin * 4, weights = (uint64_t)L.n * p.kp * 2 * (p.segments - 1);
  if (image >= (1u << 30) || weights >= (1u << 30)) return false;
  pick(L, p.kp * p.segments, p);
  p.image = 0;
  p.weights = round256(image);
  p.col_scale = p.weights + round256(weights);
  p.misc = p.col_scale + round256((size_t)L.n * 4);  // the image's inverse scale and flag, then its partial maxima
  p.part = p.misc + 256 + kImageParts * 8;
  p.bytes = p.part + (p.rsplits > 1 ? (size_t)p.rsplits * L.m * L.n * 4 : 0);
  return true;
}

}  // namespace

size_t conv_fast_scratch(const GemmLaunch& L) {
  Plan p;
  return make_plan(L, p) ? p.bytes : 0;
}

hipError_t conv_fast_launch(const GemmLaunch& L, void* scratch, hipStream_t s) {
  Plan p;
  if (!make_plan(L, p)) return hipErrorNotSupported;
  char* base = (char*)scratch;
  uint16_t* image = (uint16_t*)(base + p.image);
  uint16_t* weights = (uint16_t*)(base + p.weights);
  float* col_scale = (float*)(base + p.col_scale);
  float* inv = (float*)(base + p.misc);
  uint32_t* range = (uint32_t*)(base + p.misc + 128);
  hipError_t e =
      launch_image_f16x2((const float*)L.x, L.m, L.conv_cin, (uint32_t*)(base + p.misc + 256), image, inv, range, s);
  if (e != hipSuccess) return e;
  const int wb = L.w_dtype == F32 ? 4 : 2, wplanes = (int)p.segments - 1;
  // weight rows hi | lo (f32) or hi (bf16: 8 significant bits, exact in f16 down to 2^-31 of the row's largest: tiny ones are
  // those below, too)
  e = launch_split_f32_f16x2((const char*)L.w + (uint64_t)L.w_offset * wb, L.w_dtype, L.n, L.k, L.w_stride, weights, p.kp,
                             wplanes, wplanes == 2 ? 1 : -1, 0, col_scale, false, range, s);
  if (e != hipSuccess) return e;
  const int yb = L.y_dtype == F32 ? 4 : 2;
  FastArgs a{};
  a.x = image;
  a.w = weights;
  a.y = L.y;
  a.bias = L.bias;
  a.x_bytes = (uint32_t)((uint64_t)L.m * L.conv_cin * 4);
  a.w_bytes = (uint32_t)((uint64_t)L.n * p.kp * 2 * wplanes);
  a.m = L.m;
  a.n = L.n;
  a.k = p.kp * p.segments;
  // f32 weights are read hi, lo, hi: the third segment wraps to the first plane; bf16: the second does
  a.kwrap = wplanes == 2 ? 0xffffffffu : p.kp;
  a.kwrap2 = wplanes == 2 ? 2 * p.kp : 0xffffffffu;
  a.scale = L.scale;
  a.x_stride = 2 * L.conv_cin;
  a.w_stride = wplanes * p.kp;
  a.y_stride = L.y_stride;
  a.y_offset = L.y_offset;
  a.kc = a.k;
  a.flags = L.flags;
  a.y_dtype = (uint32_t)L.y_dtype;
  a.vec_store = ((uintptr_t)L.y % (4 * yb) == 0 && L.y_offset % 4 == 0 && L.y_stride % 4 == 0) ? 1u : 0u;
  a.row_scale = inv;
  a.col_scale = col_scale;
  a.conv_width = L.conv_width;
  a.conv_cin = L.conv_cin;
  a.conv_kp = p.kp;
  a.conv_hi = a.k - p.kp;
  a.conv_magic = (uint32_t)(((1ull << 32) + L.conv_cin - 1) / L.conv_cin);
  uint32_t splits = 1;
  if (p.rsplits > 1) {
    a.part = (float*)(base + p.part);
    a.rsplits = splits = p.rsplits;
    a.kc = p.rkc;
  }
  a.skip_if = range;
  switch (p.cfg) {
    case GEMM_CFG_256x192: e = launch_fast_cfg<256, 192, 4, 2, true, F16, 2, true, true>(a, splits, L.reduce_xcd, s); break;
    case GEMM_CFG_128x128: e = launch_fast_cfg<128, 128, 2, 2, true, F16, 2, false, true>(a, splits, L.reduce_xcd, s); break;
    default: e = launch_fast_cfg<64, 64, 2, 2, true, F16, 3, false, true>(a, splits, L.reduce_xcd, s); break;
  }
  if (e != hipSuccess) return e;
  GemmLaunch G = L;  // flagged operands: the general kernel (its workgroups return at once for any others)
  G.only_if = range;
  return gemm_launch(G, s);
}

}  // namespace we
