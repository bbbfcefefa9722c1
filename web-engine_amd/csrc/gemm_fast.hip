// Host side of the fast GEMM path (gemm_lds.h): which launches qualify, the tile shape and split-K plan of each, and
// the launches for 16-bit and fp8 weights.
#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "gemm_lds.h"

namespace we {

namespace {

// Do the operands qualify for the fast path? (16-bit activations, fp8 or matching 16-bit weights, 16-byte
// aligned rows, K a multiple of 16, operand extents under the 32-bit buffer offsets.)
bool fast_supported(const GemmLaunch& L, uint32_t kc) {
  if (L.conv_width) return false;  // the 3x3 convolution input gathers x in the general kernel
  const bool f16 = L.x_dtype == F16;
  if (!(L.x_dtype == BF16 || L.x_dtype == F16)) return false;
  if (!(L.w_dtype == FP8 || (f16 ? L.w_dtype == F16 : L.w_dtype == BF16))) return false;
  const int wb = L.w_dtype == FP8 ? 1 : 2;
  if (L.k % 16 || kc % 16) return false;
  if (((uintptr_t)L.x + (uint64_t)L.x_offset * 2) % 16 || ((uintptr_t)L.w + (uint64_t)L.w_offset * wb) % 16 ||
      (L.x_stride * 2) % 16 || (L.w_stride * wb) % 16)
    return false;
  if (L.k_wrap && (L.k_wrap % BK || L.k % L.k_wrap || L.k / L.k_wrap > 3)) return false;
  const uint64_t xb = L.k ? ((uint64_t)(L.m - 1) * L.x_stride + L.k) * 2 : 0;
  const uint64_t wbytes = L.k ? ((uint64_t)(L.n - 1) * L.w_stride + (L.k_wrap ? L.k_wrap : L.k)) * wb : 0;
  return xb < kInvalid && wbytes < kInvalid;
}

constexpr uint32_t kCUs = 256;

// readable weight bytes of a GEMM (FastArgs::w_bytes)
uint64_t weight_extent(const GemmLaunch& L) {
  const int wb = L.w_dtype == FP8 ? 1 : 2;
  return L.k ? ((uint64_t)(L.n - 1) * L.w_stride + (L.k_wrap ? L.k_wrap : L.k)) * wb : 0;
}

// Tile shape by predicted speed: score = base x (tiles / slots) / (time in rounds). base is the tile shape's own
// speed relative to 256 x 256 (one per CU, the fastest per FLOP) at full occupancy; a full round of tiles costs 1,
// the last, partly filled round 0.6 + 0.3 f (f = the fraction of slots it fills). The chip runs at its power
// limit, so tiles run faster when fewer CUs are busy, and a partial round costs far more than its share but less
// than a full one. Fitted to the tile sweep (bench.py --sweep: bf16 activations and output, fp8 weights unless
// named, M = 4096 and 8740). With fp8 weights 256 x 192 runs at 0.90 of 256 x 256's speed, 128 x 128 (two per CU)
// at 0.81, 256 x 128 at 0.77. The tail term decides two shapes: 4096 x 3072 x 12288 (256 x 256: one round at
// f = 0.75) stays with 256 x 256 (1288 against 1254 TFLOP/s for 256 x 192), while 4096 x 9216 x 3072 (256 x 256:
// two full rounds and one at f = 0.25) goes to 256 x 192 (three full rounds; 7% faster). With 16-bit weights
// 128 x 128 tiles fit one per CU only and lose to the ping-pong tiles (4096 x 9216 x 3072 bf16: 801 against 1085
// TFLOP/s), so only the two 256-row shapes compete there, 256 x 192 at 0.95.
int pick_fast_cfg(uint32_t m, uint32_t n, uint32_t splits, bool w8) {
  if (m <= 32) return GEMM_CFG_32x64;
  if (m <= 64) return GEMM_CFG_64x64;
  struct Cand {
    int cfg;
    uint32_t bm, bn, per_cu;
    double base;
  };
  const Cand cands[] = {{GEMM_CFG_256x256, 256, 256, 1, 1.00}, {GEMM_CFG_256x192, 256, 192, 1, w8 ? 0.90 : 0.95},
                        {GEMM_CFG_128x128, 128, 128, 2, 0.81}, {GEMM_CFG_256x128, 256, 128, 1, 0.77}};
  int best = GEMM_CFG_128x128;
  double best_score = -1.0;
  for (const Cand& c : cands) {
    if (c.bm == 256 && m < 256) continue;
    if (!w8 && c.cfg != GEMM_CFG_256x256 && c.cfg != GEMM_CFG_256x192) continue;
    const uint64_t tiles = (uint64_t)((m + c.bm - 1) / c.bm) * ((n + c.bn - 1) / c.bn) * splits;
    const uint64_t slots = (uint64_t)kCUs * c.per_cu;
    const uint64_t full = tiles / slots, rest = tiles % slots;
    const double rounds = (double)full + (rest ? 0.6 + 0.3 * (double)rest / (double)slots : 0.0);
    const double score = c.base * ((double)tiles / (double)slots) / rounds;
    if (score > best_score + 1e-9) {
      best_score = score;
      best = c.cfg;
    }
  }
  return best;
}

uint32_t cfg_bm(int cfg) {
  return cfg == GEMM_CFG_32x64 ? 32 : cfg == GEMM_CFG_64x64 ? 64 : cfg == GEMM_CFG_128x128 ? 128 : 256;
}
uint32_t cfg_bn(int cfg) {
  return cfg == GEMM_CFG_256x256   ? 256
         : cfg == GEMM_CFG_256x192 ? 192
         : cfg == GEMM_CFG_256x128 || cfg == GEMM_CFG_128x128 ? 128
                                                               : 64;
}

// the tile shape of a launch: forced, planned, or by shape
int launch_cfg_of(const GemmLaunch& L) {
  const uint32_t splits = L.rsplits > 1 ? L.rsplits : L.splits < 1 ? 1 : L.splits;
  return L.cfg >= 0 ? L.cfg : L.rcfg >= 0 ? L.rcfg : pick_fast_cfg(L.m, L.n, splits, L.w_dtype == FP8);
}

}  // namespace

GemmReducePlan gemm_reduce_plan(const GemmLaunch& L, uint32_t force_splits) {
  GemmReducePlan p{1, L.k, 0, -1, 1};
  if (L.generic || (L.splits > 1) || (L.flags & WE_EPI_SPLIT_K_BIT) || L.m == 0 || L.n == 0) return p;
  if (L.k < 512 || !fast_supported(L, L.k)) return p;
  const int cfg = L.cfg >= 0 ? L.cfg : pick_fast_cfg(L.m, L.n, 1, L.w_dtype == FP8);
  const uint64_t tiles = (uint64_t)((L.m + cfg_bm(cfg) - 1) / cfg_bm(cfg)) * ((L.n + cfg_bn(cfg) - 1) / cfg_bn(cfg));
  uint32_t rs;
  if (L.m <= 64) {
    if (tiles >= kCUs / 2) return p;
    // about one workgroup per CU; where the reduce pass reads the partial sums from L2 (reduce_in_l2), up to two
    // (at most 8 slices where one per CU needs fewer). Measured, 8 slices against one workgroup per CU, weights
    // cached / streamed from HBM: 64 x 3072 x 3072 9.24 / 10.22 -> 8.99 / 9.98 us, 16 x 3072 x 3072 8.07 / 9.05 ->
    // 7.61 / 8.67 us, 64 x 4096 x 4096 10.92 / 12.47 -> 10.23 / 11.78 us (12 slices of 64 x 3072 x 3072: 10.5 us);
    // without the L2 reduce more slices only add partial-sum traffic (64 x 6144 x 3072: 14.1 -> 15.9 us)
    const uint64_t one = (kCUs + tiles - 1) / tiles, two = (2 * kCUs + tiles - 1) / tiles;
    rs = reduce_in_l2(tiles, weight_extent(L), L.reduce_xcd) ? (uint32_t)std::max<uint64_t>(one, std::min<uint64_t>(8, two))
                                               : (uint32_t)one;
  } else {
    // larger M: split when the tiles fill less than half of the workgroup slots (M = 512, N = 3072:
    // 96 tiles of 128 x 128 for 512 slots), to about one workgroup per slot
    const uint64_t slots = (uint64_t)kCUs * (cfg == GEMM_CFG_128x128 ? 2 : 1);
    if (tiles * 2 > slots) return p;
    rs = (uint32_t)((slots + tiles - 1) / tiles);
    // with fp8 weights, M >= 256 and slices of at least 1024 k the slices run in 256 x 192 ping-pong tiles, about
    // one per CU: 512 x 3072 x 12288 58.2 -> 54.9 us against the 128 x 128 plan (6 slices, which the launch ran as
    // 192 workgroups of 256 x 192), same process, alternating order. At 512 x 3072 x 3072 (slices of 384 k) the
    // 128 x 128 plan stays: 30.3 against 31.4 us.
    if (L.cfg < 0 && L.m >= 256 && L.w_dtype == FP8) {
      const uint64_t t = (uint64_t)((L.m + 255) / 256) * ((L.n + 191) / 192);
      const uint32_t rs2 = (uint32_t)((kCUs + t - 1) / t);
      if (L.k / rs2 >= 1024) {
        p.rcfg = GEMM_CFG_256x192;
        rs = rs2;
      }
    }
  }
  rs = rs < L.k / 256 ? rs : L.k / 256;  // every slice keeps at least 256 of K
  if (force_splits) rs = force_splits < L.k / BK ? force_splits : L.k / BK;
  if (rs < 2) return p;
  const uint32_t kc = (L.k + rs * BK - 1) / (rs * BK) * BK;
  const uint32_t n_slices = (L.k + kc - 1) / kc;
  if (n_slices < 2) return p;
  p.rsplits = n_slices;
  p.rkc = kc;
  p.scratch_bytes = (size_t)n_slices * L.m * L.n * 4;
  return p;
}

namespace {

bool qk_fusable_cfg(int cfg) { return cfg == GEMM_CFG_256x128 || cfg == GEMM_CFG_128x128; }

// Predicted time of a launch, in us: `launch`, then rounds of tiles (a full round 1; the last, partly filled one part +
// part_f * its fraction: the chip runs at its power limit, so tiles run faster when fewer CUs are busy), each tile `block`
// per 64 k and `tile` once, and the split-K partial sums' bytes. Fitted to a sweep of tile shapes and slice counts over 37
// shapes of M 65 .. 4096, N 1040 .. 18944, K 2048 .. 32768 (rms error 6%): against pick_fast_cfg and gemm_reduce_plan the
// choice gains 12% (fp8 weights), 26% (f16 planes of f32) and 10% (16-bit weights) in the mean over those shapes.
// 700 x 3072 x 12288 fp8 96.6 -> 67.2 us (256 x 256, 6 slices), 1500 x 3072 x 12288 151 -> 107, 300 x 18000 x 2048
// 55 -> 40 (128 x 128), 128 x 3072 x 12288 36 -> 26 (64 x 64, 8 slices).
struct CostModel {
  double launch, part[2], part_f[2], reduce, reduce_mb;  // part: one, several workgroups per CU
  double block[6], tile[6];                              // by GemmCfgId
};
constexpr CostModel kCostFp8 = {7.2, {0.80, 0.46}, {0.147, 0.494}, 0.3, 0.293,
                                {1.315, 0.912, 1.026, 0.630, 0, 1.241}, {4.5, 2.7, 1.4, 0.0, 0, 2.0}};
constexpr CostModel kCostPlanes = {4.7, {0.767, 0.406}, {0.203, 0.658}, 0.0, 0.347,
                                   {1.436, 0.971, 1.008, 0.666, 0, 1.255}, {1.2, 0.1, 0.9, 0.0, 0, 1.0}};
constexpr CostModel kCost16 = {8.5, {0.874, 0.648}, {0.142, 0.234}, 0.4, 0.254,
                               {1.498, 0.898, 0.700, 0.456, 0, 1.186}, {4.0, 2.4, 1.2, 5.0, 0, 3.0}};

}  // namespace

GemmReducePlan gemm_plan(const GemmLaunch& L) {
  if (L.cfg >= 0 || L.m <= 64 || L.n == 0 || L.generic || L.splits > 1 || (L.flags & WE_EPI_SPLIT_K_BIT) || L.k < 512 ||
      !fast_supported(L, L.k))
    return gemm_reduce_plan(L);
  const bool w8 = L.w_dtype == FP8, three = L.k_wrap && L.k == 3 * L.k_wrap;
  const CostModel& c = !w8 ? kCost16 : L.k_wrap ? kCostPlanes : kCostFp8;
  // workgroups per CU by their LDS: 64 x 64 36 or 48 KB, 128 x 128 72 or 96 KB
  const uint32_t per_cu[6] = {1, 1, w8 ? 2u : 1u, w8 ? 4u : 3u, 1, 1};
  auto predict = [&](int cfg, uint32_t slices, uint32_t kc) {
    const uint64_t tiles = (uint64_t)((L.m + cfg_bm(cfg) - 1) / cfg_bm(cfg)) * ((L.n + cfg_bn(cfg) - 1) / cfg_bn(cfg));
    const uint64_t slots = (uint64_t)kCUs * per_cu[cfg];
    const int several = per_cu[cfg] > 1 || cfg == GEMM_CFG_128x128;
    const uint64_t full = tiles * slices / slots, rest = tiles * slices % slots;
    const double rounds = (double)full + (rest ? c.part[several] + c.part_f[several] * (double)rest / (double)slots : 0.0);
    double us = c.launch + rounds * ((double)((kc + BK - 1) / BK) * c.block[cfg] + c.tile[cfg]);
    if (slices > 1) us += c.reduce + c.reduce_mb * 4e-6 * L.m * (double)L.n * slices;
    // q / k norm and RoPE: a pass over those columns, or in the epilogue for about the same time less a launch (2500 x 6144
    // x 4096 bf16: 129.6 us with 256 x 256 tiles and the pass, 150.9 us fused in 256 x 128 tiles)
    if (L.qk_cols) us += (slices > 1 || !qk_fusable_cfg(cfg) ? 4.0 : 0.0) + 4.0 * L.m * (double)L.qk_cols / 3e6;
    return us;
  };
  // The older rules' choice stays unless another is predicted 6% faster, the model's error: 1500 x 4608 x 3072 took 55.2 us in
  // the 256 x 128 tiles that it put 2% ahead of the 128 x 128 ones (54.2 us), 700 x 12288 x 4096 with the q / k pass 93.3 us in
  // 256 x 192 tiles, 5% ahead of the 256 x 256 ones (91.5 us).
  GemmReducePlan best = gemm_reduce_plan(L);
  const uint32_t older = best.rsplits;
  // Where the older choice runs the q / k epilogue, so does every other: the epilogue normalizes the f32 sums, the pass of its
  // own the values rounded to y's type (400 x 9216 x 3072 bf16 in 64 x 64 tiles and the pass: 1.4 times the rounding error)
  GemmLaunch O = L;
  O.rsplits = best.rsplits;
  O.rcfg = best.rcfg;
  const bool fused = L.qk_cols && gemm_qk_fusable(O);
  best.rcfg = best.rcfg >= 0 ? best.rcfg : pick_fast_cfg(L.m, L.n, best.rsplits, w8);
  double best_us = 0.94 * predict(best.rcfg, best.rsplits, best.rsplits > 1 ? best.rkc : L.k);
  for (const int cfg : {GEMM_CFG_256x256, GEMM_CFG_256x192, GEMM_CFG_256x128, GEMM_CFG_128x128, GEMM_CFG_64x64}) {
    if ((cfg_bm(cfg) == 256 && L.m < 256) || (fused && !qk_fusable_cfg(cfg))) continue;
    const uint64_t tiles = (uint64_t)((L.m + cfg_bm(cfg) - 1) / cfg_bm(cfg)) * ((L.n + cfg_bn(cfg) - 1) / cfg_bn(cfg));
    // slices only where the tiles fill at most half of the CUs (128 x 128: twice that), as swept
    const uint32_t most = tiles * 2 <= kCUs * (cfg == GEMM_CFG_128x128 ? 2u : 1u) ? std::min(8u, L.k / 256) : 1u;
    // three planes of x: a multiple of the older plan's slices, whose shorter sums round less and may end with the planes
    // (800 x 4096 x 8192: error 3.3e-7 in 3 slices, 3.8e-7 in 4)
    for (uint32_t rs = 1; rs <= most; rs++) {
      if ((three && rs % older) || (fused && rs > 1)) continue;
      const uint32_t kc = (L.k + rs * BK - 1) / (rs * BK) * BK;
      if ((L.k + kc - 1) / kc != rs) continue;
      const double us = predict(cfg, rs, kc);
      if (us < best_us) {
        best_us = us;
        best = GemmReducePlan{rs, rs > 1 ? kc : L.k, rs > 1 ? (size_t)rs * L.m * L.n * 4 : 0, cfg, 1};
      }
    }
    // One workgroup per CU and a last round of at most half of them: its tiles in as many K slices as fill the round
    // (1103 x 16384 x 6144 f32: 320 tiles of 256 x 256 in 1.25 rounds instead of 2, less 25 us for the partial sums; the
    // gated MLP of 1103 rows 1346 -> 1176 us)
    const uint32_t rest = (uint32_t)(tiles % kCUs);
    if ((cfg == GEMM_CFG_256x256 || cfg == GEMM_CFG_256x192) && tiles > kCUs && rest && rest * 2 <= kCUs && !L.qk_cols &&
        !(three && older > 1)) {
      const uint32_t ts = std::min({kCUs / rest, 8u, L.k / 512});
      const uint32_t kc = ts > 1 ? (L.k + ts * BK - 1) / (ts * BK) * BK : 0;
      if (ts > 1 && (L.k + kc - 1) / kc == ts) {
        const double sums = (double)ts * rest * cfg_bm(cfg) * cfg_bn(cfg) * 4.0;
        const double us = c.launch + (double)(tiles / kCUs) * ((L.k + BK - 1) / BK * c.block[cfg] + c.tile[cfg]) +
                          ((double)(kc / BK) * c.block[cfg] + c.tile[cfg]) + 4.0 + c.reduce_mb * 1e-6 * sums;
        if (us < best_us) {
          best_us = us;
          best = GemmReducePlan{1, kc, (size_t)sums, cfg, ts};
        }
      }
    }
  }
  return best;
}

bool gemm_qk_fusable(const GemmLaunch& L) {
  if (L.generic || L.splits > 1 || L.rsplits > 1 || L.flags & ~WE_EPI_BIAS_BIT || L.mul || L.gate || L.res) return false;
  if (L.y_dtype == F32 || !fast_supported(L, L.k)) return false;
  const int cfg = launch_cfg_of(L);
  // head-aligned tiles with 64-column waves outside the ping-pong kernels: 256 x 128 (4 x 2), 128 x 128 (2 x 2)
  if (!qk_fusable_cfg(cfg)) return false;
  const uint32_t bn = cfg_bn(cfg);
  return L.qk_cols % bn == 0 && L.q_cols % bn == 0 && L.qk_cols <= L.n && (L.y_stride % 4) == 0 &&
         (L.y_offset % 4) == 0 && ((uintptr_t)L.y % 16) == 0 && ((uintptr_t)L.qk_norm_q % 16) == 0 &&
         ((uintptr_t)L.qk_norm_k % 16) == 0 && ((uintptr_t)L.qk_cos % 8) == 0 && ((uintptr_t)L.qk_sin % 8) == 0 &&
         (!L.bias || ((uintptr_t)L.bias % 4) == 0);
}

namespace {

// The kernel arguments of one GEMM (no split-K slices, no tile pick yet).
FastArgs fast_args(const GemmLaunch& L, uint32_t kc) {
  const int wb = L.w_dtype == FP8 ? 1 : 2;
  const int yb = L.y_dtype == F32 ? 4 : 2;
  FastArgs a{};
  a.x = (const char*)L.x + (uint64_t)L.x_offset * 2;
  a.w = (const char*)L.w + (uint64_t)L.w_offset * wb;
  a.y = L.y;
  a.bias = L.bias;
  a.gate = L.gate;
  a.res = L.res;
  a.mul = (uint32_t)L.mul;
  a.qk_cols = L.qk_cols;
  a.q_cols = L.q_cols;
  a.qk_rope_from = L.qk_rope_from;
  a.qk_eps = L.qk_eps;
  a.qk_offset = L.qk_offset;
  a.qk_norm_q = L.qk_norm_q;
  a.qk_norm_k = L.qk_norm_k;
  a.qk_cos = L.qk_cos;
  a.qk_sin = L.qk_sin;
  a.x_bytes = L.k ? (uint32_t)(((uint64_t)(L.m - 1) * L.x_stride + L.k) * 2) : 0;
  a.w_bytes = (uint32_t)weight_extent(L);
  a.m = L.m;
  a.n = L.n;
  a.k = L.k;
  a.kwrap = L.k_wrap ? L.k_wrap : 0xffffffffu;
  a.kwrap2 = L.k_wrap ? 2 * L.k_wrap : 0xffffffffu;
  a.row_scale = L.row_scale;
  a.cvt_lo = L.row_scale ? 0x1p-5f : 1.0f;
  a.cvt_hi = L.row_scale ? 0x1p7f : 1.0f;
  a.only_if = L.only_if;
  a.range = L.range;
  a.range_n = L.range_n;
  a.range_most = L.range_most;
  a.f32 = L.f32;
  a.f32_stride = L.f32_stride;
  a.skip_if = a.skip_out = L.skip_out;
  a.scale = L.scale;
  a.x_stride = L.x_stride;
  a.w_stride = L.w_stride;
  a.y_stride = L.y_stride;
  a.y_offset = L.y_offset;
  a.kc = kc;
  a.flags = L.flags;
  a.y_dtype = (uint32_t)L.y_dtype;
  a.vec_store = ((uintptr_t)L.y % (4 * yb) == 0 && (uintptr_t)L.res % (4 * yb) == 0 &&
                 (uintptr_t)L.gate % 16 == 0 && ((uint64_t)L.y_offset * yb) % (4 * yb) == 0 &&
                 ((uint64_t)L.y_stride * yb) % (4 * yb) == 0)
                    ? 1u
                    : 0u;
  a.store16 = ((uintptr_t)L.y % 16 == 0 && ((uint64_t)L.y_offset * yb) % 16 == 0 && ((uint64_t)L.y_stride * yb) % 16 == 0)
                  ? 1u
                  : 0u;
  return a;
}

}  // namespace

// Returns hipErrorNotSupported when the shape / dtypes / alignment are not for this path.
hipError_t gemm_fast_launch(const GemmLaunch& L, hipStream_t stream) {
  const bool reduce = L.rsplits > 1;
  const uint32_t splits = reduce ? L.rsplits : (L.splits < 1 ? 1 : L.splits);
  const uint32_t kc = reduce ? L.rkc : (splits > 1 ? L.kc : L.k);
  if (!fast_supported(L, kc)) return hipErrorNotSupported;
  const bool f16 = L.x_dtype == F16;
  FastArgs a = fast_args(L, kc);
  if (reduce) {
    if (!L.scratch) return hipErrorInvalidValue;
    a.part = (float*)L.scratch;
    a.rsplits = splits;
  }
  if (L.tail_splits > 1) {
    if (!L.scratch || reduce || splits > 1 || L.tail_splits > 8) return hipErrorInvalidValue;
    a.part = (float*)L.scratch;
    a.tail_splits = L.tail_splits;
    a.tail_kc = L.rkc;
  }
  const int cfg = launch_cfg_of(L);
  const int rx = L.reduce_xcd;
  if (f16) {
    if (L.w_dtype == FP8) return gemm_lds_f16_fp8(a, splits, cfg, rx, stream);
    return gemm_lds_f16_f16(a, splits, cfg, rx, stream);
  }
  if (L.w_dtype == FP8) return gemm_lds_bf16_fp8(a, splits, cfg, rx, stream);
  return gemm_lds_bf16_bf16(a, splits, cfg, rx, stream);
}

bool gemm_fast_supported(const GemmLaunch& L) {
  return L.splits <= 1 && !(L.flags & WE_EPI_SPLIT_K_BIT) && fast_supported(L, L.k);
}

bool gemm_pair_ok(const GemmLaunch& A, const GemmLaunch& B) {
  for (const GemmLaunch* L : {&A, &B})
    if (L->generic || L->conv_width || L->splits > 1 || L->qk_cols || L->k_wrap || (L->flags & WE_EPI_SPLIT_K_BIT) ||
        !fast_supported(*L, L->k))
      return false;
  return A.n == B.n && A.k == B.k && A.x_dtype == B.x_dtype && A.w_dtype == B.w_dtype && A.y_dtype == B.y_dtype &&
         A.flags == B.flags && A.mul == B.mul && A.cfg == B.cfg;
}

// Two GEMMs (gemm_pair_ok) as one launch: the tiles of both share the round(s) of workgroups, so a small GEMM
// beside a large one costs no launch and no partly empty round of its own. Full K per tile (no split-K), the
// tile shape picked for the two row counts together; each GEMM's tiles compute exactly as in a launch of its own
// with the same tile shape.
hipError_t gemm_fast_launch_pair(const GemmLaunch& A, const GemmLaunch& B, hipStream_t stream) {
  if (!gemm_pair_ok(A, B)) return hipErrorNotSupported;
  FastArgs a = fast_args(A, A.k);
  const FastArgs b = fast_args(B, B.k);
  a.g = FastArgs::Second{b.x,        b.w,        b.y,        b.bias,     b.gate,      b.res,
                         b.x_bytes,  b.w_bytes,  b.m,        b.x_stride, b.w_stride,  b.y_stride,
                         b.y_offset, 0u,         b.vec_store, b.store16, b.scale};
  a.grp = 1;
  const int cfg = A.cfg >= 0 ? A.cfg : pick_fast_cfg(A.m + B.m, A.n, 1, A.w_dtype == FP8);
  if (A.x_dtype == F16) {
    if (A.w_dtype == FP8) return gemm_lds_f16_fp8(a, 1, cfg, 0, stream);
    return gemm_lds_f16_f16(a, 1, cfg, 0, stream);
  }
  if (A.w_dtype == FP8) return gemm_lds_bf16_fp8(a, 1, cfg, 0, stream);
  return gemm_lds_bf16_bf16(a, 1, cfg, 0, stream);
}

}  // namespace we
