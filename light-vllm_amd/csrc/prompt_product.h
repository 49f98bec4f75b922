// Products of prompts of some hundreds of rows: which tiles take which, in plain numbers.
#pragma once
#include <stdint.h>

namespace lvllm {

// prompt_product.hip: tiles of up to 96 rows x 64 W rows, 128 x 128 or 128 x 256, K whole or cut into shares.
struct ProductPlan {
  int size;    // rows of a tile; 0: none, the library's product
  int nt;      // W tiles of 16 of a wave
  int shares;  // of K
};

// k-steps of 32 of a share, an even number; all shares but the last
inline int product_share(const ProductPlan& p, int k) { return (k / 64 + p.shares - 1) / p.shares * 2; }
constexpr int kProductShares = 8;  // most
inline bool product_plan_valid(const ProductPlan& p, int k) {
  if (p.shares < 1 || p.shares > kProductShares || k % 64 != 0 || (int64_t)product_share(p, k) * (p.shares - 1) >= k / 32) return false;
  return (p.nt == 1 || p.nt == 2 || p.nt == 4) && p.size % 16 == 0 && p.size >= 16 && p.size <= (p.nt == 1 ? 96 : 128);
}
inline int64_t product_units(const ProductPlan& p, int rows, int n) {
  return (int64_t)((rows + p.size - 1) / p.size) * ((n + 64 * p.nt - 1) / (64 * p.nt)) * p.shares;
}

// us of a launch: a workgroup's way in and out, its k-steps, and the megabytes that leave; of workgroups that have a CU each, and of up to two a
// CU.  Least squares over 4086 products of 65 to 2200 rows, n 768 to 11264, k 512 to 14336, all plans of up to 512 workgroups: 4 to 10 %
// (root mean square) off; what it chooses takes 0.4 % longer than the best plan with K whole, 1.0 % where it may be cut.
struct ProductTimes {
  float fixed, step, out;
};
inline double product_time(const ProductPlan& p, int rows, int n, int k) {
  static const ProductTimes kOne[6][2] = {
      {{2.723f, 0.05187f, 0.3175f}, {3.247f, 0.1022f, 0.1113f}},
      {{2.477f, 0.06026f, 0.445f}, {3.039f, 0.1207f, 0.2109f}},
      {{2.723f, 0.07458f, 0.3617f}, {3.276f, 0.1522f, 0.2328f}},
      {{2.586f, 0.08304f, 0.4016f}, {3.141f, 0.1714f, 0.2446f}},
      {{2.732f, 0.09542f, 0.3601f}, {3.265f, 0.1932f, 0.2565f}},
      {{2.691f, 0.1032f, 0.3742f}, {3.199f, 0.2142f, 0.2505f}}};  // nt = 1; 16, 32 .. 96 rows
  static const ProductTimes kTwo[5][2] = {
      {{3.063f, 0.123f, 0.3697f}, {4.133f, 0.2644f, 0.2241f}},
      {{3.205f, 0.1376f, 0.3229f}, {3.97f, 0.2876f, 0.2283f}},
      {{3.213f, 0.1513f, 0.3139f}, {4.039f, 0.3143f, 0.2192f}},
      {{3.326f, 0.1653f, 0.3002f}, {3.992f, 0.3487f, 0.2052f}},
      {{3.582f, 0.1753f, 0.2888f}, {4.465f, 0.3727f, 0.1884f}}};  // nt = 2; up to 64, 80, 96, 112, 128 rows
  static const ProductTimes kFour[5][2] = {
      {{3.328f, 0.2258f, 0.2683f}, {5.358f, 0.418f, 0.1452f}},
      {{4.188f, 0.2516f, 0.2239f}, {5.208f, 0.4717f, 0.1583f}},
      {{4.902f, 0.2954f, 0.1948f}, {5.888f, 0.5416f, 0.1476f}},
      {{5.479f, 0.3346f, 0.1796f}, {6.677f, 0.6068f, 0.136f}},
      {{5.987f, 0.3597f, 0.1672f}, {6.839f, 0.656f, 0.1376f}}};  // nt = 4
  const bool two = product_units(p, rows, n) > 256;
  const int at = p.size <= 64 ? 0 : p.size / 16 - 4;
  const ProductTimes& t = p.nt == 1 ? kOne[p.size / 16 - 1][two] : p.nt == 2 ? kTwo[at][two] : kFour[at][two];
  const double mb = (double)rows * n * 1e-6;
  double us = t.fixed + t.step * product_share(p, k) + t.out * mb * (p.shares > 1 ? 4 * p.shares : 2);
  if (p.shares > 1) us += .2 * mb * (4 * p.shares - 2);  // the slabs' way into the launch that sums them
  return us;
}

enum { kSumsAny = 0, kSumsSlabs = 1, kSumsOrdered = 2 };  // include/lvllm_hip.h LVLLM_SUMS_*

// The shortest of the plans, and the library where its products are the better ones, by the rate that the plan reaches, TFLOP/s (of those 4086, own
// time of the library's; host time, 3 us for 20, not counted):
//   * up to 900; above k = 5120 1050, and above k = 9000, where the library has too few tiles for too long, 1400.  From there on the library's,
//     both of whose operands go through LDS, take less power: 0.94 to 1.2 of its time;
//   * one share, whose sums are in the library's order but where that cuts K: 0.76 of its time in the mean up to k = 2048, 0.81 up to 5120, 0.88 above
//     (us, before and after: 300 rows of 2048 for 2048 11.2, 7.8; for 7680 19.8, 13.8; 300 rows of 5632 for 2048 20.7, 17.1; 1000 rows of 1024 for
//     3072 14.4, 10.3).  With few tiles of long K the library cuts it and is faster: 0.96 to 1.4 below 100 for k > 2048, 200 for k > 5120, 300
//     for k > 9000;
//   * K may be cut into slabs: 0.74, 0.75 and 0.70, what the slabs cost the next launch included (300 rows of 14336 for 4096 75, 51; 100 rows 48,
//     29; 300 rows of 4096 for 1024 13.8, 7.7).
inline ProductPlan prompt_product_plan(int rows, int n, int k, bool gelu, int sums) {
  ProductPlan best{0, 0, 0};
  if (rows <= 64 || rows > 8192 || n < 16 || n % 16 != 0 || k < 256 || k % 64 != 0 || (int64_t)n * k >= (int64_t)1 << 30) return best;
  const bool slabs = sums == kSumsSlabs && !gelu;
  double least = 0;
  auto take = [&](const ProductPlan& p) {
    if (!product_plan_valid(p, k) || product_units(p, rows, n) > 512 || (p.shares > 1 && k / 32 / p.shares < 8)) return;
    const double us = product_time(p, rows, n, k);
    if (best.size == 0 || us < least) best = p, least = us;
  };
  for (int shares = 1; shares <= (slabs ? kProductShares : 1); ++shares) {
    for (int size = 16; size <= 96; size += 16) take({size, 1, shares});
    int before = 0;
    for (int most = 128; most >= 64; most -= 16) {
      const int tiles = (rows + most - 1) / most;
      if (tiles == before) continue;
      before = tiles;
      const int size = ((rows + tiles - 1) / tiles + 15) / 16 * 16;
      take({size, 2, shares});
      if (!gelu) take({size, 4, shares});  // (tile_linear.hip has those)
    }
  }
  if (best.size == 0) return best;
  const double rate = 2e-6 * rows * n * k / least;
  const double fewest = slabs || k <= 2048 ? 0 : k <= 5120 ? 100 : k <= 9000 ? 200 : 300, most = k <= 5120 ? 900 : k <= 9000 ? 1050 : 1400;
  return rate >= fewest && rate <= most ? best : ProductPlan{0, 0, 0};
}

}  // namespace lvllm
