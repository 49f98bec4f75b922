// Products of prompts of some hundreds of rows: which tiles take which, in plain numbers.
#pragma once
#include "prompt_linear.h"

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
// CU.  Least squares over 3702 products of 65 to 2200 rows, n 768 to 11264, k 512 to 14336, all plans of up to 512 workgroups, weights that
// no cache holds (as in a model whose layers take turns): 5 to 12 % (root mean square) off; what it chooses takes 1.4 % longer than the best plan
// with K whole, 1.8 % where it may be cut.
struct ProductTimes {
  float fixed, step, out;
};
inline double product_time(const ProductPlan& p, int rows, int n, int k, int batch = 1) {
  static const ProductTimes kOne[6][2] = {
      {{2.623f, 0.0794f, 0.3561f}, {2.06f, 0.1357f, 0.8835f}},
      {{2.772f, 0.08631f, 0.334f}, {2.592f, 0.1521f, 0.4529f}},
      {{2.892f, 0.09792f, 0.3492f}, {2.551f, 0.1767f, 0.4665f}},
      {{2.874f, 0.1034f, 0.3875f}, {2.606f, 0.2003f, 0.3941f}},
      {{3.187f, 0.1175f, 0.3382f}, {2.689f, 0.2247f, 0.3988f}},
      {{3.315f, 0.1258f, 0.3171f}, {2.524f, 0.2421f, 0.4105f}}};  // nt = 1; 16, 32 .. 96 rows
  static const ProductTimes kTwo[5][2] = {
      {{3.552f, 0.1735f, 0.269f}, {3.288f, 0.3065f, 0.3384f}},
      {{4.268f, 0.1862f, 0.2083f}, {2.794f, 0.331f, 0.3679f}},
      {{4.584f, 0.1957f, 0.1974f}, {2.819f, 0.3559f, 0.3446f}},
      {{4.603f, 0.2101f, 0.2022f}, {2.893f, 0.3802f, 0.309f}},
      {{4.731f, 0.2273f, 0.2055f}, {3.128f, 0.4086f, 0.2885f}}};  // nt = 2; up to 64, 80, 96, 112, 128 rows
  static const ProductTimes kFour[5][2] = {
      {{3.798f, 0.2844f, 0.2426f}, {4.425f, 0.4436f, 0.2531f}},
      {{4.429f, 0.2968f, 0.2107f}, {2.732f, 0.4958f, 0.2947f}},
      {{4.823f, 0.3157f, 0.2116f}, {3.968f, 0.5675f, 0.2346f}},
      {{5.339f, 0.3472f, 0.1954f}, {4.613f, 0.6315f, 0.2096f}},
      {{5.629f, 0.3732f, 0.1902f}, {4.f, 0.6884f, 0.2167f}}};  // nt = 4
  const bool two = product_units(p, rows, n) * batch > 256;
  const int at = p.size <= 64 ? 0 : p.size / 16 - 4;
  const ProductTimes& t = p.nt == 1 ? kOne[p.size / 16 - 1][two] : p.nt == 2 ? kTwo[at][two] : kFour[at][two];
  const double mb = (double)rows * n * batch * 1e-6;
  double us = t.fixed + t.step * product_share(p, k) + t.out * mb * (p.shares > 1 ? 4 * p.shares : 2);
  // The slabs' way into the launch that sums them.  Launches of Dynamic Tanh take more (300 rows of 2048 in two slabs 1.7 us, not .7), and those with
  // the token shift behind it, which sum a row and the one before it, 2.8: 300 rows of 2048 for 2048 and such a launch 18.2, K whole 16.0;
  // 200 rows 15.0, 14.3.  Ahead of the token shift stand the products of feed-forwards, 8448 for 2048: 300 rows 29.9, 34.7; 900 49.4, 59.7.
  if (p.shares > 1) us += .2 * mb * (4 * p.shares - 2);
  return us;
}

// us of GELU behind a product in tiles of 128 rows (prompt_linear.h), where that takes it and every tile has a CU: 5.9 + .255 a k-step of 32 for half
// tiles, 8.5 + .42 for whole ones, of 69 such products of 384 to 2048 wide, 5 % off (root mean square).  0: it does not, or tiles take turns.
inline double tile_gelu_time(int rows, int n, int k) {
  const PromptLinearPlan t = prompt_linear_plan(rows, n, k, LVLLM_ACT_GELU, false, true);
  if (t.body != LVLLM_PROMPT_TILE || (int64_t)((rows + 127) / 128) * ((n + 64 * t.nt - 1) / (64 * t.nt)) > 256) return 0;
  return t.nt == 2 ? 5.9 + .255 * (k / 32) : 8.5 + .42 * (k / 32);
}

// The shortest of the plans, and the library where its products are the better ones, by the rate that the plan reaches, TFLOP/s (of those 3702, own
// time of the library's; host time, 3 us for 20, not counted):
//   * up to 900; above k = 5120 1000, and above k = 9000, where the library has too few tiles for too long, 1150.  From there on the library's,
//     both of whose operands go through LDS, take less power: 0.95 to 1.2 of its time;
//   * one share, whose sums are in the library's order but where that cuts K: 0.64 of its time in the mean up to k = 1024, 0.79 up to 2048, 0.86 up to
//     5120, 0.90 above (us, before and after: 300 rows of 2048 for 2048 12.9, 8.8; for 7680 25.4, 19.0; 300 rows of 5632 for 2048 25.7, 20.8).  With
//     few tiles of long K the library cuts it and is faster: 0.99 to 1.6 below 100 for k > 2048, below 200 for k > 5120;
//   * K may be cut into slabs: 0.64, 0.75, 0.77 and 0.70, what the slabs cost the next launch included (300 rows of 14336 for 4096 75, 50; 100 rows 48,
//     29; 300 rows of 4096 for 1024 14.6, 8.7);
//   * GELU behind a product makes it 1.15 times as long (1.11 to 1.16 in the mean by tiles and rounds, of 1100).  The tiles of prompt_linear.h keep
//     what takes them less: 4096 of 1024, 65 to 600 rows 0.41 to 0.85 of theirs or the library's; 800 rows 16.1 us for 14.1, 1000 rows 15.7 for
//     14.9, 2000 rows 23.8 for 23.3.  Of 29 other sizes it leaves two slower, 1.04; by plain products' times 18 were, up to 1.19.
// `batch` products of one size in a launch (K whole): as one of so many times the tiles.
inline ProductPlan prompt_product_plan(int rows, int n, int k, bool gelu, int sums, int batch = 1) {
  ProductPlan best{0, 0, 0};
  if (rows <= 64 || rows > 8192 || n < 16 || n % 16 != 0 || k < 256 || k % 64 != 0 || (int64_t)n * k >= (int64_t)1 << 30 || batch < 1 || batch > 64) return best;
  const bool slabs = sums == LVLLM_SUMS_SLABS && !gelu && batch == 1;
  double least = 0;
  auto take = [&](const ProductPlan& p) {
    if (!product_plan_valid(p, k) || product_units(p, rows, n) * batch > 512 || (p.shares > 1 && k / 32 / p.shares < 8)) return;
    const double us = product_time(p, rows, n, k, batch);
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
  const double rate = 2e-6 * rows * n * k * batch / least;
  if (gelu) {
    const double tile = tile_gelu_time(rows, n, k);
    if (tile > 0 && 1.15 * least > tile) return ProductPlan{0, 0, 0};
  }
  const double fewest = slabs || k <= 2048 ? 0 : k <= 5120 ? 100 : 200, most = k <= 5120 ? 900 : k <= 9000 ? 1000 : 1150;
  return rate >= fewest && rate <= most ? best : ProductPlan{0, 0, 0};
}

}  // namespace lvllm
