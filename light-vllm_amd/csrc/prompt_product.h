// Products of prompts of some hundreds of rows: which kernel takes which, in plain numbers.
#pragma once
#include <stdint.h>

namespace lvllm {

enum { kProductNone = 0, kProductShort = 1, kProductTile = 2 };

// prompt_product.hip: none (the library's), short (16 to 64 rows x 64 or 128 W rows a workgroup, K dealt to its waves) or tiles (up to 128 rows x
// 128 or 256 W rows, moe_tile.h).
struct ProductPlan {
  int body;    // kProduct*
  int size;    // rows of a tile
  int nt;      // short: W tiles of 16 of a workgroup; tile: of a wave
  int shares;  // of K
};

// k-steps of 32 that a wave of a short product asks for at once
inline int product_batch(const ProductPlan& p) { return p.body == kProductShort && p.size == 16 ? 4 : 2; }
// k-steps of a share; all shares but the last
inline int product_share(const ProductPlan& p, int k) {
  const int b = product_batch(p);
  return (k / 32 / b + p.shares - 1) / p.shares * b;
}
constexpr int kProductShares = 8;  // most
inline bool product_plan_valid(const ProductPlan& p, int k) {
  if (p.shares < 1 || p.shares > kProductShares || k % (32 * product_batch(p)) != 0 || (int64_t)product_share(p, k) * (p.shares - 1) >= k / 32) return false;
  if (p.body == kProductTile) return (p.nt == 2 || p.nt == 4) && p.size % 16 == 0 && p.size >= 16 && p.size <= 128;
  if (p.body == kProductShort) return p.nt == 8 ? p.size == 32 : p.nt == 4 && (p.size == 16 || p.size == 32 || p.size == 48 || p.size == 64);
  return false;
}
inline int64_t product_units(const ProductPlan& p, int rows, int n) {
  const int wrows = p.body == kProductShort ? 16 * p.nt : 64 * p.nt;
  return (int64_t)((rows + p.size - 1) / p.size) * ((n + wrows - 1) / wrows) * p.shares;
}

// us of a launch: a workgroup's way in and out, its k-steps, and the megabytes that leave; of workgroups that have a CU each, and of up to two a
// CU.  Least squares over 2690 products of 65 to 2200 rows, n 768 to 8192, k 512 to 14336, all plans of up to 512 workgroups: 4 to 10 %
// (root mean square) off; what it chooses takes 1.3 % longer than the best plan.
struct ProductTimes {
  float fixed, step, out;
};
inline double product_time(const ProductPlan& p, int rows, int n, int k) {
  static const ProductTimes kShort[5][2] = {{{3.15f, .0637f, .15f}, {3.0f, .128f, .2f}},   {{2.7f, .12f, .26f}, {3.05f, .192f, .15f}},
                                            {{2.95f, .154f, .24f}, {3.55f, .239f, .15f}}, {{3.0f, .184f, .215f}, {3.45f, .301f, .15f}},
                                            {{3.25f, .177f, .206f}, {3.5f, .278f, .157f}}};  // 16, 32, 48, 64 rows; 32 with nt = 8
  static const ProductTimes kTile[2][5][2] = {{{{3.05f, .16f, .28f}, {5.2f, .315f, .14f}},
                                               {{3.45f, .173f, .25f}, {4.0f, .305f, .236f}},
                                               {{3.7f, .1815f, .216f}, {3.75f, .325f, .235f}},
                                               {{4.1f, .223f, .22f}, {5.2f, .385f, .173f}},
                                               {{4.15f, .237f, .224f}, {4.0f, .405f, .26f}}},
                                              {{{3.3f, .268f, .27f}, {7.9f, .565f, .1f}},
                                               {{4.3f, .276f, .206f}, {3.85f, .507f, .214f}},
                                               {{4.95f, .304f, .183f}, {4.4f, .559f, .191f}},
                                               {{5.65f, .3435f, .163f}, {7.3f, .648f, .123f}},
                                               {{6.25f, .367f, .147f}, {4.0f, .67f, .21f}}}};  // nt = 2, 4; up to 64, 80, 96, 112, 128 rows
  const bool two = product_units(p, rows, n) > 256;
  const ProductTimes& t = p.body == kProductShort ? kShort[p.nt == 8 ? 4 : p.size / 16 - 1][two]
                                                  : kTile[p.nt == 4][p.size <= 64 ? 0 : p.size / 16 - 4][two];
  const double mb = (double)rows * n * 1e-6;
  double us = t.fixed + t.step * product_share(p, k) + t.out * mb * (p.shares > 1 ? 4 * p.shares : 2);
  if (p.shares > 1) us += .2 * mb * (4 * p.shares - 2);  // the slabs' way into the launch that sums them
  return us;
}

// The shortest of the plans, and the library where its products are the better ones, by the rate that the plan reaches, TFLOP/s (of those 2690, own
// time of the library's; host time, 3 us for 20, not counted):
//   * K may be cut into slabs: up to 750; above k = 5120, where the library cuts too little, wherever it is cut.  0.76 in the mean, one in ten above 0.96: 300 rows of 14336 for 4096 62 us, 42 (and 2 more to sum them); 1000 131, 100 (10); 100 rows 38, 22 (4); 300 rows of 4096 for
//     4096 24.7, 17.5; of 4096 for 1024 13.9, 8.4.  From there on many tiles fill the chip, and the library's, both of whose operands go
//     through LDS, take less power: up to 1.22.
//   * one share: k <= 1024 up to 850, 0.84 (1000 rows of 1024 for 3072 14.0, 12.0; 100 rows of 1024 for 1024 8.4, 5.2).  Longer ones have too few
//     workgroups in between: k <= 2048 below 100 and from 400 to 800, 0.87; k <= 5120 from 550 to 850, 0.93; 0.95 to 1.5 elsewhere.
inline ProductPlan prompt_product_plan(int rows, int n, int k, bool gelu, bool slabs) {
  ProductPlan best{kProductNone, 0, 0, 0};
  if (rows <= 64 || rows > 8192 || n < 16 || n % 16 != 0 || k < 256 || k % 64 != 0 || (int64_t)n * k >= (int64_t)1 << 30) return best;
  double least = 0;
  auto take = [&](const ProductPlan& p) {
    if (!product_plan_valid(p, k) || product_units(p, rows, n) > 512 || (p.shares > 1 && k / 32 / p.shares < 8)) return;
    const double us = product_time(p, rows, n, k);
    if (best.body == kProductNone || us < least) best = p, least = us;
  };
  for (int shares = 1; shares <= (slabs ? kProductShares : 1); ++shares) {
    for (int size = 16; size <= 64; size += 16) take({kProductShort, size, 4, shares});
    take({kProductShort, 32, 8, shares});
    if (gelu) continue;  // (tile_linear.hip has those)
    int before = 0;
    for (int most = 128; most >= 64; most -= 16) {
      const int tiles = (rows + most - 1) / most;
      if (tiles == before) continue;
      before = tiles;
      const int size = ((rows + tiles - 1) / tiles + 15) / 16 * 16;
      take({kProductTile, size, 2, shares});
      take({kProductTile, size, 4, shares});
    }
  }
  if (best.body == kProductNone) return best;
  const double rate = 2e-6 * rows * n * k / least;
  const bool good = slabs        ? (k <= 5120 ? rate <= 750 : best.shares > 1)
                    : k <= 1024  ? rate <= 850
                    : k <= 2048  ? rate < 100 || (rate >= 400 && rate <= 800)
                    : k <= 5120  ? rate >= 550 && rate <= 850
                                 : false;
  return good ? best : ProductPlan{kProductNone, 0, 0, 0};
}

}  // namespace lvllm
