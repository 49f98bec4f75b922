// Projections of prompts with an activation behind them: which kernel takes which, in whole numbers.
#pragma once
#include <stdint.h>

#include "../../include/lvllm_hip.h"

namespace lvllm {

// Gated units: an output is made of a gate row and a value row.
constexpr bool prompt_pairs(int act) { return act == LVLLM_ACT_SILU_AND_MUL || act == LVLLM_ACT_CLAMPED_UNIT; }

// What takes a projection: the library and a launch of the activation (none of these), tiles of up to 64 groups rows x 256 W rows one a CU
// over row-major weights (wide_linear.hip), or tiles of 128 rows x 64 nt W rows two a CU over packed weights (tile_linear.hip).
struct PromptLinearPlan {
  int body;    // LVLLM_PROMPT_*
  int groups;  // wide
  int nt;      // tile
};

// Times in hundredths of a launch of at most one whole tile (nt = 4) a CU, 32 us at k = 2048, as measured (gated units of 5632 and
// 11264, 2048 wide, 65 to 8192 rows):
//   * whole tiles: a CU's second one beside the first 0.50 to 0.81 (0.65 to 0.81 from k = 3072 on); from the third on a round of both at 1.58
//     (1.64), and 0.70 of ends;
//   * half tiles (nt = 2): 0.71 alone, 0.85 to 1.19 two, then 1.05 a round and 0.45 (0.9 to 1.0 of that where k is a multiple of 64, deep_tile.h; no
//     choice between them and the others turned on it);
//   * wide ones take turns, 256 tiles at a time, of 0.97, 1.28 and 1.64 with 2, 3 and 4 groups; of 0.88, 1.17, 1.50 from k = 3072 on, where
//     their way in and out counts less.  Nothing covers their activations: 4 % more with SwiGLU, 10 % with the clamped unit, whose
//     exponential and division are the mathematical library's.
inline int64_t tile_time(int64_t units, int nt, int k) {
  const int second = k < 3072 ? 150 : 165;
  if (nt == 4) return units <= 256 ? 100 : units <= 512 ? second + (181 - second) * (units - 256) / 256 : (k < 3072 ? 158 : 164) * units / 512 + 70;
  return units <= 256 ? 71 : units <= 512 ? 85 + 34 * (units - 256) / 256 : 105 * units / 512 + 45;
}
inline int64_t wide_time(int64_t units, int groups, int k, int act) {
  static const int kTurn[2][5] = {{0, 0, 97, 128, 164}, {0, 0, 88, 117, 150}};
  const int more = act == LVLLM_ACT_CLAMPED_UNIT ? 110 : act == LVLLM_ACT_SILU_AND_MUL ? 104 : 100;
  return (units + 255) / 256 * kTurn[k >= 3072][groups] * more / 100;
}

// The shortest of these; `row_major`, `packed`: the orders of the weights that are there.  Nothing where the half tiles are too few to fill
// half of the chip: the library cuts K then.  Nor where its products are the better ones, of 1750 random sizes of 65 to 9000 rows:
//   * k > 5120: 0.71 to 1.23 of the library and the activation, whatever the rest.  (Up to 256 rows of k >= 8192 have a kernel of their own,
//     stream_gemm_kernel, which is ahead of both: SwiGLU of 8192, 100 rows 68.5 us, here 92.5.)
//   * 2048 < k: tiles that are filled to less than 0.6 of what MFMAs do in the time, but for half tiles that take most of the CUs once, 0.94 to
//     1.22 (SwiGLU of 9728, 2560 wide, 214 rows 47.8, 52.4; of 18944, 3584 wide, 89 rows 80, 88; of 14336, 4096 wide, 129 rows 74, 82);
//   * GELU from k = 1025 on, to less than 0.7, with the same exception: 0.8 to 1.12.
// What is left takes 0.46 to 1.09 of the two (1000 other sizes, three above 1.03), mean 0.84.  us, the two launches, then this:
//   * SwiGLU of 14336, 4096 wide: 65 rows 58, 45; 300 88, 84; 700 163, 144; 1000 206, 195; 2000 382, 376; 3000 575, 515; 4875 990, 855; 8192 1398,
//     1346; of 11264, 2048 wide: 128 rows 32, 27; 700 99, 77; 1000 106, 85; 2000 193, 164; 4096 402, 320; 8192 634, 577;
//   * the clamped unit of 5632, 2048 wide: 100 rows (88 half tiles) 21.1, 23.0; 200 30.6, 22.7; 300 32.6, 27.2; 512 39, 34; 1000 58, 55; 2000 99, 88;
//     4096 191, 161; of 11008, 4096 wide: 300 75, 76; 2000 425, 300;
//   * squared ReLU of 8448, 2048 wide: 100 rows (66) 19.4, 20.8; 300 27.9, 21.4; 700 37.7, 31.1; 1000 43.6, 40.4; 4096 141, 120; 8192 311, 223;
//   * GELU of 4096, 1024 wide: 100 rows (32) 11.7, 12.3; 300 (96) 13.9, 12.6; 1000 20.8, 14.2; 3000 37.3, 31.8; 16384 164, 131.  Its
//     instructions run beside another tile's MFMAs, where a wide tile (149) has nobody beside it.
// (Cards differ: one measured 154 and 125 for the last, and 891 + 73 and 842 for 4875 rows of SwiGLU.)
inline PromptLinearPlan prompt_linear_plan(int rows, int outputs, int k, int act, bool row_major, bool packed) {
  PromptLinearPlan plan{LVLLM_PROMPT_NONE, 0, 0};
  const int64_t wrows = (int64_t)outputs * (prompt_pairs(act) ? 2 : 1);
  const bool gelu = act == LVLLM_ACT_GELU;
  if (rows <= 64 || outputs < 128 || outputs % 16 != 0 || k > 5120 || wrows * k >= (int64_t)1 << 30) return plan;
  const int64_t tiles = (rows + 127) / 128, half = tiles * ((wrows + 127) / 128);
  if (half < (gelu ? 96 : 128)) return plan;
  int64_t best = 0;
  auto take = [&](int body, int groups, int nt, int64_t time) {
    if (plan.body == LVLLM_PROMPT_NONE || time < best) plan = {body, groups, nt}, best = time;
  };
  if (row_major && !gelu && k % 64 == 0 && k >= 512)
    for (int g = 4; g >= 2; --g) take(LVLLM_PROMPT_WIDE, g, 0, wide_time((rows + 64 * g - 1) / (64 * g) * ((wrows + 255) / 256), g, k, act));
  if (packed && k % 32 == 0 && (!gelu || k <= 2048)) {
    take(LVLLM_PROMPT_TILE, 0, 4, tile_time(tiles * ((wrows + 255) / 256), 4, k));
    take(LVLLM_PROMPT_TILE, 0, 2, tile_time(half, 2, k));
  }
  // What 2^23 products of rows with W rows, one whole tile a CU, take at the rate of full tiles is 80 of tile_time.
  auto filled = [&](int most) { return best << 23 <= (int64_t)rows * wrows * most; };
  const bool once = plan.body == LVLLM_PROMPT_TILE && plan.nt == 2 && half >= 160 && half <= 256;
  if (!once && (gelu ? k > 1024 && !filled(114) : k > 2048 && !filled(132))) plan = {LVLLM_PROMPT_NONE, 0, 0};
  return plan;
}

// Rows of a launch's tiles of up to 128, in 16s.
inline int tile_groups(int rows) { return ((rows + (rows + 127) / 128 - 1) / ((rows + 127) / 128) + 15) / 16; }

// Half tiles whose loads are dealt among their MFMAs (deep_tile.h), k a multiple of 64.  What they take of the others' time, of 114 products, weights
// from memory, by groups of 16 rows in a tile: 0.97 with 8 and 0.96 with 7 (0.88 to 1.02) where up to 256 tiles have a CU each, 0.96 and 0.94
// beyond; 0.99 with 5 up to 256 tiles, 1.02 beyond; with 6, which the others have a body of, 1.02 and 1.05 (SwiGLU of 5632, 2048 wide, 288 rows
// 26.3 us, 28.0).  GELU, 0.94 with 7 and 0.97 with 8 but 0.86 to 1.18, is left to the others.  us: squared ReLU of 8448, 2048 wide, 300 rows
// (198 tiles) 20.8, 20.2; 500 (264) 31.9, 29.2; the clamped unit of 5632, 200 rows (176) 22.9, 21.8; 400 (352) 34.8, 31.9; SwiGLU of 14336,
// 4096 wide, 65 to 128 rows level.
inline bool dealt_half_tiles(int rows, int wrows, int k, int act) {
  const int groups = tile_groups(rows);
  const int64_t units = (int64_t)((rows + 127) / 128) * ((wrows + 127) / 128);
  return k % 64 == 0 && act != LVLLM_ACT_GELU && (groups > 6 || (groups < 6 && units <= 256));
}

int launch_wide_linear(void* out, const void* x, const void* w, int rows, int outputs, int k, int act, float limit, int groups,
                       void* stream);
int launch_tile_linear(void* out, const void* x, const void* w, const void* bias, int rows, int outputs, int k, int act, float limit,
                       int nt, void* stream);

}  // namespace lvllm
