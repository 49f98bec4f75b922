// Projections of prompts with an activation behind them: which kernel takes which, in whole numbers.
#pragma once
#include <stdint.h>

#include "../../include/lvllm_hip.h"

namespace lvllm {

// What takes a projection: the library and a launch of the activation (none of these), tiles of up to 64 groups rows x 256 W rows one a CU
// over row-major weights (wide_linear.hip), or tiles of 128 rows x 64 nt outputs two a CU over packed weights (tile_linear.hip).
struct PromptLinearPlan {
  int body;    // LVLLM_PROMPT_*
  int groups;  // wide
  int nt;      // tile
};

// Wide tiles take turns of one a CU, 256 at a time; a turn of 64, 128, 192, 256 rows takes 40, 59, 78, 100 %.  `fill`: the share of the
// turns' time that is work on rows and outputs that are there.  us, library and activation, then this:
//   * SwiGLU of 14336, 4096 wide: 3000 rows (fill 94 %) 575, 524; 4875 964, 842; 8192 (100 %) 1397, 1323; 2000 (88 %) 380, 373; but 1000
//     (85 %) 201, 207; 1500 (85 %) 285, 292.  Of 11264, 2048 wide, where the activation is twice as large a part: 1000 (76 %) 104, 95;
//     4096 408, 308; 8192 632, 576; of 5632: 2000 (86 %) 95, 80; 8192 407, 301;
//   * at a few hundred rows the library fills the chip no better: 14336, 4096 wide, 300 rows (66 %) 88, 78; 700 (77 %) 164, 135; 512 (88 %)
//     109, 106; of 5632, 2048 wide, 512 (58 %) 38, 35; 300 (34 %) 33, 34;
//   * squared ReLU of 8448, 2048 wide: 1000 (65 %) 43.6, 40.3; 2000 80, 73; 4096 138, 114; 8192 311, 223.
inline PromptLinearPlan wide_plan(int rows, int outputs, int k, int act) {
  static const int kTurn[5] = {0, 40, 59, 78, 100};
  const int pairs = act == LVLLM_ACT_SILU_AND_MUL ? 2 : 1;
  const int64_t blocks = ((int64_t)pairs * outputs + 255) / 256;
  int64_t best = 0;
  int groups = 0;
  for (int g = 4; g >= 2; --g) {
    const int64_t turns = (((rows + 64 * g - 1) / (64 * g)) * blocks + 255) / 256, time = turns * kTurn[g];
    if (groups == 0 || time < best) best = time, groups = g;
  }
  const int64_t fill = (int64_t)rows * pairs * outputs * 100 / 256 / 256 * 100 / 256 / best;  // in per cent
  const int64_t least = rows <= 768 ? 50 : k <= 2048 ? 60 : 87;
  return {fill >= least ? LVLLM_PROMPT_WIDE : LVLLM_PROMPT_NONE, groups, 0};
}

// Tiles of 64 nt outputs: GELU, whose instructions then run beside another tile's MFMAs (a wide tile has nobody beside it), and squared ReLU
// of few rows.  Half blocks (nt = 2) up to 512 of them, from 96 on; whole ones of squared ReLU while they fit a CU each.  us, library and
// activation, then half and whole blocks: GELU of 4096, 1024 wide, 100 rows (32 half blocks) 11.7, 12.3, 18.6; 300 rows (96) 13.9,
// 12.6, 18.9; 1000 (256) 20.8, 14.2, 20.3; 2000 (512) 29.8, 22.8, 23.0; 3000 37.3, 33.7, 31.8; 16384 154, 125 whole, 149 wide; squared ReLU
// of 8448, 2048 wide, 100 rows (66) 19.4, 20.8, 29.8; 300 (198) 27.9, 21.4, 29.6; 700 (396; 198 whole) 37.7, 33.4, 31.1; 1000 (528; 264) 43.7, 50.4,
// 47.4.
inline PromptLinearPlan tile_plan(int rows, int outputs, int act) {
  const int64_t tiles = (rows + 127) / 128, half = tiles * ((outputs + 127) / 128), whole = tiles * ((outputs + 255) / 256);
  if (half < 96) return {LVLLM_PROMPT_NONE, 0, 0};
  if (act == LVLLM_ACT_GELU) return {LVLLM_PROMPT_TILE, 0, half <= 512 ? 2 : 4};
  if (half <= 264) return {LVLLM_PROMPT_TILE, 0, 2};
  return {whole <= 256 ? LVLLM_PROMPT_TILE : LVLLM_PROMPT_NONE, 0, 4};
}

// `row_major`, `packed`: the orders of the weights that are there.
inline PromptLinearPlan prompt_linear_plan(int rows, int outputs, int k, int act, bool row_major, bool packed) {
  const PromptLinearPlan none{LVLLM_PROMPT_NONE, 0, 0};
  const int64_t weights = (int64_t)outputs * (act == LVLLM_ACT_SILU_AND_MUL ? 2 : 1) * k;
  if (rows <= 64 || outputs < 128 || weights >= (int64_t)1 << 30) return none;
  if (packed && act != LVLLM_ACT_SILU_AND_MUL && outputs % 16 == 0 && k % 32 == 0 && k <= 2048) {
    const PromptLinearPlan t = tile_plan(rows, outputs, act);
    if (t.body != LVLLM_PROMPT_NONE) return t;
  }
  if (row_major && act != LVLLM_ACT_GELU && outputs % 16 == 0 && k % 64 == 0 && k >= 512) return wide_plan(rows, outputs, k, act);
  return none;
}

int launch_wide_linear(void* out, const void* x, const void* w, int rows, int outputs, int k, int act, int groups, void* stream);
int launch_tile_linear(void* out, const void* x, const void* w, const void* bias, int rows, int outputs, int k, int act, int nt,
                       void* stream);

}  // namespace lvllm
