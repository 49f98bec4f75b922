// Projections of prompts with an activation behind them (GELU, squared ReLU, SwiGLU, the clamped unit), in the tiles of moe_tile.h over packed weights:
// two workgroups share a CU, and one's activations, 13 vector instructions a GELU, run beside the other's MFMAs.  16384 rows of 1024, GELU of
// 4096: 125 us for 105 and 49 in two launches (one workgroup a CU 149), on another card 143 for 162; prompt_linear.h has more.
#include <type_traits>

#include "deep_tile.h"
#include "gelu.h"
#include "prompt_act.h"
#include "prompt_linear.h"

namespace lvllm {

struct TileLinear {
  uint16_t* out;                  // [rows, outputs]
  const uint16_t *x, *w, *bias;   // x [rows, k], w packed [n, k] (pairs: [gate rows | value rows]), bias [n] (GELU)
  int rows, outputs, k, tiles, size, blocks;  // tiles of `size` rows, up to 128, blocks of W rows
  float limit;                    // CLAMPED_UNIT
};

template <int ACT, int NT, int MT, bool DEEP>
__device__ __forceinline__ void tile_linear(const TileLinear& p, const TileWork& t, char* lds) {
  constexpr bool GELU = ACT == LVLLM_ACT_GELU, PAIRS = prompt_pairs(ACT);
  e_f32x4_t acc[NT][MT];
  // PAIRS: 16 gate rows, the 16 value rows that belong to them, ...
  auto tile_of = [&](int tile) { return PAIRS ? (tile & 1) * (p.outputs >> 4) + (tile >> 1) : tile; };
  if constexpr (DEEP) deep_sums(acc, p.x, p.k, p.w, t, lds, tile_of);
  else tile_sums<false>(acc, p.x, p.k, p.w, t, reinterpret_cast<char(*)[kStageBytes]>(lds), [](int slot) { return slot; }, tile_of);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nt0 = (t.block * 4 + wave) * NT, g = (threadIdx.x & 63) >> 4;
  float z[NT][4];
  if constexpr (GELU)
#pragma unroll
    for (int n = 0; n < NT; ++n) load4<BF16>(p.bias + min(nt0 + n, t.ntiles - 1) * 16 + 4 * g, z[n]);
  tile_store<PAIRS>(p.out, p.outputs, acc, lds + wave * 2048, nt0, t.ntiles, t.s0, t.s1, [](int) { return 1.f; },
                    [&](float, int n, const e_f32x4_t& a, const e_f32x4_t& b, float (&v)[4]) {
#pragma unroll
                      for (int r = 0; r < 4; ++r) {
                        if constexpr (GELU) v[r] = gelu_of(a[r] + z[n][r]);
                        else v[r] = prompt_act<ACT>(a[r], b[r], p.limit);
                      }
                    });
}

// An eighth of the tiles to each XCD, 1024 rows side by side, W block after W block.  DEEP: half tiles by deep_tile.h (dealt_half_tiles).
template <int ACT, int NT, bool DEEP>
__global__ __launch_bounds__(256, 2) void tile_linear_kernel(const TileLinear p) {
  __shared__ __attribute__((aligned(16))) char ring[DEEP ? deep_lds_bytes(8) : tile_steps(NT) / 2 * kStageBytes];
  constexpr int kSide = 1024 / kMoeTile;
  const int units = p.tiles * p.blocks, per = (units + 7) >> 3, mine = blockIdx.x >> 3, unit = (blockIdx.x & 7) * per + mine;
  if (mine >= per || unit >= units) return;
  const int strip = unit / (kSide * p.blocks), side = min(kSide, p.tiles - strip * kSide), in = unit - strip * kSide * p.blocks;
  TileWork t{};
  t.block = in / side;
  const int size = p.size;
  t.s0 = (strip * kSide + in - t.block * side) * size;
  t.s1 = min(t.s0 + size, p.rows);
  if (t.s0 >= t.s1) return;
  t.steps = t.all = p.k >> 5;
  t.ntiles = (prompt_pairs(ACT) ? 2 : 1) * (p.outputs >> 4);
  const int groups = (t.s1 - t.s0 + 15) >> 4;
  if (groups <= 4) tile_linear<ACT, NT, 4, DEEP>(p, t, ring);
  else if (DEEP && groups <= 5) tile_linear<ACT, NT, DEEP ? 5 : 6, DEEP>(p, t, ring);
  else if (groups <= 6) tile_linear<ACT, NT, 6, DEEP>(p, t, ring);
  else if (DEEP && groups <= 7) tile_linear<ACT, NT, DEEP ? 7 : 8, DEEP>(p, t, ring);
  else tile_linear<ACT, NT, 8, DEEP>(p, t, ring);
}

int launch_tile_linear(void* out, const void* x, const void* w, const void* bias, int rows, int outputs, int k, int act, float limit,
                       int nt, void* stream) {
  TileLinear p{};
  p.out = (uint16_t*)out; p.x = (const uint16_t*)x; p.w = (const uint16_t*)w; p.bias = (const uint16_t*)bias;
  p.rows = rows; p.outputs = outputs; p.k = k; p.limit = limit;
  p.tiles = (rows + kMoeTile - 1) / kMoeTile;
  p.size = 16 * tile_groups(rows);
  const bool dealt = dealt_half_tiles(rows, (prompt_pairs(act) ? 2 : 1) * outputs, k, act);
  auto launch = [&](auto act, auto nt, auto deep) {
    constexpr int ACT = decltype(act)::value, NT = decltype(nt)::value;
    p.blocks = ((prompt_pairs(ACT) ? 2 : 1) * outputs + 64 * NT - 1) / (64 * NT);
    hipLaunchKernelGGL((tile_linear_kernel<ACT, NT, decltype(deep)::value>), dim3((p.tiles * p.blocks + 7) / 8 * 8), dim3(256), 0, (hipStream_t)stream, p);
  };
  auto with = [&](auto act) {
    constexpr std::integral_constant<int, 2> two{};
    if (nt == 4) launch(act, std::integral_constant<int, 4>{}, std::false_type{});
    else if (dealt) launch(act, two, std::integral_constant<bool, decltype(act)::value != LVLLM_ACT_GELU>{});
    else launch(act, two, std::false_type{});
  };
  if (act == LVLLM_ACT_GELU) with(std::integral_constant<int, LVLLM_ACT_GELU>{});
  else if (act == LVLLM_ACT_RELU_SQUARED) with(std::integral_constant<int, LVLLM_ACT_RELU_SQUARED>{});
  else if (act == LVLLM_ACT_SILU_AND_MUL) with(std::integral_constant<int, LVLLM_ACT_SILU_AND_MUL>{});
  else with(std::integral_constant<int, LVLLM_ACT_CLAMPED_UNIT>{});
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm
