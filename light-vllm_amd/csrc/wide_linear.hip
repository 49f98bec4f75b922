// Projections of prompts with a gated unit or squared ReLU behind them, in the tiles of wide_tile.h over the library's row-major weights: what
// they leave is the activation of what the projection would, in one launch and without its way through memory.  4875 rows of 4096, SwiGLU of
// 14336: 842 us (1.36 PFLOP/s) for 891 and 73 in two launches, on another card 855 for 990; prompt_linear.h has more.
#include <algorithm>
#include <type_traits>

#include "prompt_act.h"
#include "prompt_linear.h"
#include "wide_tile.h"

namespace lvllm {

struct WideLinear {
  uint16_t* out;                      // [rows, outputs]
  const uint16_t *x, *w;              // x [rows, k], w [n, k]; gated units: [gate rows | value rows]
  int rows, outputs, k, tile, tiles;  // tiles of `tile` rows
  int blocks;                         // of 256 W rows
  float limit;                        // CLAMPED_UNIT
};

// W block `block` of rows row0 .. row1 - 1
struct WideLinearUnit {
  int block, row0, row1;
};
template <int ACT>
__device__ __forceinline__ void wide_linear_tile(const WideLinear& p, const WideLinearUnit& u, WideTile& t) {
  constexpr bool PAIRS = prompt_pairs(ACT);
  const int lane = wide_lane(), wave = wide_wave(), ld = p.k * 2;
  t.iters = p.k >> 6;
  t.groups = (u.row1 - u.row0 + 63) >> 6;
  t.x = p.x + (int64_t)u.row0 * p.k;
  t.x_bytes = (unsigned)((u.row1 - u.row0) * ld);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    t.x_at[j] = min((wave * 2 * t.groups + j) * 8 + (lane >> 3), u.row1 - u.row0 - 1) * ld + wide_chunk(lane) * 16;
  t.w = p.w;
  t.w_bytes = (unsigned)(p.outputs * (PAIRS ? 2 : 1)) * (unsigned)ld;
  t.w_lane = (lane >> 3) * ld + wide_chunk(lane) * 16;
#pragma unroll
  for (int j = 0; j < 8; ++j) {  // 8 rows; PAIRS: 16 gate rows, the 16 value rows that belong to them, ...
    const int r = wave * 64 + j * 8, row = PAIRS ? u.block * 128 + (r >> 5) * 16 + (r & 8) : u.block * 256 + r;
    t.w_at[j] = (min(row, p.outputs - 8) + (PAIRS && (r & 16) ? p.outputs : 0)) * ld;
  }
}

template <int ACT, int MT>
__device__ __forceinline__ void wide_linear_store(const WideLinear& p, const WideLinearUnit& u, const WideSums<MT>& sums, char* lds) {
  constexpr bool PAIRS = prompt_pairs(ACT);
  constexpr int kOuts = PAIRS ? 64 : 128;  // of a wave
  const int wave = wide_wave(), first = (u.block * 2 + (wave >> 1)) * kOuts, r0 = u.row0 + (wave & 1) * 32 * MT;
  wide_store<PAIRS>(sums, lds, p.out + (int64_t)r0 * p.outputs + first, p.outputs, u.row1 - r0, p.outputs - first,
                    [&](int, const w_f32x4_t& a, const w_f32x4_t& b, float (&v)[4]) {
#pragma unroll
                      for (int r = 0; r < 4; ++r) v[r] = prompt_act<ACT>(a[r], b[r], p.limit);
                    });
}

// An eighth of the tiles to each XCD, 8 row tiles side by side, W block after W block; a workgroup takes every 32nd of its XCD's.
template <int ACT>
__global__ __launch_bounds__(256, 1) void wide_linear_kernel(const WideLinear p) {
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int units = p.tiles * p.blocks, per = (units + 7) >> 3, step = gridDim.x >> 3;
  int mine = blockIdx.x >> 3;
  auto unit_of = [&](int at) {
    constexpr int kSide = 8;
    const int unit = (blockIdx.x & 7) * per + at;
    const int strip = unit / (kSide * p.blocks), side = min(kSide, p.tiles - strip * kSide), in = unit - strip * kSide * p.blocks;
    const int block = in / side, row0 = (strip * kSide + in - block * side) * p.tile;
    return WideLinearUnit{block, row0, min(row0 + p.tile, p.rows)};
  };
  auto any = [&](int at) { return at < per && (int)(blockIdx.x & 7) * per + at < units; };
  if (!any(mine)) return;
  WideLinearUnit u = unit_of(mine);
  WideTile t;
  wide_linear_tile<ACT>(p, u, t);
  wide_begin(t, lds);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  bool more = true;
  while (more) {
    const WideLinearUnit now = u;
    auto go = [&](auto groups) __attribute__((always_inline)) {
      constexpr int MT = decltype(groups)::value;
      WideSums<MT> sums;
      wide_walk(sums, t, lds);
      mine += step;
      more = any(mine);
      if (more) {
        u = unit_of(mine);
        wide_linear_tile<ACT>(p, u, t);
        wide_begin(t, lds);
      }
      wide_linear_store<ACT, MT>(p, now, sums, lds);
    };
    if (t.groups == 1) go(std::integral_constant<int, 1>{});
    else if (t.groups == 2) go(std::integral_constant<int, 2>{});
    else if (t.groups == 3) go(std::integral_constant<int, 3>{});
    else go(std::integral_constant<int, 4>{});
  }
}

template <int ACT>
static int launch(const WideLinear& p, hipStream_t s) {
  (void)hipFuncSetAttribute((const void*)wide_linear_kernel<ACT>, hipFuncAttributeMaxDynamicSharedMemorySize, kWideLds);
  hipLaunchKernelGGL(wide_linear_kernel<ACT>, dim3(std::min(kWideCus, (p.tiles * p.blocks + 7) / 8 * 8)), dim3(256), kWideLds, s, p);
  LV_LAUNCH_CHECK();
  return 0;
}

int launch_wide_linear(void* out, const void* x, const void* w, int rows, int outputs, int k, int act, float limit, int groups,
                       void* stream) {
  WideLinear p{};
  p.out = (uint16_t*)out; p.x = (const uint16_t*)x; p.w = (const uint16_t*)w;
  p.rows = rows; p.outputs = outputs; p.k = k; p.limit = limit;
  p.tile = 64 * groups;
  p.tiles = (rows + p.tile - 1) / p.tile;
  const int per = prompt_pairs(act) ? 128 : 256;
  p.blocks = (outputs + per - 1) / per;
  hipStream_t s = (hipStream_t)stream;
  if (act == LVLLM_ACT_SILU_AND_MUL) return launch<LVLLM_ACT_SILU_AND_MUL>(p, s);
  if (act == LVLLM_ACT_CLAMPED_UNIT) return launch<LVLLM_ACT_CLAMPED_UNIT>(p, s);
  return launch<LVLLM_ACT_RELU_SQUARED>(p, s);
}

}  // namespace lvllm

using namespace lvllm;

extern "C" int lvllm_prompt_linear_body(int rows, int outputs, int k, int act, int row_major, int packed) {
  return prompt_linear_plan(rows, outputs, k, act, row_major != 0, packed != 0).body;
}

extern "C" int lvllm_prompt_linear(void* out, const void* x, const void* w, const void* w_packed, const void* bias, int rows, int outputs,
                                   int k, int act, float limit, int dtype, void* stream) {
  if (rows == 0) return 0;
  LV_CHECK(act >= LVLLM_ACT_GELU && act <= LVLLM_ACT_CLAMPED_UNIT, "unknown activation");
  LV_CHECK(dtype == LVLLM_BF16, "bf16 only");
  LV_CHECK((bias != nullptr) == (act == LVLLM_ACT_GELU), "GELU takes a bias, the others none");
  LV_CHECK((((uintptr_t)out | (uintptr_t)x | (uintptr_t)w | (uintptr_t)w_packed | (uintptr_t)bias) & 15) == 0, "16-byte aligned pointers");
  const PromptLinearPlan plan = prompt_linear_plan(rows, outputs, k, act, w != nullptr, w_packed != nullptr);
  LV_CHECK(plan.body != LVLLM_PROMPT_NONE, "sizes that lvllm_prompt_linear_body does not take");
  if (plan.body == LVLLM_PROMPT_TILE) return launch_tile_linear(out, x, w_packed, bias, rows, outputs, k, act, limit, plan.nt, stream);
  return launch_wide_linear(out, x, w, rows, outputs, k, act, limit, plan.groups, stream);
}
