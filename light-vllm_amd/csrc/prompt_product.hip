// Products of prompts of some hundreds of rows over packed weights, with a bias and GELU behind them or as fp32 slabs of shares of K that the
// next launch sums.  The library's are the better ones where there are many rows (prompt_product.h has the rule).
#include <algorithm>

#include "deep_tile.h"
#include "gelu.h"
#include "prompt_product.h"

namespace lvllm {

struct PromptProduct {
  uint16_t* out;                   // [batch, rows, n]; shares > 1: slabs
  float* slabs;                    // [shares, rows, n]
  const uint16_t *x, *w, *bias;    // x [rows, k] in rows of ld, w packed [n, k], bias [n] or null
  int64_t ld, x_batch;             // of x's rows, of x's batches; w's lie back to back
  int rows, n, k, gelu;
  int tiles, size, blocks;         // tiles of `size` rows, blocks of W rows
  int shares, per;                 // `per` k-steps each; or batches, K whole
  int batch;
};

// A workgroup's rows, W block and k-steps; an eighth of all units to each XCD, the row tiles of a block side by side, so that its L2 serves
// a block's weights to all of them.
struct ProductUnit {
  int row0, row1, block, share, step0, steps, batch;
  bool any;
};
__device__ __forceinline__ ProductUnit product_unit(const PromptProduct& p) {
  const int units = p.tiles * p.blocks * p.shares * p.batch, per = (units + 7) >> 3, mine = blockIdx.x >> 3, unit = (blockIdx.x & 7) * per + mine;
  ProductUnit u{};
  if (mine >= per || unit >= units) return u;
  const int tile = unit % p.tiles, rest = unit / p.tiles;
  u.block = rest % p.blocks;
  u.share = rest / p.blocks;
  if (p.batch > 1) u.batch = u.share, u.share = 0;
  u.row0 = tile * p.size;
  u.row1 = min(u.row0 + p.size, p.rows);
  u.step0 = u.share * p.per;
  u.steps = min(p.per, (p.k >> 5) - u.step0);
  u.any = u.row0 < u.row1 && u.steps > 0;
  return u;
}

// Up to 128 rows x 64 NT W rows, two workgroups a CU, each a share of K: NT = 4 as moe_tile.h has them, the others, whose workgroups are few, as
// deep_tile.h.
template <int NT, int MT>
__device__ __forceinline__ void tile_product(const PromptProduct& p, const ProductUnit& u, char* lds) {
  e_f32x4_t acc[NT][MT];
  TileWork t{};
  t.block = u.block;
  t.s0 = u.row0;
  t.s1 = u.row1;
  t.steps = u.steps;
  t.all = p.k >> 5;
  t.ntiles = p.n >> 4;
  const uint16_t* const x = p.x + u.batch * p.x_batch + u.step0 * 32;
  const uint16_t* const w = p.w + (int64_t)u.batch * p.n * p.k + u.step0 * 512;
  auto same = [](int i) { return i; };
  if constexpr (NT <= 2) deep_sums(acc, x, p.ld, w, t, lds, same);
  else tile_sums<false>(acc, x, p.ld, w, t, reinterpret_cast<char(*)[kStageBytes]>(lds), same, same);
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), nt0 = (t.block * 4 + wave) * NT;
  if (p.shares > 1) {
    float* const out = p.slabs + (int64_t)u.share * p.rows * p.n;
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int row = t.s0 + m * 16 + c;
#pragma unroll
      for (int n = 0; n < NT; ++n)
        if (row < t.s1 && nt0 + n < t.ntiles) *reinterpret_cast<e_f32x4_t*>(out + (int64_t)row * p.n + (nt0 + n) * 16 + 4 * g) = acc[n][m];
    }
    return;
  }
  float z[NT][4];
#pragma unroll
  for (int n = 0; n < NT; ++n) {
#pragma unroll
    for (int r = 0; r < 4; ++r) z[n][r] = 0.f;
    if (p.bias != nullptr) load4<BF16>(p.bias + min(nt0 + n, t.ntiles - 1) * 16 + 4 * g, z[n]);
  }
  tile_store<false>(p.out + (int64_t)u.batch * p.rows * p.n, p.n, acc, lds + wave * 2048, nt0, t.ntiles, t.s0, t.s1, [](int) { return 1.f; },
                    [&](float, int n, const e_f32x4_t& a, const e_f32x4_t&, float (&v)[4]) {
#pragma unroll
                      for (int r = 0; r < 4; ++r) v[r] = NT < 4 && p.gelu ? gelu_of(a[r] + z[n][r]) : a[r] + z[n][r];
                    });
}
template <int NT>
__global__ __launch_bounds__(256, 2) void tile_product_kernel(const PromptProduct p) {
  __shared__ __attribute__((aligned(16))) char lds[NT == 4 ? tile_steps(4) / 2 * kStageBytes : deep_lds_bytes(NT == 2 ? 8 : 6)];
  const ProductUnit u = product_unit(p);
  if (!u.any) return;
  const int groups = (u.row1 - u.row0 + 15) >> 4;
  if constexpr (NT == 1) {
    if (groups <= 1) return tile_product<NT, 1>(p, u, lds);
    if (groups <= 2) return tile_product<NT, 2>(p, u, lds);
    if (groups <= 3) return tile_product<NT, 3>(p, u, lds);
  }
  if (groups <= 4) return tile_product<NT, 4>(p, u, lds);
  if (groups <= 5) return tile_product<NT, 5>(p, u, lds);
  if (NT == 1 || groups <= 6) return tile_product<NT, 6>(p, u, lds);
  if constexpr (NT > 1) {
    if (groups <= 7) return tile_product<NT, 7>(p, u, lds);
    tile_product<NT, 8>(p, u, lds);
  }
}

static int launch_product(PromptProduct p, const ProductPlan& plan, hipStream_t s) {
  p.shares = plan.shares;
  p.per = product_share(plan, p.k);
  p.size = plan.size;
  p.tiles = (p.rows + plan.size - 1) / plan.size;
  auto launch = [&](auto kernel, int wrows) {
    p.blocks = (p.n + wrows - 1) / wrows;
    hipLaunchKernelGGL(kernel, dim3((p.tiles * p.blocks * p.shares * p.batch + 7) / 8 * 8), dim3(256), 0, s, p);
  };
  if (plan.nt == 4) launch(tile_product_kernel<4>, 256);
  else if (plan.nt == 2) launch(tile_product_kernel<2>, 128);
  else launch(tile_product_kernel<1>, 64);
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm

using namespace lvllm;

extern "C" int lvllm_prompt_product_plan(int rows, int n, int k, int gelu, int sums, int batch, int* plan) {
  const ProductPlan p = prompt_product_plan(rows, n, k, gelu != 0, sums, batch);
  if (plan != nullptr) plan[0] = p.size, plan[1] = p.nt, plan[2] = p.shares;
  return p.size == 0 ? 0 : p.shares;
}

extern "C" int lvllm_prompt_product(void* out, float* slabs, const void* x, int64_t x_stride, int64_t x_batch_stride,
                                    const void* w_packed, const void* bias, int rows, int n, int k, int gelu, int batch, const int* plan, void* stream) {
  if (rows == 0) return 0;
  LV_CHECK(plan != nullptr && x != nullptr && w_packed != nullptr, "a plan, x and weights");
  const ProductPlan p{plan[0], plan[1], plan[2]};
  LV_CHECK(rows > 0 && n > 0 && k > 0 && n % 16 == 0 && k % 64 == 0, "n a multiple of 16 and k of 64");
  LV_CHECK(x_stride >= k && x_stride % 8 == 0, "rows of x 16-byte aligned, one after the other");
  LV_CHECK(batch >= 1 && batch <= 64 && x_batch_stride % 8 == 0 && (batch == 1 || (p.shares == 1 && bias == nullptr && !gelu)), "batches: plain, K whole");
  LV_CHECK((int64_t)rows * k < (int64_t)1 << 31 && (int64_t)rows * n < (int64_t)1 << 31 && (int64_t)n * k < (int64_t)1 << 31, "operands of fewer than 2^31 elements");
  LV_CHECK(((uintptr_t)out | (uintptr_t)slabs | (uintptr_t)x | (uintptr_t)w_packed | (uintptr_t)bias) % 16 == 0, "16-byte aligned pointers");
  LV_CHECK(product_plan_valid(p, k), "a plan of lvllm_prompt_product_plan");
  LV_CHECK(p.shares == 1 ? out != nullptr : slabs != nullptr && bias == nullptr && !gelu, "slabs are plain sums");
  LV_CHECK(!gelu || p.nt < 4, "GELU behind tiles of up to 128 W rows only");
  PromptProduct q{};
  q.out = (uint16_t*)out; q.slabs = slabs; q.x = (const uint16_t*)x; q.w = (const uint16_t*)w_packed; q.bias = (const uint16_t*)bias;
  q.ld = x_stride; q.x_batch = x_batch_stride; q.batch = batch; q.rows = rows; q.n = n; q.k = k; q.gelu = gelu;
  return launch_product(q, p, (hipStream_t)stream);
}
