// Products of prompts of some hundreds of rows over packed weights, with a bias and GELU behind them or as fp32 slabs of shares of K that the
// next launch sums.  The library's are the better ones where there are many rows (prompt_product.h has the rule).
#include <algorithm>
#include <type_traits>

#include "gelu.h"
#include "moe_tile.h"
#include "prompt_product.h"

namespace lvllm {

struct PromptProduct {
  uint16_t* out;                   // [rows, n]; shares > 1: slabs
  float* slabs;                    // [shares, rows, n]
  const uint16_t *x, *w, *bias;    // x [rows, k], w packed [n, k], bias [n] or null
  int rows, n, k, gelu;
  int tiles, size, blocks;         // tiles of `size` rows, blocks of W rows
  int shares, per;                 // `per` k-steps each
};

// A workgroup's rows, W block and k-steps; an eighth of all units to each XCD, the row tiles of a block side by side, so that its L2 serves
// a block's weights to all of them.
struct ProductUnit {
  int row0, row1, block, share, step0, steps;
  bool any;
};
__device__ __forceinline__ ProductUnit product_unit(const PromptProduct& p) {
  const int units = p.tiles * p.blocks * p.shares, per = (units + 7) >> 3, mine = blockIdx.x >> 3, unit = (blockIdx.x & 7) * per + mine;
  ProductUnit u{};
  if (mine >= per || unit >= units) return u;
  const int tile = unit % p.tiles, rest = unit / p.tiles;
  u.block = rest % p.blocks;
  u.share = rest / p.blocks;
  u.row0 = tile * p.size;
  u.row1 = min(u.row0 + p.size, p.rows);
  u.step0 = u.share * p.per;
  u.steps = min(p.per, (p.k >> 5) - u.step0);
  u.any = u.row0 < u.row1 && u.steps > 0;
  return u;
}

// Short prompts: 16 MT rows x 16 NT W rows a workgroup, whose four waves take a quarter of its k-steps each and meet in LDS.  What bounds these
// launches is the way to memory and back, so that nothing goes through LDS first: both operands come straight to the registers, B k-steps at
// once and the next B behind them, and 1024 of K is two round trips.
template <int MT, int NT, int B>
__global__ __launch_bounds__(256, 2) void short_product_kernel(const PromptProduct p) {
  constexpr int kWaves = 4, kTiles = MT * NT;
  static_assert(kTiles % kWaves == 0, "a wave sums its share of the tiles");
  __shared__ __attribute__((aligned(16))) char sums[kWaves][kTiles][1024];
  const ProductUnit u = product_unit(p);
  if (!u.any) return;
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int all = p.k >> 5, ntiles = p.n >> 4;
  const int each = (u.steps / B + kWaves - 1) / kWaves * B, k0 = u.step0 + min(wave * each, u.steps), mine = min(each, u.step0 + u.steps - k0);
  const uint16_t *w[NT], *x[MT];
#pragma unroll
  for (int n = 0; n < NT; ++n) w[n] = p.w + (int64_t)min(u.block * NT + n, ntiles - 1) * all * 512 + lane * 8;
#pragma unroll
  for (int m = 0; m < MT; ++m) x[m] = p.x + (int64_t)min(u.row0 + m * 16 + c, p.rows - 1) * p.k + 8 * g;
  e_f32x4_t acc[NT][MT];
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = e_f32x4_t{0.f, 0.f, 0.f, 0.f};
  e_u32x4_t a[2][B][NT], b[2][B][MT];
  auto fetch = [&](int i, int at) __attribute__((always_inline)) {  // (past the end: the last step once more)
#pragma unroll
    for (int j = 0; j < B; ++j) {
      const int k = min(k0 + i + j, all - 1);
#pragma unroll
      for (int m = 0; m < MT; ++m) b[at][j][m] = *reinterpret_cast<const e_u32x4_t*>(x[m] + k * 32);
#pragma unroll
      for (int n = 0; n < NT; ++n) a[at][j][n] = *reinterpret_cast<const e_u32x4_t*>(w[n] + k * 512);
    }
  };
  auto use = [&](int at) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < B; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n][m] = moe_mfma(a[at][j][n], b[at][j][m], acc[n][m]);
  };
  fetch(0, 0);
  int i = 0;
  for (; i + 2 * B < mine; i += 2 * B) {
    fetch(i + B, 1);
    use(0);
    fetch(i + 2 * B, 0);
    use(1);
  }
  if (i + B < mine) {
    fetch(i + B, 1);
    use(0);
    use(1);
  } else if (i < mine) {
    use(0);
  }
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) *reinterpret_cast<e_f32x4_t*>(&sums[wave][m * NT + n][lane * 16]) = acc[n][m];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < kTiles / kWaves; ++i) {
    const int t = wave * (kTiles / kWaves) + i, row = u.row0 + t / NT * 16 + c, tile = u.block * NT + t % NT, col = tile * 16 + 4 * g;
    e_f32x4_t s = *reinterpret_cast<const e_f32x4_t*>(&sums[0][t][lane * 16]);
#pragma unroll
    for (int q = 1; q < kWaves; ++q) s += *reinterpret_cast<const e_f32x4_t*>(&sums[q][t][lane * 16]);
    if (row >= u.row1 || tile >= ntiles) continue;
    if (p.shares > 1) {
      *reinterpret_cast<e_f32x4_t*>(p.slabs + ((int64_t)u.share * p.rows + row) * p.n + col) = s;
      continue;
    }
    float z[4] = {0.f, 0.f, 0.f, 0.f}, v[4];
    if (p.bias != nullptr) load4<BF16>(p.bias + col, z);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = p.gelu ? gelu_of(s[r] + z[r]) : s[r] + z[r];
    store4<BF16>(p.out + (int64_t)row * p.n + col, v);
  }
}

// Longer ones: the tiles of moe_tile.h, 64 NT W rows x up to 128 rows, two workgroups a CU, each a share of K.
template <int NT, int MT>
__device__ __forceinline__ void tile_product(const PromptProduct& p, const ProductUnit& u, char (*ring)[kStageBytes]) {
  e_f32x4_t acc[NT][MT];
  TileWork t{};
  t.block = u.block;
  t.s0 = u.row0;
  t.s1 = u.row1;
  t.steps = u.steps;
  t.all = p.k >> 5;
  t.ntiles = p.n >> 4;
  tile_sums<false>(acc, p.x + u.step0 * 32, p.k, p.w + u.step0 * 512, t, ring, [](int row) { return row; }, [](int tile) { return tile; });
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
  tile_store<false>(p.out, p.n, acc, ring[0] + wave * 2048, nt0, t.ntiles, t.s0, t.s1, [](int) { return 1.f; },
                    [&](float, int n, const e_f32x4_t& a, const e_f32x4_t&, float (&v)[4]) {
#pragma unroll
                      for (int r = 0; r < 4; ++r) v[r] = a[r] + z[n][r];
                    });
}
template <int NT>
__global__ __launch_bounds__(256, 2) void tile_product_kernel(const PromptProduct p) {
  __shared__ __attribute__((aligned(16))) char ring[tile_steps(NT) / 2][kStageBytes];
  const ProductUnit u = product_unit(p);
  if (!u.any) return;
  const int groups = (u.row1 - u.row0 + 15) >> 4;
  if (groups <= 4) tile_product<NT, 4>(p, u, ring);
  else if (groups <= 5) tile_product<NT, 5>(p, u, ring);
  else if (groups <= 6) tile_product<NT, 6>(p, u, ring);
  else if (groups <= 7) tile_product<NT, 7>(p, u, ring);
  else tile_product<NT, 8>(p, u, ring);
}

static int launch_product(PromptProduct p, const ProductPlan& plan, hipStream_t s) {
  p.shares = plan.shares;
  p.per = product_share(plan, p.k);
  p.size = plan.size;
  p.tiles = (p.rows + plan.size - 1) / plan.size;
  auto launch = [&](auto kernel, int wrows) {
    p.blocks = (p.n + wrows - 1) / wrows;
    hipLaunchKernelGGL(kernel, dim3((p.tiles * p.blocks * p.shares + 7) / 8 * 8), dim3(256), 0, s, p);
  };
  if (plan.body == kProductTile) {
    if (plan.nt == 4) launch(tile_product_kernel<4>, 256);
    else launch(tile_product_kernel<2>, 128);
  } else if (plan.nt == 8) {
    launch(short_product_kernel<2, 8, 2>, 128);
  } else if (plan.size == 16) {
    launch(short_product_kernel<1, 4, 4>, 64);
  } else if (plan.size == 32) {
    launch(short_product_kernel<2, 4, 2>, 64);
  } else if (plan.size == 48) {
    launch(short_product_kernel<3, 4, 2>, 64);
  } else {
    launch(short_product_kernel<4, 4, 2>, 64);
  }
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm

using namespace lvllm;

extern "C" int lvllm_prompt_product_plan(int rows, int n, int k, int gelu, int slabs, int* plan) {
  const ProductPlan p = prompt_product_plan(rows, n, k, gelu != 0, slabs != 0);
  if (plan != nullptr) plan[0] = p.body, plan[1] = p.size, plan[2] = p.nt, plan[3] = p.shares;
  return p.body == kProductNone ? 0 : p.shares;
}

extern "C" int lvllm_prompt_product(void* out, float* slabs, const void* x, const void* w_packed, const void* bias, int rows, int n, int k,
                                    int gelu, const int* plan, void* stream) {
  if (rows == 0) return 0;
  const ProductPlan p{plan[0], plan[1], plan[2], plan[3]};
  LV_CHECK(rows > 0 && n > 0 && k > 0 && n % 16 == 0 && k % 32 == 0, "n a multiple of 16 and k of 32");
  LV_CHECK((int64_t)rows * k < (int64_t)1 << 31 && (int64_t)rows * n < (int64_t)1 << 31 && (int64_t)n * k < (int64_t)1 << 31, "operands of fewer than 2^31 elements");
  LV_CHECK(((uintptr_t)out | (uintptr_t)slabs | (uintptr_t)x | (uintptr_t)w_packed | (uintptr_t)bias) % 16 == 0, "16-byte aligned pointers");
  LV_CHECK(product_plan_valid(p, k), "a plan of lvllm_prompt_product_plan");
  LV_CHECK(p.shares == 1 ? out != nullptr : slabs != nullptr && bias == nullptr && !gelu, "slabs are plain sums");
  LV_CHECK(!gelu || p.body == kProductShort, "GELU behind short products only");
  PromptProduct q{};
  q.out = (uint16_t*)out; q.slabs = slabs; q.x = (const uint16_t*)x; q.w = (const uint16_t*)w_packed; q.bias = (const uint16_t*)bias;
  q.rows = rows; q.n = n; q.k = k; q.gelu = gelu;
  return launch_product(q, p, (hipStream_t)stream);
}
