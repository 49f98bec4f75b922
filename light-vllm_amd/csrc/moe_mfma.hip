// The products of moe.h on 16x16x32 bf16 MFMAs over packed weights: W rows are the A operand, slots the columns, so that a
// lane ends up with consecutive outputs of one slot, and gate and value of an activation in the same register of two tiles.
//
//   * few slots per expert (decode steps): bound by the weights' bytes.  A workgroup takes 16 slots of one expert and a share
//     of its outputs; the slots' rows sit in LDS in fragment order (2048 of K at a time), every wave streams the two W tiles
//     of its own (1 KiB a load, eight k-steps in flight behind the eight in use) and needs no other wave;
//   * prompts: tiles of up to 128 slots x 256 W rows, or 128 where those are few (moe_tile_kernel).  A slot's 128 bytes of two k-steps
//     are eight chunks, exchanged so that a fragment read is free of bank conflicts.
#include <algorithm>

#include "moe_tile.h"
#include "moe_turns.h"

namespace lvllm {

constexpr int kStreamBatch = 8, kStreamChunk = 64;  // k-steps per batch, per LDS chunk

// grid (shares of the outputs, tiles of 16 slots); a wave computes W tiles 2 u and 2 u + 1, or (KS > 1, when few
// experts have work) a KS-th of their k-steps, 64 / KS of every LDS chunk
template <int PRODUCT, int KS, bool ONCE>
__device__ __forceinline__ void stream_product(const MoeParams& p, const int e, const int s0, const int s1, char* sx,
                                               e_f32x4_t (*red)[2][64]) {
  constexpr bool UP = PRODUCT != kMoeDown, GATED = PRODUCT == kMoeGated;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int ff = p.ff[e], K = UP ? p.width : ff, steps = K >> 5;
  const int units = GATED ? ff >> 4 : (UP ? ff : p.width) >> 5;
  constexpr int U = 4 / KS, P = kStreamChunk / KS;  // units of a workgroup; this wave's k-steps of a chunk
  if ((int)blockIdx.x * U >= units) return;
  const int u = min((int)blockIdx.x * U + wave / KS, units - 1), kq = wave % KS;  // (a wave too many repeats the last unit)
  // k-steps, some missing ones of the last chunk included
  const int mine = KS == 1 ? (steps + 2 * kStreamBatch - 1) / (2 * kStreamBatch) * (2 * kStreamBatch)
                           : (steps + kStreamChunk - 1) / kStreamChunk * P;
  auto step_of = [&](int v) { return KS == 1 ? v : v / P * kStreamChunk + kq * P + v % P; };  // of batch v, a multiple of 8
  const uint16_t* w = (const uint16_t*)p.w + p.w_offset[e] + (int64_t)2 * u * steps * 512 + lane * 8;
  e_u32x4_t a[2][2][kStreamBatch];
  auto fetch = [&](int v, e_u32x4_t (&t)[2][kStreamBatch]) __attribute__((always_inline)) {
    const int b = step_of(v);
#pragma unroll
    for (int j = 0; j < kStreamBatch; ++j)
#pragma unroll
      for (int i = 0; i < 2; ++i)  // (a missing step: the last one again)
        t[i][j] = load_weights<ONCE>(w + ((int64_t)i * steps + min(b + j, steps - 1)) * 512);
  };
  fetch(0, a[0]);
  const int64_t ld = UP ? p.width : p.ff_max;
  const int my_slot = s0 + (threadIdx.x & 15);
  const int64_t row = my_slot >= s1 ? -1 : UP ? min(max(p.token[my_slot], 0), p.rows - 1) : my_slot;
  const uint16_t* x = (const uint16_t*)p.x + (row < 0 ? 0 : row) * ld;
  auto stage = [&](int step0) __attribute__((always_inline)) {
    const int n = min(kStreamChunk, steps - step0) * 64;
    for (int i = threadIdx.x; i < n; i += 256) {  // 16-byte chunk i: slot i % 16, entries 8 (i / 16) ..
      e_u32x4_t v{0, 0, 0, 0};
      if (row >= 0) v = *reinterpret_cast<const e_u32x4_t*>(x + step0 * 32 + (i >> 4) * 8);
      *reinterpret_cast<e_u32x4_t*>(sx + i * 16) = v;
    }
    __syncthreads();
  };
  const char* xf = sx + lane * 16;
  e_f32x4_t acc[2] = {e_f32x4_t{0.f, 0.f, 0.f, 0.f}, e_f32x4_t{0.f, 0.f, 0.f, 0.f}};
  auto use = [&](int v, const e_u32x4_t (&t)[2][kStreamBatch]) __attribute__((always_inline)) {
    const int b = step_of(v), at = b % kStreamChunk;
    auto one = [&](int j) __attribute__((always_inline)) {
      const e_u32x4_t xv = *reinterpret_cast<const e_u32x4_t*>(xf + (at + j) * 1024);
      acc[0] = moe_mfma(t[0][j], xv, acc[0]);
      acc[1] = moe_mfma(t[1][j], xv, acc[1]);
    };
    if (b + kStreamBatch <= steps) {
#pragma unroll
      for (int j = 0; j < kStreamBatch; ++j) one(j);
    } else {
#pragma unroll
      for (int j = 0; j < kStreamBatch; ++j)
        if (b + j < steps) one(j);
    }
  };
  stage(0);
  for (int v = 0; v < mine; v += 2 * kStreamBatch) {
    fetch(v + kStreamBatch, a[1]);
    if (v > 0 && v % P == 0) {
      __syncthreads();
      stage(v / P * kStreamChunk);
    }
    use(v, a[0]);
    fetch(v + 2 * kStreamBatch, a[0]);
    use(v + kStreamBatch, a[1]);
  }
  if constexpr (KS > 1) {
    red[wave][0][lane] = acc[0];
    red[wave][1][lane] = acc[1];
    __syncthreads();
    if (kq != 0 || (int)blockIdx.x * U + wave / KS >= units) return;
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int q = 1; q < KS; ++q) acc[i] += red[wave + q][i][lane];
  }
  const int slot = s0 + c;
  if (slot >= s1) return;
  float v[4];
  const float f = UP ? slot_weight_of(p, slot) : 1.f;
  if constexpr (GATED) {
    const MoeActivation act(p, e);
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = act(acc[0][r] * f, acc[1][r] * f);
    store4<BF16>((uint16_t*)p.out + (int64_t)slot * p.ff_max + 16 * u + 4 * g, v);
  } else {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int r = 0; r < 4; ++r) v[r] = UP ? relu_squared_of(acc[i][r] * f) : acc[i][r];
      store4<BF16>((uint16_t*)p.out + (int64_t)slot * (UP ? p.ff_max : p.width) + 32 * u + 16 * i + 4 * g, v);
    }
  }
}

// Of an expert's two to four tiles of 16 slots those that run at the same time share little by way of the L2 (they are on several
// XCDs), and past the caches is faster as long as other experts' weights are most of what is read: 2 of 8 experts of 1408 and a shared
// one of 2816, 2048 wide, up, us by way of the L2 and past it: 32 rows 38.2, 32.0, 64 rows 39.5, 37.8; 6 of 64, down, 64 rows 76.4,
// 70.2.  Not going up where the launch is experts that most rows take and as large as needs no KS: 64 rows that all take the same 2 of
// 16 experts of 2816, 4096 wide, 50, 68, the same 8 163, 207; down 27.7, 24.2 and 73, 84, with a shared expert 54, 51.  There the
// tiles are full: 14 slots of 16 and more (12.8 in the second case above, 16 in these).
template <int PRODUCT, int KS>
__global__ __launch_bounds__(256, 2) void moe_stream_kernel(const MoeParams p) {
  extern __shared__ __attribute__((aligned(16))) char sx[];  // [k-steps of a chunk][4][16][8]
  __shared__ e_f32x4_t red[KS > 1 ? 4 : 1][2][64];
  // the last expert's tiles first: it may be larger than the others, and its work is not to be what is left at the end
  const int all = p.tiles[4 * p.max_tiles + 1], tile = all - 1 - (int)blockIdx.y;
  if (tile < 0) return;
  const int e = p.tiles[4 * tile];
  if (e < 0 || e >= p.experts) return;
  const int s0 = p.tiles[4 * tile + 1], s1 = min(min(p.offsets[e + 1], s0 + 16), p.slots);
  if (s0 >= s1) return;
  if constexpr (PRODUCT != kMoeDown && KS == 1)
    if (p.tiles[4 * tile + 3] >= 3 && p.slots >= 14 * all) return stream_product<PRODUCT, KS, false>(p, e, s0, s1, sx, red);
  stream_product<PRODUCT, KS, true>(p, e, s0, s1, sx, red);
}

// A workgroup's unit (moe_turns.h).  Units of an expert are up to 1024 of its slots side by side, W block after W block, so that an
// XCD's L2 serves a W block to all of them and their rows to the next blocks.
template <int PRODUCT, int TILE, int TILEW>
__device__ __forceinline__ TileWork tile_work(const MoeParams& p, const int blocks_first, const int blocks_last) {
  constexpr bool UP = PRODUCT != kMoeDown, GATED = PRODUCT == kMoeGated;
  constexpr int kSide = 1024 / TILE;
  TileWork t{};
  const int tiles_first = p.tiles[4 * p.max_tiles], tiles_last = p.tiles[4 * p.max_tiles + 1] - tiles_first;
  const TurnUnit u = turn_unit(tiles_first * blocks_first, tiles_last * blocks_last, blockIdx.x & 7, blockIdx.x >> 3);
  if (!u.any) return t;
  const int blocks = u.last ? blocks_last : blocks_first;
  int unit = u.unit + (u.last ? tiles_first * blocks : 0), tile = unit / blocks;
  t.e = p.tiles[4 * tile];
  const int tile0 = p.tiles[4 * tile + 2], count = p.tiles[4 * tile + 3];
  if (t.e < 0 || t.e >= p.experts || count <= 0) return t;
  unit -= tile0 * blocks;  // of this expert's
  const int group = unit / (kSide * blocks), side = min(kSide, count - group * kSide);
  unit -= group * kSide * blocks;
  t.block = unit / side;
  tile = tile0 + group * kSide + unit - t.block * side;
  t.s0 = p.tiles[4 * tile + 1];
  const int end = tile + 1 < min(tile0 + count, p.max_tiles) ? p.tiles[4 * tile + 5] : p.offsets[t.e + 1];
  t.s1 = min(min(end, t.s0 + TILE), p.slots);
  const int ff = p.ff[t.e];
  t.steps = t.all = (UP ? p.width : ff) >> 5;
  t.ntiles = GATED ? ff >> 3 : (UP ? ff : p.width) >> 4;
  t.any = t.block * TILEW < t.ntiles && t.s0 < t.s1;
  t.once = count == 1;
  return t;
}

template <int PRODUCT, bool ONCE, int NT, int MT>
__device__ __forceinline__ void tile_product(const MoeParams& p, const TileWork& t, char (*ring)[kStageBytes]) {
  constexpr bool UP = PRODUCT != kMoeDown, GATED = PRODUCT == kMoeGated;
  e_f32x4_t acc[NT][MT];
  tile_sums<ONCE>(acc, (const uint16_t*)p.x, UP ? p.width : p.ff_max, (const uint16_t*)p.w + p.w_offset[t.e], t, ring,
                  [&](int slot) { return UP ? min(max(p.token[slot], 0), p.rows - 1) : slot; }, [](int tile) { return tile; });
  [[maybe_unused]] const MoeActivation act(p, GATED ? t.e : -1);
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  tile_store<GATED>((uint16_t*)p.out, UP ? p.ff_max : p.width, acc, ring[0] + wave * 2048, (t.block * 4 + wave) * NT, t.ntiles, t.s0,
                    t.s1, [&](int slot) { return UP ? slot_weight_of(p, slot) : 1.f; },
                    [&](float f, int, const e_f32x4_t& a, const e_f32x4_t& b, float (&v)[4]) {
#pragma unroll
                      for (int r = 0; r < 4; ++r) {
                        if constexpr (GATED) v[r] = act(a[r] * f, b[r] * f);
                        else v[r] = UP ? relu_squared_of(a[r] * f) : a[r];
                      }
                    });
}

// EVERY: a body per height in groups of 16 slots, from four on, for launches that power bounds, where products with slots that are not there cost as
// much as others (takes_every_height, moe_turns.h); else bodies of 4, 6 and 8.
template <int PRODUCT, int NT, bool EVERY>
__global__ __launch_bounds__(256, 2) void moe_tile_kernel(const MoeParams p, const int blocks_first, const int blocks_last) {
  __shared__ __attribute__((aligned(16))) char ring[tile_steps(NT) / 2][kStageBytes];
  const TileWork t = tile_work<PRODUCT, kMoeTile, 4 * NT>(p, blocks_first, blocks_last);
  if (!t.any) return;
  const int groups = (t.s1 - t.s0 + 15) >> 4;
  auto go = [&](auto once) __attribute__((always_inline)) {
    constexpr bool O = decltype(once)::value;
    if (groups <= 4) tile_product<PRODUCT, O, NT, 4>(p, t, ring);
    else if (EVERY && groups == 5) tile_product<PRODUCT, O, NT, EVERY ? 5 : 6>(p, t, ring);
    else if (groups <= 6) tile_product<PRODUCT, O, NT, 6>(p, t, ring);
    else if (EVERY && groups == 7) tile_product<PRODUCT, O, NT, EVERY ? 7 : 8>(p, t, ring);
    else tile_product<PRODUCT, O, NT, 8>(p, t, ring);
  };
  if (t.once) go(std::true_type{});
  else go(std::false_type{});
}

// The router's logits on packed weights (experts and the shared gate, up to a multiple of 16 rows): 16 rows of h and a share
// of the k-steps a workgroup; its 8 waves take every eighth step of eight tiles of weights and meet in LDS in wave order.
// z [rows 16 at a time][ld] in LDS, without the bias.
constexpr int kRouteTiles = 8, kRouteBatch = 4;  // tiles and k-steps in flight
constexpr int kRouteShares = 16;              // most shares of the k-steps
constexpr int kRouteLds = 8 * kRouteTiles * 1024;

__device__ __forceinline__ void route_logits(float* z, int ld, e_f32x4_t* red, const uint16_t* h, const uint16_t* w, int row0,
                                             int rows, int width, int ntiles, int step0, int step1) {
  constexpr int TG = kRouteTiles, B = kRouteBatch;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15, steps = width >> 5;
  const uint16_t* x = h + (int64_t)min(row0 + c, rows - 1) * width + 8 * g;
  for (int t0 = 0; t0 < ntiles; t0 += TG) {
    e_f32x4_t acc[TG];
#pragma unroll
    for (int i = 0; i < TG; ++i) acc[i] = e_f32x4_t{0.f, 0.f, 0.f, 0.f};
    for (int k0 = step0 + wave; k0 < step1; k0 += 8 * B) {
      e_u32x4_t xv[B], wv[B][TG];
#pragma unroll
      for (int j = 0; j < B; ++j) {
        const int k = min(k0 + 8 * j, step1 - 1);
        xv[j] = k0 + 8 * j < step1 ? *reinterpret_cast<const e_u32x4_t*>(x + 32 * k) : e_u32x4_t{0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < TG; ++i)
          if (t0 + i < ntiles) wv[j][i] = *reinterpret_cast<const e_u32x4_t*>(w + ((int64_t)(t0 + i) * steps + k) * 512 + lane * 8);
      }
#pragma unroll
      for (int i = 0; i < TG; ++i)
        if (t0 + i < ntiles) {
#pragma unroll
          for (int j = 0; j < B; ++j) acc[i] = moe_mfma(wv[j][i], xv[j], acc[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < TG; ++i) red[(wave * TG + i) * 64 + lane] = acc[i];
    __syncthreads();
    if (t0 + wave < ntiles) {  // wave i sums tile i
      e_f32x4_t s = red[threadIdx.x];
#pragma unroll
      for (int v = 1; v < 8; ++v) s += red[v * TG * 64 + threadIdx.x];
#pragma unroll
      for (int r = 0; r < 4; ++r) z[c * ld + (t0 + wave) * 16 + 4 * g + r] = s[r];
    }
    __syncthreads();
  }
}

// many rows: logits and choice in one launch, a wave chooses for two rows.  What one step leaves to the next stays in LDS (by way of
// memory, every step of the chain is two more round trips).  us with counted places and now: 300 rows 11.4, 8.4; 1943 17.6, 13.2;
// 8192 41, 33.4.
__global__ __launch_bounds__(512) void moe_route_mfma_kernel(int32_t* ids, float* __restrict__ weights,
                                                             const uint16_t* __restrict__ h, const uint16_t* __restrict__ w,
                                                             const float* __restrict__ bias, const MoeRouting r,
                                                             const int rows, const int width, const int keep,
                                                             const MoeGroups groups) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* z = reinterpret_cast<float*>(smem + kRouteLds);
  const int ntiles = (r.logits() + 15) >> 4, ld = ntiles * 16 + 1, row0 = blockIdx.x * 16, n = r.per_row();
  int* kept = reinterpret_cast<int*>(z + 16 * ld);
  route_logits(z, ld, reinterpret_cast<e_f32x4_t*>(smem), h, w, row0, rows, width, ntiles, 0, width >> 5);
  const int lane = threadIdx.x & 63;
  for (int i = threadIdx.x >> 6; i < 16 && row0 + i < rows; i += 8) {
    if (bias != nullptr)
      for (int e = lane; e < r.experts; e += 64) z[i * ld + e] += bias[e];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wave's own next reads see it)
    choose_experts(z + i * ld, r, ids + (int64_t)(row0 + i) * n, weights + (int64_t)(row0 + i) * n, kept + i * n, keep);
  }
  __syncthreads();  // (the logits' partial sums make room for the counts)
  auto count = [&](const int* of) __attribute__((always_inline)) {
    moe_count_assignments(of, row0, min(16, rows - row0), n, r.all(), r.shared, reinterpret_cast<int*>(smem), groups);
  };
  if (keep) count(kept);
  else count(ids + (int64_t)row0 * n);
}

__global__ __launch_bounds__(256) void moe_zero_kernel(int32_t* __restrict__ p, const int n) {
  for (int i = threadIdx.x; i < n; i += 256) p[i] = 0;
}

// few rows: the k-steps are dealt to workgroups as well (grid.y), whose logits leave as part [share][16-row tiles][16][ld]
__global__ __launch_bounds__(512) void moe_logits_kernel(float* __restrict__ part, const uint16_t* __restrict__ h,
                                                         const uint16_t* __restrict__ w, const int ntiles, const int rows,
                                                         const int width, const int per) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  float* z = reinterpret_cast<float*>(smem + kRouteLds);
  const int ld = ntiles * 16, step0 = blockIdx.y * per, step1 = min(step0 + per, width >> 5);
  route_logits(z, ld, reinterpret_cast<e_f32x4_t*>(smem), h, w, blockIdx.x * 16, rows, width, ntiles, step0, step1);
  float* out = part + ((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * 16 * ld;
  for (int i = threadIdx.x; i < 16 * ld; i += 512) out[i] = z[i];
}

// ... and one workgroup adds them, chooses (a wave per row) and groups the assignments, `batch` rows at a time.  A thread asks for all
// shares of its logits at once, up to S of them (further shares stand for the last one: a condition would be a branch, and a wait
// before the next load); choices and ranks stay in LDS.  One CU does it all, so that round trips to memory and the vector
// instructions of a choice bound it, and the size of the code, which comes from memory as well.  Both launches, 6 of 64 experts, 32 / 64
// rows, us: widths of up to 4 shares (2048) 12.3 / 15.3, of up to 16 (4096) 13.8 / 18.5, where a wave asked for its own row's shares one
// row ahead 15.4 / 21.2 and 17.5 / 25.0.
template <int S>
__global__ __launch_bounds__(1024) void moe_choose_group_kernel(int32_t* ids, float* weights, const float* __restrict__ part,
                                                                const float* __restrict__ bias, const int shares,
                                                                const int row_tiles, const int ld, const MoeRouting r,
                                                                const int rows, const int batch, const int keep,
                                                                const MoeGroups groups) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int n = r.per_row();
  float* z = reinterpret_cast<float*>(smem);  // [batch][ld]
  int* kept = reinterpret_cast<int*>(smem + batch * ld * 4);
  const int64_t share = (int64_t)row_tiles * 16 * ld;
  constexpr int U = 16 / S < 2 ? 2 : 16 / S;  // logits of a thread
  for (int row0 = 0; row0 < rows; row0 += batch) {
    const int here = min(batch, rows - row0), count = here * ld;
    const float* from = part + (int64_t)row0 * ld;
    if (row0 > 0) __syncthreads();
    for (int i0 = threadIdx.x; i0 < count; i0 += 1024 * U) {
      float t[U][S], v[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int i = min(i0 + 1024 * u, count - 1), e = i % ld;
#pragma unroll
        for (int s = 0; s < S; ++s) t[u][s] = from[min(s, shares - 1) * share + i];
        v[u] = bias != nullptr ? bias[min(e, r.experts - 1)] : 0.f;
        if (e >= r.experts) v[u] = 0.f;
      }
#pragma unroll
      for (int u = 0; u < U; ++u) {
#pragma unroll
        for (int s = 0; s < S; ++s) v[u] += s < shares ? t[u][s] : 0.f;
        if (i0 + 1024 * u < count) z[i0 + 1024 * u] = v[u];
      }
    }
    __syncthreads();
    for (int i = threadIdx.x >> 6; i < here; i += 16) {
      const int row = row0 + i;
      choose_experts(z + i * ld, r, ids + (int64_t)row * n, weights + (int64_t)row * n, kept + row * n, keep);
    }
  }
  __syncthreads();
  if (keep) group_assignments(kept, kept + rows * n, rows * n, n, r.all(), r.shared, groups);
  else group_assignments(ids, groups.slot, rows * n, n, r.all(), r.shared, groups);
}

static int route_shares(int width) {
  const int steps = width / 32;
  return steps < 16 ? 1 : steps / 16 > kRouteShares ? kRouteShares : steps / 16;  // (at least two k-steps a wave)
}

int64_t moe_route_mfma_workspace(const MoeRouting& r, int rows, int width) {
  if (rows > kMoeFewRows) return (int64_t)r.all() * 4;  // (the experts' counts)
  return (int64_t)route_shares(width) * ((rows + 15) / 16) * 16 * ((r.logits() + 15) / 16 * 16) * 4;
}

int launch_moe_route_mfma(int32_t* ids, float* weights, const void* h, const void* w, const float* bias, const MoeRouting& r,
                          int rows, int width, const MoeGroups& groups, float* workspace, hipStream_t s) {
  const int ntiles = (r.logits() + 15) / 16, row_tiles = (rows + 15) / 16;
  if (rows <= kMoeFewRows) {
    const int shares = route_shares(width), per = (width / 32 + shares - 1) / shares, ld = ntiles * 16;
    const int lds = kRouteLds + 16 * ld * 4, numbers = 2 * rows * r.per_row() * 4;
    const int keep = numbers <= 32 * 1024;  // (many experts a row: by way of memory)
    const int batch = std::min(std::max(1, 64 * 1024 / (ld * 4) / 16), row_tiles) * 16;
    const int lds_choose = batch * ld * 4 + (keep ? numbers : 0);
    (void)hipFuncSetAttribute((const void*)moe_logits_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    hipLaunchKernelGGL(moe_logits_kernel, dim3(row_tiles, shares), dim3(512), lds, s, workspace, (const uint16_t*)h,
                       (const uint16_t*)w, ntiles, rows, width, per);
    LV_LAUNCH_CHECK();
    auto choose = [&](auto most) {
      constexpr int S = decltype(most)::value;
      (void)hipFuncSetAttribute((const void*)moe_choose_group_kernel<S>, hipFuncAttributeMaxDynamicSharedMemorySize, lds_choose);
      hipLaunchKernelGGL(moe_choose_group_kernel<S>, dim3(1), dim3(1024), lds_choose, s, ids, weights, workspace, bias, shares,
                         row_tiles, ld, r, rows, batch, keep, groups);
    };
    if (shares <= 4) choose(std::integral_constant<int, 4>{});
    else choose(std::integral_constant<int, kRouteShares>{});
    LV_LAUNCH_CHECK();
    return 0;
  }
  const int keep = r.per_row() <= 256, lds = kRouteLds + 16 * (ntiles * 16 + 1) * 4 + (keep ? 16 * r.per_row() * 4 : 0);
  (void)hipFuncSetAttribute((const void*)moe_route_mfma_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  hipLaunchKernelGGL(moe_zero_kernel, dim3(1), dim3(256), 0, s, groups.count, r.all());
  LV_LAUNCH_CHECK();
  hipLaunchKernelGGL(moe_route_mfma_kernel, dim3(row_tiles), dim3(512), lds, s, ids, weights, (const uint16_t*)h,
                     (const uint16_t*)w, bias, r, rows, width, keep, groups);
  LV_LAUNCH_CHECK();
  return launch_moe_group(ids, rows * r.per_row(), r.per_row(), r.all(), r.shared, true, groups, s);
}

bool moe_takes_mfma(int width, int dtype) { return dtype == LVLLM_BF16 && width % 32 == 0; }

template <int PRODUCT>
static void go(const MoeParams& p, hipStream_t s) {
  constexpr bool UP = PRODUCT != kMoeDown, GATED = PRODUCT == kMoeGated;
  if (p.rows <= kMoeFewRows) {
    const int steps = (UP ? p.width : p.ff_max) / 32;  // of the largest expert
    const int units = GATED ? p.ff_max / 16 : (UP ? p.ff_max : p.width) / 32;
    const int smem = (steps < kStreamChunk ? steps : kStreamChunk) * 1024;
    // workgroups with work, were every wave to take whole units
    const int64_t wgs = (int64_t)p.max_tiles * (((GATED ? p.ff_first / 16 : UP ? p.ff_first / 32 : units) + 3) / 4);
    const unsigned t = p.max_tiles;
    if (wgs <= 256) hipLaunchKernelGGL((moe_stream_kernel<PRODUCT, 4>), dim3(units, t), dim3(256), smem, s, p);
    else if (wgs <= 512) hipLaunchKernelGGL((moe_stream_kernel<PRODUCT, 2>), dim3((units + 1) / 2, t), dim3(256), smem, s, p);
    else hipLaunchKernelGGL((moe_stream_kernel<PRODUCT, 1>), dim3((units + 3) / 4, t), dim3(256), smem, s, p);
  } else {
    const int tile = moe_tile(true, p.rows);
    // more tiles than there are of 64 slots: they may be of 16 (a router that is not packed), which the body takes as well
    const bool small = p.max_tiles >= p.slots || p.max_tiles > p.slots / kMoeCountedTile + p.experts;
    const int least = small ? kMoeSmallTile : tile;
    const int64_t tiles = small ? p.max_tiles : std::min<int64_t>(p.max_tiles, p.slots / tile + p.experts);
    const int64_t last_tiles = (p.rows + least - 1) / least;  // a token takes an expert once
    auto blocks = [&](int nt, int ff) { return ((GATED ? ff / 8 : (UP ? ff : p.width) / 16) + 4 * nt - 1) / (4 * nt); };
    const BlockCounts whole{blocks(4, p.ff_first), blocks(4, p.ff_last)}, half{blocks(2, p.ff_first), blocks(2, p.ff_last)};
    auto launch = [&](auto nt, auto every, const BlockCounts& b) {
      const unsigned grid = (unsigned)unit_workgroups(tiles * b.first, last_tiles * b.last);
      hipLaunchKernelGGL((moe_tile_kernel<PRODUCT, decltype(nt)::value, decltype(every)::value>), dim3(grid), dim3(256), 0, s, p, b.first, b.last);
    };
    if (takes_half_blocks(p.rows, p.slots, p.experts, least, whole, half, UP, p.ff_last > p.ff_first))
      launch(std::integral_constant<int, 2>{}, std::false_type{}, half);
    else if (takes_every_height(p.rows, p.slots, p.experts, least, whole))
      launch(std::integral_constant<int, 4>{}, std::true_type{}, whole);
    else
      launch(std::integral_constant<int, 4>{}, std::false_type{}, whole);
  }
}

int launch_moe_mfma(const MoeParams& p, int product, hipStream_t s) {
  LV_CHECK(p.experts <= 65535 && p.ff_first > 0 && p.ff_last > 0 && p.ff_first <= p.ff_max && p.ff_last <= p.ff_max,
           "sizes of the experts");
  if (product == kMoeGated) go<kMoeGated>(p, s);
  else if (product == kMoePlain) go<kMoePlain>(p, s);
  else go<kMoeDown>(p, s);
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm
