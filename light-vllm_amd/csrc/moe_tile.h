// Tiles of up to 128 rows x 64 NT W rows on 16x16x32 bf16 MFMAs over packed weights, two workgroups a CU: the grouped products of prompts
// (moe_mfma.hip) and projections with an activation behind them (tile_linear.hip).
#pragma once
#include "moe.h"

namespace lvllm {

typedef __bf16 e_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float e_f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int e_u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ e_f32x4_t moe_mfma(e_u32x4_t a, e_u32x4_t b, e_f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(e_bf16x8_t, a), __builtin_bit_cast(e_bf16x8_t, b), c, 0, 0,
                                                 0);
}

// Weights past the caches (ONCE) or by way of the L2.  Those that one workgroup reads go past them.  Up + down, us, without and with:
// moe_stream_kernel, 32 rows, 6 of 64 experts of 2816, 268, 238; tiles of 128 slots, 1000 rows, 6 of 64 experts of 1408 and a shared
// one 276, 259, 2 of 32 193, 175.  What several tiles of 128 slots share does not: all tiles so, 1943 rows 376, 516; for several of 16
// see moe_stream_kernel.
template <bool ONCE>
__device__ __forceinline__ e_u32x4_t load_weights(const uint16_t* p) {
  if constexpr (ONCE) return __builtin_nontemporal_load(reinterpret_cast<const e_u32x4_t*>(p));
  else return *reinterpret_cast<const e_u32x4_t*>(p);
}

// W block `block` (4 NT tiles of 16 rows) of slots s0 .. s1 - 1 of expert e
struct TileWork {
  int e, block, s0, s1, steps, ntiles;  // slots s0 .. s1 - 1, k-steps, W tiles of 16 rows of the expert
  int all;  // k-steps that lie side by side in w: more than `steps` where a workgroup takes a share of them
  bool any, once;  // once: the expert's only tile
};
// A wave's results by way of 2 KiB of LDS of its own: W tiles nt0 .. of groups of 16 slots from slot0 on, a group at a time, so that a
// store is a line of a slot's row and not the 8 bytes a lane that the products leave.  PAIRS: one output of two W tiles.  value (slot of
// the group, W tile, this lane's sums of it, of the one behind it -> v): `begin` a group, then its W tiles.
template <bool PAIRS, int NT, int MT, class BEGIN, class VALUE>
__device__ __forceinline__ void tile_store(uint16_t* out, int64_t out_ld, const e_f32x4_t (&acc)[NT][MT], char* lds, int nt0, int ntiles,
                                           int slot0, int s1, BEGIN begin, VALUE value) {
  constexpr int kOuts = NT * (PAIRS ? 8 : 16), kChunks = kOuts / 8;  // of 8 outputs
  const int lane = threadIdx.x & 63, g = lane >> 4, c = lane & 15;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int slot = slot0 + m * 16;
    if (slot >= s1) break;
    const float f = begin(min(slot + c, s1 - 1));
#pragma unroll
    for (int n = 0; n < NT; n += PAIRS ? 2 : 1) {
      float v[4];
      value(f, n, acc[n][m], acc[PAIRS ? n + 1 : n][m], v);
      const int chunk = (PAIRS ? n : 2 * n) + (g >> 1);
      store4<BF16>(reinterpret_cast<uint16_t*>(lds + c * (kOuts * 2) + ((chunk ^ c) & (kChunks - 1)) * 16 + (g & 1) * 8), v);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wave's own next reads see it)
    const int first = nt0 * (PAIRS ? 8 : 16), outs = (ntiles - nt0) * (PAIRS ? 8 : 16);
#pragma unroll
    for (int j = 0; j < (kChunks + 3) / 4; ++j) {
      const int r = j * (64 / kChunks) + lane / kChunks, q = lane % kChunks;
      if (kChunks < 4 && r >= 16) break;
      const e_u32x4_t v = *reinterpret_cast<const e_u32x4_t*>(lds + r * (kOuts * 2) + ((q ^ r) & (kChunks - 1)) * 16);
      if (slot + r < s1 && q * 8 < outs) *reinterpret_cast<e_u32x4_t*>(out + (slot + r) * out_ld + first + q * 8) = v;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (read before it is written again)
  }
}

// 16 bytes a lane to consecutive LDS
__device__ __forceinline__ void to_lds16(const char* from, void* dst) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)from,
                                   (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

// Prompts: 64 NT W rows x up to 128 slots a workgroup, a wave 16 NT x 128, two workgroups a CU, a unit each.  W goes straight to the
// operand registers of the one wave that uses it, slots by way of LDS.
// NT = 4.  With many slots the chip's power bounds it: 1.8 GHz at 55 % of the MFMA cycles.  8192 rows, 6 of 64 experts of 2816, 2048
// wide: 1.08 PFLOP/s going up and 1.10 down, where the library's plain products of these sizes run at 1.33 and 1.45; 256 slots a
// workgroup, both operands through LDS, were no faster.  Between 128 and 400 slots an expert neither memory (4.3 TB/s of weights), the L1, LDS
// nor MFMA (each near 40 %) is at its limit by itself; one workgroup a CU that goes on from unit to unit, with 8 steps of weights on
// their way, was slower (1943 rows, 6 of 64 experts of 1408, up: 237 us; 262 with 8 waves, 322 with 4).
// NT = 2 (takes_half_blocks, moe_turns.h): a step costs less and eight of them, not four, are under way, so that the memory's latency
// bounds a walk no more.
// A slot's eight chunks trade places by the slot's three low bits: a fragment read takes one chunk of each of 16 slots, 128 bytes
// apart.  4 to 8 % of the cycles in which LDS is active are conflicts, those of the results' way out included.
constexpr int kStageBytes = kMoeTile * 128;  // two k-steps of 32: a slot's 128 bytes, 8 slots a copy
constexpr int tile_steps(int NT) { return NT == 4 ? 4 : 8; }  // k-steps of weights in registers; half as many stages of slots
// row_of: where in x (of row length ld) a slot's row lies; tile_of: where in w a W tile lies.  Ends with LDS free, for every wave.
template <bool ONCE, int NT, int MT, class ROW, class TILE>
__device__ __forceinline__ void tile_sums(e_f32x4_t (&acc)[NT][MT], const uint16_t* x_rows, const int64_t ld, const uint16_t* w_tiles,
                                          const TileWork& t, char (*ring)[kStageBytes], ROW row_of, TILE tile_of) {
  constexpr int S = tile_steps(NT), X = S / 2, kCopies = (MT + 1) / 2;  // (MT groups of 16 slots)
  constexpr int kYounger = (X - 2) * kCopies + (X - 1) * 2 * NT;  // loads behind a stage's copies when it is needed
  constexpr int kBehind = (X - 1) * kCopies + (S - 1) * NT;       // ... behind a second k-step's weights
  const int s0 = t.s0, s1 = t.s1, block = t.block, steps = t.steps, ntiles = t.ntiles;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15;
  const int nt0 = (block * 4 + wave) * NT;
  // this wave's W tiles, and the slots it copies: lane l moves chunk l % 8, exchanged by the slot, of slot l / 8 of eight
  const uint16_t *wsrc[NT], *xsrc[kCopies];
  const uint16_t* w = w_tiles + lane * 8;
#pragma unroll
  for (int j = 0; j < NT; ++j) wsrc[j] = w + (int64_t)tile_of(min(nt0 + j, ntiles - 1)) * t.all * 512;
  const int chunk = (lane & 7) ^ (lane >> 3);
#pragma unroll
  for (int j = 0; j < kCopies; ++j) {
    const int slot = min(s0 + (wave * kCopies + j) * 8 + (lane >> 3), s1 - 1);
    xsrc[j] = x_rows + (int64_t)row_of(slot) * ld;
  }
  e_u32x4_t a[S][NT];
  auto copy = [&](int k, int stage) __attribute__((always_inline)) {  // of k-steps k and k + 1 (a missing one: the one before)
    k = min(k, (steps - 1) & ~1);
    const int at = k * 32 + (k + 1 < steps ? chunk : chunk & 3) * 8;
#pragma unroll
    for (int j = 0; j < kCopies; ++j) to_lds16((const char*)(xsrc[j] + at), ring[stage] + (wave * kCopies + j) * 1024);
    asm volatile("" ::: "memory");  // (in this order: what is outstanding is counted)
  };
  auto fetch = [&](int k, int at) __attribute__((always_inline)) {  // (past the end: the last step once more)
    k = min(k, steps - 1);
#pragma unroll
    for (int j = 0; j < NT; ++j) a[at][j] = load_weights<ONCE>(wsrc[j] + k * 512);
    asm volatile("" ::: "memory");
  };
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = e_f32x4_t{0.f, 0.f, 0.f, 0.f};
  const int xoff[2] = {c * 128 + ((g ^ (c & 7)) * 16), c * 128 + (((4 + g) ^ (c & 7)) * 16)};
  auto multiply = [&](int at) __attribute__((always_inline)) {
    constexpr int W = NT == 4 && MT > 5 ? 5 : MT;  // fragments read ahead
    e_u32x4_t x[W];
    auto read = [&](int m) { x[m % W] = *reinterpret_cast<const e_u32x4_t*>(ring[at / 2] + xoff[at & 1] + m * 2048); };
#pragma unroll
    for (int m = 0; m < W; ++m) read(m);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[n][m] = moe_mfma(a[at][n], x[m % W], acc[n][m]);
      if (m + W < MT) read(m + W);
      if (W < MT) __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int j = 0; j < X - 1; ++j) {
    copy(2 * j, j);
    fetch(2 * j, 2 * j);
    fetch(2 * j + 1, 2 * j + 1);
  }
  fetch(S - 2, S - 2);
  int k = 0;
  for (; k + S <= steps; k += S)
#pragma unroll
    for (int j = 0; j < X; ++j) {
      // loads retire in order: with only the younger ones outstanding, this stage's have landed; what was read, too
      __builtin_amdgcn_s_waitcnt((kYounger & 15) | (kYounger >> 4) << 14 | (7 << 4));
      asm volatile("s_barrier" ::: "memory");  // ... for every wave; and everyone is done with the stage that is filled next
      copy(k + 2 * (j + X - 1), (j + X - 1) % X);
      fetch(k + 2 * j + S - 1, (2 * j + S - 1) % S);
      multiply(2 * j);
      fetch(k + 2 * j + S, 2 * j);
      __builtin_amdgcn_s_waitcnt((kBehind & 15) | (kBehind >> 4) << 14 | (7 << 4) | (15 << 8));  // (the compiler would wait for all)
      multiply(2 * j + 1);
    }
  if (k < steps) {  // the rest, but for its last stage, is on its way (a count would not do: loads that nothing uses are not made)
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    if (steps - k == S - 1) copy(k + S - 2, X - 1);
#pragma unroll
    for (int j = 0; j < S - 2; ++j)
      if (k + j < steps) multiply(j);
    if (steps - k == S - 1) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
      multiply(S - 2);
    }
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (no copy to LDS is under way, and everyone has read the last stage)
}

}  // namespace lvllm
