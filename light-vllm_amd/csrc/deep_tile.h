// Tiles of up to 128 rows x 64 or 128 W rows for launches of few workgroups, a CU each or two: the same sums in the same order as tile_sums
// (moe_tile.h).  There a workgroup's waves are on their own: what one of them waits for, no other covers.  A wave issues in order, 16 cycles
// a MFMA, and a load of 1 KiB keeps the CU's one address unit for as long, so that four waves whose loads stand together wait 64 cycles for each:
// loads and MFMAs took turns (80 rows x 128: 356 cycles a k-step, 160 of MFMAs and 224 of loads).  Here the loads are dealt
// among the MFMAs, and fragments are read a k-step ahead.  us of 64 k-steps, weights in the last cache, a workgroup a CU: 64 rows x 64 9.4, 8.0; 96 x
// 128 14.6, 11.2; 128 x 128 18.3, 13.3; two a CU: 112 x 128 29.5, 27.7, but 64 x 128 37.4, 39.0: a plan of
// products counts with that (prompt_product.h), and half tiles with an activation are dealt where they gain (prompt_linear.h).  From memory,
// 4096 x 4096, 300 rows 25.9 (the library's), 19.8.
#pragma once
#include <type_traits>

#include "moe_tile.h"

namespace lvllm {

// stages of two k-steps under way: as many as leave two workgroups a CU (80 KiB each) and registers for their weights.  Three are slower (2048 x 2048,
// 300 rows from memory 11.3 us, 8.8), four to eight alike
constexpr int deep_stages(int MT) { return MT <= 6 ? 6 : 5; }
constexpr int deep_stage_bytes(int MT) { return 4096 * ((MT + 1) / 2); }
constexpr int deep_lds_bytes(int MT) { return deep_stages(MT) * deep_stage_bytes(MT); }

// t.steps: even.  `ring`: deep_lds_bytes.  tile_of: where in w a W tile lies.  Ends with LDS free, for every wave.
template <int NT, int MT, class TILE>
__device__ __forceinline__ void deep_sums(e_f32x4_t (&acc)[NT][MT], const uint16_t* x_rows, const int64_t ld, const uint16_t* w_tiles,
                                          const TileWork& t, char* ring, TILE tile_of) {
  constexpr int X = deep_stages(MT), S = 2 * X, kCopies = (MT + 1) / 2, kStage = deep_stage_bytes(MT);
  constexpr int kNow = (kCopies + 1) / 2, kLater = kCopies - kNow;  // of a stage's copies: with its first k-step's weights, with its second's
  constexpr int kYounger = NT + (X - 2) * (2 * NT + kCopies);       // loads behind the copies of the next stage
  constexpr int kFirst = kYounger + NT + kNow;
  static_assert(kFirst < 64, "what is outstanding can be counted");
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g = lane >> 4, c = lane & 15, nt0 = (t.block * 4 + wave) * NT, stages = t.steps >> 1;
  // this wave's W tiles, and the rows it copies: lane l moves chunk l % 8, exchanged by the row, of row l / 8 of eight
  const uint16_t *wsrc[NT], *xsrc[kCopies];
#pragma unroll
  for (int n = 0; n < NT; ++n) wsrc[n] = w_tiles + (int64_t)tile_of(min(nt0 + n, t.ntiles - 1)) * t.all * 512 + lane * 8;
#pragma unroll
  for (int i = 0; i < kCopies; ++i)
    xsrc[i] = x_rows + min(t.s0 + (wave * kCopies + i) * 8 + (lane >> 3), t.s1 - 1) * ld + ((lane & 7) ^ (lane >> 3)) * 8;
  const int xoff[2] = {c * 128 + ((g ^ (c & 7)) * 16), c * 128 + (((4 + g) ^ (c & 7)) * 16)};
  e_u32x4_t a[S][NT], x[2][MT];
  // (past the end: the last stage once more)
  auto copy = [&](int stage, int at, int i) __attribute__((always_inline)) {
    to_lds16((const char*)(xsrc[i] + min(stage, stages - 1) * 64), ring + at * kStage + (wave * kCopies + i) * 1024);
    asm volatile("" ::: "memory");  // (in this order: what is outstanding is counted)
  };
  auto fetch = [&](int stage, int at, int n) __attribute__((always_inline)) {  // at: of S
    a[at][n] = *reinterpret_cast<const e_u32x4_t*>(wsrc[n] + (2 * min(stage, stages - 1) + (at & 1)) * 512);
    asm volatile("" ::: "memory");
  };
  auto read = [&](int at, int m) __attribute__((always_inline)) {
    x[at & 1][m] = *reinterpret_cast<const e_u32x4_t*>(ring + (at >> 1) * kStage + xoff[at & 1] + m * 2048);
  };
  // a k-step: the next one's fragments, this one's MFMAs, `loads` loads among them
  auto step = [&](int at, auto loads, auto load) __attribute__((always_inline)) {
    constexpr int kMfmas = NT * MT, kLoads = decltype(loads)::value, kReads = (3 * kMfmas + 3) / 4;  // reads in front: they take 64 cycles and more
#pragma unroll
    for (int i = 0; i < kMfmas; ++i) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (m * kReads / MT == i) read((at + 1) % S, m);
      __builtin_amdgcn_sched_barrier(0);
      acc[i % NT][i / NT] = moe_mfma(a[at][i % NT], x[at & 1][i / NT], acc[i % NT][i / NT]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int l = 0; l < kLoads; ++l)
        if (l * kMfmas / (kLoads > 0 ? kLoads : 1) == i) load(l);
      __builtin_amdgcn_sched_barrier(0);
    }
  };
#pragma unroll
  for (int n = 0; n < NT; ++n)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[n][m] = e_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < X; ++j) {
#pragma unroll
    for (int n = 0; n < NT; ++n) fetch(j, 2 * j, n);
#pragma unroll
    for (int i = 0; i < (j < X - 1 ? kCopies : kNow); ++i) copy(j, j, i);
#pragma unroll
    for (int n = 0; n < (j < X - 1 ? NT : 0); ++n) fetch(j, 2 * j + 1, n);
  }
  __builtin_amdgcn_s_waitcnt((kFirst & 15) | (kFirst >> 4) << 14 | (7 << 4) | (15 << 8));
  asm volatile("s_barrier" ::: "memory");
#pragma unroll
  for (int m = 0; m < MT; ++m) read(0, m);
  int s = 0;
  for (; s + X <= stages; s += X)
#pragma unroll
    for (int j = 0; j < X; ++j) {
      __builtin_amdgcn_s_waitcnt(15 | 3 << 14 | (7 << 4));  // the fragments are here
      __builtin_amdgcn_sched_barrier(0);
      step(2 * j, std::integral_constant<int, kLater + NT>(), [&](int l) __attribute__((always_inline)) {
        if (l < kLater) copy(s + j - 1 + X, (j - 1 + X) % X, kNow + l);
        else fetch(s + j - 1 + X, (2 * j - 1 + S) % S, l - kLater);
      });
      // loads retire in order: with only the younger ones outstanding the next stage has landed, and everyone is done with this one
      __builtin_amdgcn_s_waitcnt((kYounger & 15) | (kYounger >> 4) << 14 | (7 << 4));
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      step(2 * j + 1, std::integral_constant<int, NT + kNow>(), [&](int l) __attribute__((always_inline)) {
        if (l < NT) fetch(s + j + X, 2 * j, l);
        else copy(s + j + X, j, l - NT);
      });
    }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // the rest is here (of stage s + X - 1, which is none of it, a part)
#pragma unroll
  for (int j = 0; j < X - 1; ++j) {
    if (s + j >= stages) break;
    step(2 * j, std::integral_constant<int, 0>(), [](int) {});
    step(2 * j + 1, std::integral_constant<int, 0>(), [](int) {});
  }
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (everyone has read the last stage)
}

}  // namespace lvllm
