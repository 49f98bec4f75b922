// Products X W^T in tiles of 256 W rows x up to 256 X rows on 16x16x32 bf16 MFMAs: four waves that have a CU to themselves and go on
// from tile to tile, a wave 128 W rows x 32 MT X rows.
//
// With many tiles the chip's power bounds it, and the sums' way in and out of the MFMAs is a large part of that: 32x32x16 ones, which move
// twice as many a cycle, reach 1.41 PFLOP/s at 8192^3 where these reach 1.52.
// Both operands go through LDS, 64 of K a stage: X two stages, W three (160 KiB in all), so that a copy has at least half a stage, 1024
// MFMA cycles with MT = 4, to land.  Fragments of the next 32 of K are read while those of these 32 multiply.  Reads and copies that are
// due are dealt evenly over the MFMAs of a stage: one wave a SIMD has nothing else to run while they issue (all copies of a stage in one
// row behind its barrier: 7 to 10 % slower).  The first two stages of the next tile are on their way while this one's results leave.
//
// A row's 128 bytes of a stage are eight 16-byte chunks, which trade places by the row's three low bits: a fragment read takes one chunk of
// each of 16 rows and meets no conflict.
#pragma once
#include "common.h"

namespace lvllm {

typedef __bf16 w_bf16x8_t __attribute__((ext_vector_type(8)));
typedef float w_f32x4_t __attribute__((ext_vector_type(4)));
typedef unsigned int w_u32x4_t __attribute__((ext_vector_type(4)));

constexpr int kWideRows = 256;               // of W, and most of X
constexpr int kWideStage = kWideRows * 128;  // bytes of an operand
constexpr int kWideLds = 5 * kWideStage;     // X: two stages, W: three
constexpr int kWideCus = 256;                // workgroups of a launch: one a CU
constexpr int kWideStoreLds = kWideStage / 4;  // of a wave, for results

// A tile's operands: a base, the bytes from there that may be read, and byte offsets of K = 0 of each of a wave's copies.  X: 2 MT
// copies, whose rows may lie anywhere (an offset a lane).  W: offsets of the wave, and of the lane.
struct WideTile {
  const void *x, *w;
  unsigned x_bytes, w_bytes;
  int x_at[8], w_at[8], w_lane;
  int iters, groups;  // stages; MT
};
// Copy j of a wave holds rows (wave * copies + j) * 8 .., lane l the row l / 8 of them and this chunk of it.
__device__ __forceinline__ int wide_chunk(int lane) { return (lane & 7) ^ (lane >> 3); }

// [16 W rows][16 X rows]: lane l column l % 16, register r row 4 (l / 16) + r
template <int MT>
struct WideSums {
  w_f32x4_t v[8][2 * MT];
};

__device__ __forceinline__ void wide_copy(const void* base, unsigned bytes, char* to, int lane_at, int at) {
#if defined(__HIP_DEVICE_COMPILE__)  // (buffer descriptors are no type of the host's)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), 0, bytes, 0x00020000),
                                           (__attribute__((address_space(3))) void*)to, 16, lane_at, at, 0, 0);
#endif
}
// The lane, by a way that the compiler does not follow: what depends on it is made anew for every tile, and not kept over the walk.
__device__ __forceinline__ int wide_lane() {
  int lane = threadIdx.x & 63;
  asm volatile("" : "+v"(lane));
  return lane;
}
__device__ __forceinline__ int wide_wave() { return __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); }
// Copy j of stage k into LDS stage s.  `any` false: nothing is read, and LDS gets zeros.
__device__ __forceinline__ void wide_copy_x(const WideTile& t, int groups, int j, int s, int k, bool any, char* lds) {
  wide_copy(any ? t.x : nullptr, any ? t.x_bytes : 0, lds + s * kWideStage + (wide_wave() * 2 * groups + j) * 1024, t.x_at[j], k * 128);
}
__device__ __forceinline__ void wide_copy_w(const WideTile& t, int j, int s, int k, bool any, char* lds) {
  wide_copy(any ? t.w : nullptr, any ? t.w_bytes : 0, lds + (2 + s) * kWideStage + (wide_wave() * 8 + j) * 1024, t.w_lane,
            t.w_at[j] + k * 128);
}
// Asks for a tile's first two stages: LDS but for the last of W's stages must be free.
__device__ __forceinline__ void wide_begin(const WideTile& t, char* lds) {
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const int k = min(s, t.iters - 1);
#pragma unroll
    for (int j = 0; j < 8; ++j) wide_copy_w(t, j, s, k, true, lds);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (j < 2 * t.groups) wide_copy_x(t, t.groups, j, s, k, true, lds);
  }
}

// The sums of a tile whose first two stages have landed, for every wave.  Behind it LDS is free.
template <int MT>
__device__ __forceinline__ void wide_walk(WideSums<MT>& sums, const WideTile& t, char* lds) {
  auto& acc = sums.v;
  constexpr int MX = 2 * MT, NM = 8 * MX, kReads = 8 + MX, kCopiesX = 2 * MT;  // MFMAs of 32 of K and the fragments they take
  const int lane = wide_lane(), wave = wide_wave(), c = lane & 15, g = lane >> 4, iters = t.iters;
  char *const lx = lds + (wave & 1) * MT * 4096, *const lw = lds + 2 * kWideStage + (wave >> 1) * 16384;
  const int at[2] = {c * 128 + ((g ^ (c & 7)) * 16), c * 128 + (((4 + g) ^ (c & 7)) * 16)};  // of a fragment of 32 of K in 16 rows
  w_u32x4_t f[2][kReads];  // [32 of K][8 of W, then MX of X]
  auto read = [&](int i, int xs, int ws, int half) __attribute__((always_inline)) {
    f[half][i] = *reinterpret_cast<const w_u32x4_t*>(i < 8 ? lw + ws * kWideStage + at[half] + i * 2048
                                                           : lx + xs * kWideStage + at[half] + (i - 8) * 2048);
  };
  auto multiply = [&](int i, int half) __attribute__((always_inline)) {
    const int m = i >> 3, n = i & 7;
    acc[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(w_bf16x8_t, f[half][n]),
                                                        __builtin_bit_cast(w_bf16x8_t, f[half][8 + m]), acc[n][m], 0, 0, 0);
  };
#pragma unroll
  for (int n = 0; n < 8; ++n)
#pragma unroll
    for (int m = 0; m < MX; ++m) acc[n][m] = w_f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < kReads; ++i) read(i, 0, 0, 0);
  int x0 = 0, w0 = 0, w1 = 1, w2 = 2;  // X's stage, and W's: this one, the next, the one behind
  for (int it = 0; it < iters; ++it) {
    const bool more = it + 2 < iters;
    const int k = more ? it + 2 : 0;
    auto half = [&](int now, int xs, int ws) __attribute__((always_inline)) {
      int reads = 0, copies = 0;
      const int due = now == 0 ? 8 : kCopiesX;
#pragma unroll
      for (int i = 0; i < NM; ++i) {
        multiply(i, now);
#pragma unroll
        for (; reads < ((i + 1) * kReads + NM - 1) / NM; ++reads) read(reads, xs, ws, now ^ 1);
        if (copies < (i + 1) * due / NM) {
          if (now == 0) wide_copy_w(t, copies, w2, k, more, lds);
          else wide_copy_x(t, MT, copies, x0, k, more, lds);
          ++copies;
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    half(0, x0, w0);
    // All of this stage has been read and the next one has landed, for every wave: copies land in order, and the eight of the one behind
    // are the only ones that may be under way.
    asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    half(1, x0 ^ 1, w1);
    x0 ^= 1;
    const int was = w0;
    w0 = w1, w1 = w2, w2 = was;
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// Sums on their way out, by way of the last of W's stages, a quarter each wave: stores are whole lines of rows.  Outputs of a wave: 128
// W rows, or (PAIRS) 64 of 16 W rows and the 16 behind them.  `value` (16 W rows n and the four sums of this lane, those of the rows
// behind them -> v) sees every sum once; X rows and outputs from `rows` and `outs` (a multiple of 8) on are not stored.  Ends with
// everything that was asked for in front of it landed, for every wave.
template <bool PAIRS, int MT, class VALUE>
__device__ __forceinline__ void wide_store(const WideSums<MT>& sums, char* lds, uint16_t* out, const int64_t ld, const int rows,
                                           const int outs, VALUE value) {
  constexpr int kOuts = PAIRS ? 64 : 128, kChunks = kOuts / 8, kStores = 32 * kChunks / 64;  // of 8 outputs; of 32 rows
  const int lane = wide_lane(), c = lane & 15, g = lane >> 4;
  char* const mine = lds + 4 * kWideStage + wide_wave() * kWideStoreLds;
#pragma unroll
  for (int m = 0; m < MT; ++m) {
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int n = 0; n < 8; n += PAIRS ? 2 : 1) {
        float v[4];
        value(n, sums.v[n][2 * m + i], sums.v[PAIRS ? n + 1 : n][2 * m + i], v);
        const int r = i * 16 + c, chunk = (PAIRS ? n : 2 * n) + (g >> 1);
        store4<BF16>(reinterpret_cast<uint16_t*>(mine + r * (kOuts * 2) + ((chunk ^ r) & (kChunks - 1)) * 16 + 8 * (g & 1)), v);
        if (n % 4 == (PAIRS ? 2 : 3)) __builtin_amdgcn_sched_barrier(0);  // (else all of them are begun at once, and registers run out)
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wave's own next reads see it)
    w_u32x4_t line[kStores];
#pragma unroll
    for (int i = 0; i < kStores; ++i) {
      const int r = i * (64 / kChunks) + lane / kChunks, q = lane % kChunks;
      line[i] = *reinterpret_cast<const w_u32x4_t*>(mine + r * (kOuts * 2) + ((q ^ r) & (kChunks - 1)) * 16);
    }
    // (the last stores need not have left)
    if (m == MT - 1) asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
    for (int i = 0; i < kStores; ++i) {
      const int r = m * 32 + i * (64 / kChunks) + lane / kChunks, q = lane % kChunks;
      if (r < rows && q * 8 < outs) *reinterpret_cast<w_u32x4_t*>(out + r * ld + q * 8) = line[i];
    }
  }
  asm volatile("s_barrier" ::: "memory");
}

}  // namespace lvllm
