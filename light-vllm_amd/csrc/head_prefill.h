// The chunk body of head_attention.h: causal attention of prompt portions over the paged cache on 32x32x16 bf16 MFMAs.
//
// A workgroup is 4 waves = 128 columns, a column being a (query token, head of the GQA group, map) triple; the waves share one
// stream of 64-key tiles, copied straight to LDS: three stages where two workgroups a CU have room for them, else two, one
// barrier per tile (with three in front of the last products of the tile before).  A portion's last columns walk all keys one tile after the other, and that walk is how long the launch
// takes: pages are looked up 16 tiles at a time, and copies are a tile ahead of their use.
// With two maps, waves 0 and 1 take the first one, waves 2 and 3 the second one of the same 64 (token, head) pairs: each reads
// its half of the keys, and the two results meet in LDS at the end.
//   * S^T = K Q^T: a lane holds 32 keys of ONE column, so the column's maximum is in-lane plus one exchange of halves;
//   * the cache layouts are the operand layouts: a K fragment is a 16-byte chunk per lane of [kpad / 8][16][8], a V^T
//     fragment 8 consecutive tokens of a [vpad][16] row.  K goes to LDS verbatim; V's chunks are permuted on the way so
//     that a fragment read is 32 consecutive chunks;
//   * probabilities never move between lanes: MFMA row i of S^T holds a permuted key (groups of four 1 and 2 of every 16
//     trade places), which makes a lane's accumulators the consecutive keys that P V wants as its B operand;
//   * accumulators are rescaled only when a column's maximum grew;
//   * with two workgroups a CU the vector instructions of the softmax bound a tile (half of them exponentials), so that the maximum
//     takes three scores at a time.  The scale stays a product of its own, rounded ahead of the subtraction (6 to 10 % of such a
//     launch): fused with it, other roundings moved tokens of a mixture behind the attention to other experts;
//   * tiles of kept first keys come ahead of the window's.
// The longest walk is one wave a SIMD for much of a launch, so that what a tile's chain waits for counts as much as what it issues:
// fragments are read eight ahead of their MFMAs, the first of V in front of the softmax; the maximum is four chains and one exchange
// of halves in registers; pages become addresses once in 16 tiles, in the lanes, and a copy's address is scalar; a masked tile's
// comparisons are taken four at a time (all at once, their results were kept in lanes: 64 writes and as many reads a tile).
// With three stages a tile's first fragments of K are read beside the last products of the one before.
// us before these and now, same bits: one prompt of 4096, 16 heads over 4, 128 + 64, 104, 92 (95 with K's fragments read behind the barrier);
// of 1000 29.4, 25.2; of 2000, 128 + 128, 59.5, 53.4; of 300 18.8, 14.4; two maps of 64 + 128, 2000 tokens 65, 61; 4 prompts of 2048, 16
// heads, 192 + 128 (two stages) 140, 127; 3 of 777 35, 35.  Heads of up to 64 + 64 keep three workgroups a CU (64 + 32: four) by half as many
// fragments of K ahead; 32 heads over 8 of 64 + 64, before, with two workgroups, now: 2300 tokens, a window of 256, 22.0, 23.6, 19.5; 3100, of
// 1500, 54.9, 60.2, 51.1; 4096 101, 109, 97.
#pragma once
#include <float.h>

#include "head_attention.h"

namespace lvllm {

__device__ __forceinline__ h_f32x16_t mfma32(h_u32x4_t a, h_u32x4_t b, h_f32x16_t c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(h_bf16x8_t, a), __builtin_bit_cast(h_bf16x8_t, b), c,
                                                 0, 0, 0);
}

// 16 bytes a lane, 1 KiB a wave, from lane offsets `at` and `skip` into a block's head slice.  (Addresses of a descriptor are the scalar
// unit's work, and not 64-bit additions of the lanes.)
__device__ __forceinline__ void to_lds(const uint16_t* slice, int bytes, int at, int skip, char* dst) {
#if defined(__HIP_DEVICE_COMPILE__)
  __builtin_amdgcn_raw_ptr_buffer_load_lds(__builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(slice), 0, bytes, 0x00020000),
                                           (__attribute__((address_space(3))) void*)dst, 16, at, skip, 0, 0);
#endif
}
// The largest of three; fmaxf takes three instructions of what might be a signalling NaN.  The compiler does not look into this
// one: where b and c are results of MFMAs, `a` has to come from an instruction behind the same ones, which has waited for them.
__device__ __forceinline__ float max3(float a, float b, float c) {
  float m;
  asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(a), "v"(b), "v"(c));
  return m;
}

constexpr int prefill_stages(int nk, int nv) { return 3 * 4 * (nk + nv) <= 80 ? 3 : 2; }
// Workgroups a CU that LDS has room for, and registers with it.
constexpr int prefill_workgroups(int nk, int nv) { return nk + nv <= 3 ? 4 : nk + nv <= 4 ? 3 : nk + nv <= 10 ? 2 : 1; }

template <int NK, int NV, int MAPS>
__global__ __launch_bounds__(256, prefill_workgroups(NK, NV)) void head_prefill_kernel(const HeadAttnParams p) {
  constexpr int KP = 32 * NK, VP = 32 * NV, KS = 2 * NK / MAPS;  // KS: k-steps of a column
  constexpr int kPrefillCols = 128 / MAPS;                       // (token, head) pairs of a workgroup
  constexpr int kKBlock = KP * 16 * 2, kVBlock = VP * 16 * 2;  // bytes of a block's head slice
  constexpr int kImageK = 4 * kKBlock, kStage = kImageK + 4 * kVBlock, S = prefill_stages(NK, NV);
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lc = lane & 31, hi = lane >> 5;
  const int map = MAPS == 2 ? wave >> 1 : 0, cwave = MAPS == 2 ? wave & 1 : wave;
  const int kvh = blockIdx.x, seq = blockIdx.z;
  // The end of the chunk, which sees the most keys, first.  Where all workgroups run at once, two a CU, those that come second on
  // their CUs (behind p.fold tiles) come in the other order, the shortest walk beside the longest: one prompt of 4096, 16 heads over
  // 4, 128 + 64, 111 us without, 105 with (as the tiles were then).
  const int tile_q = (int)blockIdx.y < p.fold ? gridDim.y - 1 - blockIdx.y : blockIdx.y - p.fold;
  const int G = p.heads / p.kv_heads;
  const int qbeg = p.query_start_loc[seq], qlen = p.query_start_loc[seq + 1] - qbeg;
  const int ncols = qlen * G;
  if (qlen <= 0 || qlen < p.min_query_len || takes_decode_body(qlen, G * MAPS) || tile_q * kPrefillCols >= ncols) return;
  const int ctx = p.seq_lens[seq] - qlen;
  if (ctx < 0) return;
  const int col0 = tile_q * kPrefillCols + cwave * 32;
  const int col = min(col0 + lc, ncols - 1);
  const bool col_ok = col0 + lc < ncols;
  const int tok = col / G, head = kvh * G + (col - tok * G);
  const int64_t row = qbeg + tok;
  const int pos = ctx + tok, low = first_seen(p, pos);  // the last and the first key this lane's column sees
  const int wg_last = ctx + (min(tile_q * kPrefillCols + kPrefillCols, ncols) - 1) / G;
  const bool wave_ok = col0 < ncols;
  const int wave_first = ctx + min(col0, ncols - 1) / G, wave_last = ctx + min(col0 + 31, ncols - 1) / G;
  const int wave_low = first_seen(p, wave_first), wave_all = first_seen(p, wave_last);
  const int tile0 = first_seen(p, ctx + tile_q * kPrefillCols / G) / 64;
  const int kept = min((p.keep_first + 63) / 64, tile0);  // tiles of kept keys ahead of the window's
  const int ntiles = wg_last / 64 + 1 - tile0 + kept;
  auto tile_of = [&](int t) { return t < kept ? t : t - kept + tile0; };

  h_u32x4_t qf[KS];
  {
    const uint16_t* q = (const uint16_t*)p.q + (row * p.heads + head) * KP + map * (KP / MAPS) + 8 * hi;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) qf[ks] = *reinterpret_cast<const h_u32x4_t*>(q + 16 * ks);
  }
  const int32_t* table = p.block_tables + (int64_t)seq * p.max_blocks;
  const uint16_t* kc = (const uint16_t*)p.k_cache + (int64_t)kvh * KP * 16;
  const uint16_t* vc = (const uint16_t*)p.v_cache + (int64_t)kvh * VP * 16;
  const int k_lane = lane * 16, v_lane = (lane & 31) * 32 + (lane >> 5) * 16;
  // Where the pages of 16 tiles lie, a lane each (multiplied there: scalar 64-bit products are chains of their own).
  uint64_t k_page = 0, v_page = 0;
  int run = -1;
  auto copy = [&](int stage, int tile) __attribute__((always_inline)) {
    if (tile >> 4 != run) {
      run = tile >> 4;
      const int page = min(max(table[min(run * 64 + lane, p.max_blocks - 1)], 0), p.max_block);
      k_page = (uint64_t)kc + (uint64_t)((int64_t)page * p.k_block_stride) * 2;
      v_page = (uint64_t)vc + (uint64_t)((int64_t)page * p.v_block_stride) * 2;
    }
    char* base = smem + stage * kStage;
    auto of = [&](uint64_t page, int b) __attribute__((always_inline)) {
      const int at = (tile & 15) * 4 + b;
      return (const uint16_t*)((uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)page, at) |
                               (uint64_t)(uint32_t)__builtin_amdgcn_readlane((int)(page >> 32), at) << 32);
    };
#pragma unroll
    for (int j = 0; j < NK; ++j) {
      const int b = (wave + 4 * j) / NK, w = (wave + 4 * j) - b * NK;  // 64-chunk group w of block b
      to_lds(of(k_page, b), kKBlock, k_lane, w * 1024, base + b * kKBlock + w * 1024);
    }
#pragma unroll
    for (int j = 0; j < NV; ++j) {  // of a 32-row group: the first tokens' chunks of all rows, then the second ones'
      const int b = (wave + 4 * j) / NV, w = (wave + 4 * j) - b * NV;
      to_lds(of(v_page, b), kVBlock, v_lane, w * 1024, base + kImageK + b * kVBlock + w * 1024);
    }
  };

  const ScoreScale score(p);
  float m = -1e30f, l = 0.f;
  h_f32x16_t o[NV];
#pragma unroll
  for (int i = 0; i < NV; ++i) o[i] = h_f32x16_t{};
  // MFMA row lc of S^T is key perm(lc) of the 32: groups of four 1 and 2 of every 16 trade places
  const int r16 = lc & 15, grp = r16 >> 2;
  const int key16 = (((grp & 1) << 1 | grp >> 1) << 2) | (r16 & 3);
  const int klds = (lc >> 4) * kKBlock + map * (kKBlock / MAPS) + (hi * 16 + key16) * 16;
  const int vlds = kImageK + lane * 16;  // (hi * 32 + lc) * 16

  constexpr int kCopies = NK + NV;  // of a wave and tile
  // Fragments read ahead of their MFMAs; where more than two workgroups share a CU, which then have the registers of half of K's.
  constexpr int kMostK = prefill_workgroups(NK, NV) > 2 ? 4 : 8, kWinK = 2 * KS < kMostK ? 2 * KS : kMostK, kWinV = 4 * NV < 8 ? 4 * NV : 8;
  __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));  // (the queries are here: what is on its way below are copies)
#pragma unroll
  for (int t = 0; t < S - 1; ++t)
    if (t < ntiles) copy(t, tile_of(t));
  constexpr bool kAhead = S == 3;  // a tile's first fragments of K are read beside the last products of the one before
  h_u32x4_t kw[kWinK];
  auto key = [&](int stage, int i) __attribute__((always_inline)) {  // fragment i: keys of half i % 2, k-step i / 2
    return *reinterpret_cast<const h_u32x4_t*>(smem + stage * kStage + klds + (i & 1) * 2 * kKBlock + (i >> 1) * 512);
  };
  auto read_keys = [&](int stage) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < kWinK; ++i) kw[i] = key(stage, i);
    __builtin_amdgcn_sched_barrier(0);
  };
  // Tile t is in LDS, for every wave, and everyone is done with the stage that is filled next.
  auto publish = [&](int t, int stage) __attribute__((always_inline)) {
    // loads retire in order: with only the youngest tile's copies outstanding, this one's have landed
    if (kAhead && t == 0 && ntiles > 1) __builtin_amdgcn_s_waitcnt(kCopies | (7 << 4) | (15 << 8));
    else __builtin_amdgcn_s_waitcnt(0 | (7 << 4) | (15 << 8));
    asm volatile("s_barrier" ::: "memory");
    read_keys(stage);
    const int next = kAhead ? t + 1 : t + S - 1;
    if ((!kAhead || t > 0) && next < ntiles) copy(stage + 1 == S ? 0 : stage + 1, tile_of(next));
  };
  if (kAhead) publish(0, 0);
  int stage = 0;
  for (int t = 0; t < ntiles; ++t) {
    if (!kAhead) publish(t, stage);
    const int after = stage + 1 == S ? 0 : stage + 1;
    bool published = !kAhead || t + 1 == ntiles;
    const int k0 = tile_of(t) * 64;
    if (wave_ok && k0 <= wave_last && (k0 + 63 >= wave_low || k0 < p.keep_first)) {
      const char* base = smem + stage * kStage;
      h_f32x16_t s[2] = {h_f32x16_t{}, h_f32x16_t{}};
      h_u32x4_t vw[kWinV];
      auto value = [&](int i) __attribute__((always_inline)) {  // ... keys of step i / NV, rows of block i % NV
        return *reinterpret_cast<const h_u32x4_t*>(base + vlds + (i / NV) * kVBlock + (i % NV) * 1024);
      };
#pragma unroll
      for (int i = 0; i < 2 * KS; ++i) {
        s[i & 1] = mfma32(kw[i % kWinK], qf[i >> 1], s[i & 1]);
        if (i + kWinK < 2 * KS) kw[i % kWinK] = key(stage, i + kWinK);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int i = 0; i < kWinV; ++i) vw[i] = value(i);
      __builtin_amdgcn_sched_barrier(0);
      if (score.cap > 0.f) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[h][i] = score.capped(s[h][i]);
      } else {  // (rounded here, ahead of the subtraction, as in the other bodies)
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 16; ++i) s[h][i] *= score.mul;
      }
      if (k0 + 63 > wave_first || k0 < wave_all) {  // the diagonal or the window's edge passes through it for some column
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const int key = k0 + 32 * h + 16 * (i >> 3) + 8 * hi + (i & 7);
            s[h][i] = sees(p, key, pos, low) ? s[h][i] : -INFINITY;
            if (i % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // (else all are compared first, and their masks kept in lanes)
          }
      }
      float part[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) part[i] = fmaxf(s[0][i], s[1][i]);  // (behind this both products' results are there)
#pragma unroll
      for (int i = 4; i < 16; ++i) part[i & 3] = max3(part[i & 3], s[0][i], s[1][i]);
      float mx = fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3]));
      const auto both = halves_apart(mx);
      mx = fmaxf(both.a, both.b);
      if (__any(mx > m)) {
        const float mn = fmaxf(m, mx), corr = exp2f(m - mn);
        m = mn;
        l *= corr;
#pragma unroll
        for (int i = 0; i < NV; ++i) o[i] *= corr;
      }
      float sum = 0.f;
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          s[h][i] = __builtin_amdgcn_exp2f(s[h][i] - m);
          sum += s[h][i];
        }
      l += sum;
      h_u32x4_t pf[4];
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) pf[j][r] = pack_bf16(s[j >> 1][8 * (j & 1) + 2 * r], s[j >> 1][8 * (j & 1) + 2 * r + 1]);
      __builtin_amdgcn_sched_barrier(0);
      if (!published) publish(t + 1, after);
      published = true;
#pragma unroll
      for (int i = 0; i < 4 * NV; ++i) {
        o[i % NV] = mfma32(vw[i % kWinV], pf[i / NV], o[i % NV]);
        if (i + kWinV < 4 * NV) {
          vw[i % kWinV] = value(i + kWinV);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
    if (!published) publish(t + 1, after);
    stage = after;
  }
  if constexpr (MAPS == 2) __syncthreads();  // (the stages make room for the second map's results)
  l += __shfl_xor(l, 32);
  l += sink_term(p, head, m);
  float f = 1.f / l;
  if constexpr (MAPS == 2) {
    constexpr int LD = VP + 4;
    float* other = reinterpret_cast<float*>(smem) + (cwave * 32 + lc) * LD + 4 * hi;  // the second map's result
    if (map == 1) {
#pragma unroll
      for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int r4 = 0; r4 < 4; ++r4)
          *reinterpret_cast<float4*>(other + 32 * i + 8 * r4) =
              float4{o[i][4 * r4] * f, o[i][4 * r4 + 1] * f, o[i][4 * r4 + 2] * f, o[i][4 * r4 + 3] * f};
    }
    __syncthreads();
    if (map == 1) return;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
      for (int r4 = 0; r4 < 4; ++r4) {
        const float4 b = *reinterpret_cast<const float4*>(other + 32 * i + 8 * r4);
        const float bv[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float v = fmaf(-p.map_weight, bv[r], o[i][4 * r4 + r] * f);
          o[i][4 * r4 + r] = v;
          ss = fmaf(v, v, ss);
        }
      }
    ss += __shfl_xor(ss, 32);
    f = 1.f / sqrtf(ss / (float)p.vdim + p.map_eps);
  }
  if (!col_ok) return;
  f *= gate_of<BF16>(p, row, head);
  uint16_t* out = (uint16_t*)p.out + row * p.out_stride + (int64_t)head * p.vdim;
  const bool vec = ((p.vdim | (int)p.out_stride) & 3) == 0 && (((uintptr_t)p.out) & 7) == 0;
#pragma unroll
  for (int i = 0; i < NV; ++i)
#pragma unroll
    for (int r4 = 0; r4 < 4; ++r4) {
      const int d = 32 * i + 8 * r4 + 4 * hi;
      if (vec) {
        if (d < p.vdim) {
          const float v[4] = {o[i][4 * r4] * f, o[i][4 * r4 + 1] * f, o[i][4 * r4 + 2] * f, o[i][4 * r4 + 3] * f};
          store4<BF16>(out + d, v);
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (d + r < p.vdim) out[d + r] = BF16::from_float(o[i][4 * r4 + r] * f);
      }
    }
}

template <int NK, int NV, int MAPS>
static void go_prefill(const HeadAttnParams& p, hipStream_t s) {
  constexpr int smem = prefill_stages(NK, NV) * 4 * (NK + NV) * 32 * 16 * 2, kCols = 128 / MAPS;
  static_assert(MAPS == 1 || 64 * (32 * NV + 4) * 4 <= smem, "the second map's results take the place of the stages");
  if (smem > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)head_prefill_kernel<NK, NV, MAPS>, hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  const int64_t cols = (int64_t)p.max_query_len * (p.heads / p.kv_heads);
  const int64_t tiles = (cols + kCols - 1) / kCols;
  HeadAttnParams folded = p;
  folded.fold = (int)tiles;  // (no second ones)
  // (windows much shorter than the portion make walks alike, which are as well off in order: 16 heads over 2, 64 + 128, 4096 tokens in
  // windows of 512: 32.7 us, 34.3 with the other order behind)
  const bool alike = p.window > 0 && p.chunk <= 0 && (int64_t)p.window * 4 < p.max_query_len;
  if (NK + NV <= 10 && !alike && p.num_seqs == 1 && tiles * p.kv_heads > 256 && tiles * p.kv_heads <= 512 && 256 % p.kv_heads == 0)
    folded.fold = 256 / p.kv_heads;
  hipLaunchKernelGGL((head_prefill_kernel<NK, NV, MAPS>), dim3(p.kv_heads, (unsigned)tiles, p.num_seqs), dim3(256), smem, s, folded);
}

template <int MAPS>
static int prefill_of_size(const HeadAttnParams& p, hipStream_t s) {
  LV_CHECK((int64_t)p.max_query_len * (p.heads / p.kv_heads) <= (int64_t)65535 * (128 / MAPS), "portion too long");
#define LV_HEAD_V(NK_)                               \
  switch (p.vpad / 32) {                             \
    case 1: go_prefill<NK_, 1, MAPS>(p, s); break;   \
    case 2: go_prefill<NK_, 2, MAPS>(p, s); break;   \
    case 3: go_prefill<NK_, 3, MAPS>(p, s); break;   \
    case 4: go_prefill<NK_, 4, MAPS>(p, s); break;   \
    case 6: go_prefill<NK_, 6, MAPS>(p, s); break;   \
    case 8: go_prefill<NK_, 8, MAPS>(p, s); break;   \
    default: LV_CHECK(false, "value size");          \
  }
  switch (p.kpad / 32) {
    case 2: LV_HEAD_V(2); break;
    case 3:
      if constexpr (MAPS == 1) { LV_HEAD_V(3); }
      else { LV_CHECK(false, "key size"); }
      break;
    case 4: LV_HEAD_V(4); break;
    case 6: LV_HEAD_V(6); break;
    case 8: LV_HEAD_V(8); break;
    default: LV_CHECK(false, "key size");
  }
#undef LV_HEAD_V
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm
