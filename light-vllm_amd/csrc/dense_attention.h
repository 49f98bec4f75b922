// Attention of whole sequences over the caller's row-major [token][KVH][64] rows (slices of a fused qkv projection), causal or not, without
// a pack pass: heads of 64, 16-bit types (lvllm_varlen_attention, where lengths are alike or many: dense_rule.h).
//
// The arithmetic is that of prefill_mfma32.h, sum for sum: S^T = K Q^T and O^T += V^T P^T on 32x32x16 MFMAs, P never moving between lanes,
// sums rescaled where a column's maximum grew by more than 2^6.  What differs is how a wave is kept busy:
//   * with CG = 2 a wave has two groups of 32 columns, which share every fragment of K and V that it reads, and while the MFMAs of one run
//     it issues the other's exponentials: K Q^T of the first; of the second beside the softmax of the first; P V of the first beside the
//     softmax of the second; P V of the second.  An MFMA of a chain never waits for the one in front of it: two chains take turns.  The next
//     tile is published in front of the last of these, and its fragments of K are read beside it;
//   * CG = 1: three workgroups a CU instead of two, for walks so short that their beginnings and ends weigh most;
//   * copies go straight to LDS, a tile ahead, 8 rows of 128 bytes a copy; chunk c of row r sits at r * 128 + 16 * (c ^ f(r)), which makes the
//     row reads of K and the transposed reads of V (ds_read_b64_tr_b16: the hardware transposes 4 keys x 16 columns per 16 lanes)
//     free of conflicts.
// Vector instructions bound a walk: 64 columns take 1390 cycles of them a tile and wave, 512 of them exponentials, where the MFMAs take 1024;
// two waves a SIMD get through a tile each in 4090 cycles, 707 of them waits.  With 8 tiles a walk the way in and out takes as long again.
// 16 heads, bidirectional, us with copies through registers, a group of columns a wave and two waves a SIMD, and now: 32 x 512 tokens 69, 61;
// 128 x 128 41, 37.5; 24 x 400 40.7, 36; 8 x 2048 171, 153; 2 x 1024 22.5, 19; causal: 53.6, 49.3; 42, 41.8; 30.2, 27.2; 105, 93; 22, 19.
#pragma once
#include "prefill_mfma32.h"

namespace lvllm {

constexpr int kDenseKeys = 64, kDenseHead = 64;       // keys of a tile, head size
constexpr int kDenseRow = kDenseHead * 2;             // bytes of a row
constexpr int kDenseImage = kDenseKeys * kDenseRow;   // of a tile's K or V
constexpr int kDenseStage = 2 * kDenseImage;

__device__ __forceinline__ int dense_chunk(int row, int c) { return c ^ ((((row >> 1) & 1) << 2) | ((row >> 2) & 3)); }
__device__ __forceinline__ int dense_at(int row, int c) { return row * kDenseRow + (dense_chunk(row, c) << 4); }

// A wave's copies of one operand: rows 8 wave .. and 32 + 8 wave .. of every tile, lane l chunk dense_chunk(row, l & 7) of row l >> 3.  What lies
// past the sequence's last row is past the descriptor's end and becomes zeros.
struct DenseRows {
  const char* base;
  int64_t bytes, row;
  uint32_t at;
  __device__ __forceinline__ DenseRows(const void* rows, int64_t stride, int64_t readable, int first, int kvh, int n, int lane, int wave) {
    row = stride * 2;
    const int64_t skip = first * row + (int64_t)kvh * kDenseRow;
    base = (const char*)rows + skip;
    bytes = min((int64_t)(n - 1) * row + kDenseRow, readable - skip);
    const int r = wave * 8 + (lane >> 3);
    at = (uint32_t)(r * (int)row + (dense_chunk(r, lane & 7) << 4));
  }
  __device__ __forceinline__ void copy(int tile, char* image, int wave) const {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int64_t skip = (int64_t)(tile * kDenseKeys + 32 * i) * row;
      const __amdgpu_buffer_rsrc_t r =
          __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(base) + skip, 0, (int)max(bytes - skip, (int64_t)0), kSrdFlags);
      __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)(image + (i * 4 + wave) * 1024), 16, at, 0, 0, 0);
    }
#endif
  }
};

template <typename T, int CG>
__global__ __launch_bounds__(256, CG == 2 ? 2 : 3) void dense_attention_kernel(const PrefillParams p) {
  using S = typename T::store_t;
  constexpr bool kAhead = CG == 2;  // a tile's fragments of K are read beside the one before
  constexpr float kLog2e = 1.4426950408889634f, kMasked = -FLT_MAX, kGrow = 6.f, kSumLimit = 32.f * 64.f;
  __shared__ __attribute__((aligned(1024))) char stage0[kDenseStage];  // (two objects: a read of one does not wait for copies to the other)
  __shared__ __attribute__((aligned(1024))) char stage1[kDenseStage];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 31, hi = lane >> 5;
  const int GP = 1 << p.gp_shift;    // heads per query token among 32 columns (group size rounded up)
  const int TQ = 32 >> p.gp_shift;   // query tokens of a group of columns
  const int G = p.num_heads / p.num_kv_heads, HG = (G + 31) >> 5;
  const int kvh = blockIdx.x / HG, hg = blockIdx.x - kvh * HG;
  const int head0 = kvh * G + hg * 32, nh = min(GP, G - hg * 32);
  const int qtile = gridDim.z - 1 - blockIdx.z;  // the longest walks first
  const int qbeg = p.query_start_loc[blockIdx.y], n = p.query_start_loc[blockIdx.y + 1] - qbeg;
  if (qtile * 4 * CG * TQ >= n) return;
  const int t0 = (qtile * 4 + wave) * CG * TQ;  // this wave's first query token
  const int walk = p.causal ? min(n, (qtile + 1) * 4 * CG * TQ) : n;  // keys of the workgroup
  // (a wave's columns are queries of one aligned block of 64 tokens at most: all of them end in the same tile)
  const int mine = t0 >= n ? 0 : p.causal ? min(n, t0 + CG * TQ) : n;
  const int ntiles = (walk + kDenseKeys - 1) / kDenseKeys, my_tiles = (mine + kDenseKeys - 1) / kDenseKeys;
  const int plain = min(my_tiles, (p.causal ? min(t0 + 1, n) : n) / kDenseKeys);  // tiles that every query sees whole

  const DenseRows k(p.k_cache, p.dense_k_stride, p.dense_k_bytes, qbeg, kvh, n, lane, wave);
  const DenseRows v(p.v_cache, p.dense_v_stride, p.dense_v_bytes, qbeg, kvh, n, lane, wave);
  auto copy = [&](int j, char* to) __attribute__((always_inline)) {
    k.copy(j, to, wave);
    v.copy(j, to + kDenseImage, wave);
  };
  copy(0, stage0);
  if (kAhead && ntiles > 1) copy(1, stage1);

  // this lane's columns: query token t0 + c TQ + col / GP, head head0 + col % GP
  const int cq = col >> p.gp_shift, ch = col & (GP - 1);
  u32x4_t qf[CG][4];
  int last[CG];  // last visible key
#pragma unroll
  for (int c = 0; c < CG; ++c) {
    const int t = t0 + c * TQ + cq;
    const bool live = ch < nh && t < n;
    last[c] = live ? (p.causal ? t : n - 1) : -1;
    const S* row = (const S*)p.q + (int64_t)(qbeg + t) * p.q_stride + (int64_t)(head0 + ch) * kDenseHead;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      qf[c][ks] = u32x4_t{0, 0, 0, 0};
      if (live) qf[c][ks] = *reinterpret_cast<const u32x4_t*>(row + 16 * ks + 8 * hi);
    }
  }
  const float kf = p.scale * kLog2e;
  float m_run[CG], l_run[CG];
  f32x16_t acc[CG][2];
#pragma unroll
  for (int c = 0; c < CG; ++c) {
    m_run[c] = -1e30f, l_run[c] = 0.f;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[c][0][r] = acc[c][1][r] = 0.f;
  }

  // K fragment (32 kh + ..., 16 ks ..): MFMA row col holds key krow of the half, so that a lane's sums are the keys 8 hi .. 8 hi + 7 of every
  // 16, as P V takes them.  V^T fragment (32 db .., 16 ks ..): lane 4 q + i of every 16 addresses row q of a block of 4 keys.
  const int krow = (col & ~0xc) | ((col & 4) << 1) | ((col & 8) >> 1);
  const int tr_q = (lane & 15) >> 2, tr_c = 2 * (col >> 4) + ((lane & 3) >> 1), tr_b = 8 * (lane & 1);
  // A fragment's place: the chunk's bits that a k-step or a block of rows sets are not those of f, so that they come in by an exclusive or.
  const int k_at = dense_at(krow, hi), v_at = dense_at(8 * hi + tr_q, tr_c) + tr_b;
  auto kread = [&](const char* lds, int base, int i) __attribute__((always_inline)) -> u32x4_t {
    return *reinterpret_cast<const u32x4_t*>(lds + (base ^ ((i >> 1) << 5)) + (i & 1) * 32 * kDenseRow);
  };
  auto vread = [&](const char* lds, int base, int i) __attribute__((always_inline)) -> u32x4_t {
    typedef __attribute__((address_space(3))) i16x4_t* lds_tr_t;
    const char* at = lds + kDenseImage + (i >> 1) * 16 * kDenseRow;
    const i16x4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + (base ^ ((i & 1) << 6))));
    const i16x4_t up = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_tr_t)(at + (base ^ ((i & 1) << 6) ^ 16) + 4 * kDenseRow));
    const u32x2_t a = __builtin_bit_cast(u32x2_t, lo), b = __builtin_bit_cast(u32x2_t, up);
    return u32x4_t{a.x, a.y, b.x, b.y};
  };
  u32x4_t kw[8];
  auto read_keys = [&](const char* from) __attribute__((always_inline)) {
    int base = k_at;
    asm volatile("" : "+v"(base));  // (addresses made from it are made for every tile, and not kept)
#pragma unroll
    for (int i = 0; i < 8; ++i) kw[i] = kread(from, base, i);
  };
  // the next tile is in LDS, and everyone has left the one before: its stage may take the one behind
  auto publish = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
  auto tile = [&](auto masked, int j, char* now, char* next) __attribute__((always_inline)) {  // its fragments of K are there
    constexpr bool MASKED = decltype(masked)::value;
    if constexpr (!kAhead) {
      publish();
      if (j + 1 < ntiles) copy(j + 1, next);
      read_keys(now);
      __builtin_amdgcn_sched_barrier(0);
    }
    int vb = v_at;
    asm volatile("" : "+v"(vb));
    u32x4_t vw[8], pb[CG][4];
    f32x16_t s[CG][2];
    f32x2_t part[CG][4];
    auto logit = [&](int c, int q, int i) __attribute__((always_inline)) -> float {  // i of eight, keys 32 (q / 2) + 16 (q & 1) + 8 hi ..
      const float y = s[c][q >> 1][8 * (q & 1) + i];
      if constexpr (!MASKED) return y;
      return 32 * (q >> 1) + 16 * (q & 1) + i <= last[c] - j * kDenseKeys - 8 * hi ? y : kMasked;
    };
    auto softmax = [&](int c, int h) __attribute__((always_inline)) {  // four of a lane's 32 keys
      const float mk = m_run[c] * kf;
      float e[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) e[i] = __builtin_amdgcn_exp2f(fmaf(logit(c, h >> 1, 4 * (h & 1) + i), kf, -mk));
#pragma unroll
      for (int i = 0; i < 2; ++i) {  // (four chains)
        const f32x2_t x = {e[2 * i], e[2 * i + 1]};
        f32x2_t& sum = part[c][2 * (h & 1) + i];
        sum = h < 2 ? x : sum + x;
        pb[c][h >> 1][2 * (h & 1) + i] = pack2<T>(x.x, x.y);
      }
    };
    auto maximum = [&](int c) __attribute__((always_inline)) -> float {  // of the column, in both of its lanes
      float m = kMasked;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < 8; ++i) m = fmaxf(m, logit(c, q, i));
      uint32_t a = __builtin_bit_cast(uint32_t, m), b = a;
      half_swap(a, b);
      return fmaxf(__builtin_bit_cast(float, a), __builtin_bit_cast(float, b));
    };
    auto sum = [&](int c) __attribute__((always_inline)) -> f32x2_t { return (part[c][0] + part[c][1]) + (part[c][2] + part[c][3]); };
    auto start = [&](int c) __attribute__((always_inline)) {  // the first tile: nothing to rescale yet
      if (j > 0) return;
      const float m = maximum(c);
      if ((m - m_run[c]) * kf > kGrow) m_run[c] = fmaxf(m_run[c], m);
    };
    // A probability above 2^kGrow shows in the lane's sum (all terms are >= 0); only then the maximum is taken, and a column whose own grew
    // that much is rescaled and its exponentials taken again.
    auto settle = [&](int c) __attribute__((always_inline)) {
      f32x2_t l = sum(c);
      if (__builtin_amdgcn_ballot_w64(!(l.x + l.y <= kSumLimit)) != 0) {
        const float m = maximum(c);
        const bool grew = (m - m_run[c]) * kf > kGrow;
        if (__builtin_amdgcn_ballot_w64(grew) != 0) {
          const float m_new = grew ? fmaxf(m_run[c], m) : m_run[c];
          const float alpha = __builtin_amdgcn_exp2f((m_run[c] - m_new) * kf);
          l_run[c] *= alpha;
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[c][0][r] *= alpha, acc[c][1][r] *= alpha;
          m_run[c] = m_new;
#pragma unroll
          for (int h = 0; h < 8; ++h) softmax(c, h);
          l = sum(c);
        }
      }
      l_run[c] += l.x + l.y;
    };
#pragma unroll
    for (int c = 0; c < CG; ++c)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[c][0][r] = s[c][1][r] = 0.f;
    // K Q^T of a group (its two halves in turn: neither waits for itself), beside it the softmax of the one before, and the fragments of V
#pragma unroll
    for (int c = 0; c < CG; ++c) {
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        s[c][i & 1] = mfma32<T>(kw[i], qf[c][i >> 1], s[c][i & 1]);
        if (c == CG - 1) vw[i] = vread(now, vb, i);
        if (c > 0) {
          softmax(c - 1, i);
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (c > 0) settle(c - 1);
      start(c);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if (CG == 2) acc[0][i & 1] = mfma32<T>(vw[i], pb[0][i >> 1], acc[0][i & 1]);
      softmax(CG - 1, i);
      __builtin_amdgcn_sched_barrier(0);
    }
    settle(CG - 1);
    if constexpr (kAhead) {
      if (j + 1 < ntiles) publish();
      read_keys(next);
      __builtin_amdgcn_sched_barrier(0);
      if (j + 2 < ntiles) copy(j + 2, now);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) acc[CG - 1][i & 1] = mfma32<T>(vw[i], pb[CG - 1][i >> 1], acc[CG - 1][i & 1]);
    __builtin_amdgcn_sched_barrier(0);
  };
  if constexpr (kAhead) {
    publish();
    read_keys(stage0);
  }
  int j = 0;
#pragma nounroll
  for (; j + 1 < plain; j += 2) {  // (a tile's stage is a constant: fragment addresses are made once)
    tile(std::false_type{}, j, stage0, stage1);
    tile(std::false_type{}, j + 1, stage1, stage0);
  }
#pragma nounroll
  for (; j < my_tiles; ++j) tile(std::true_type{}, j, (j & 1) ? stage1 : stage0, (j & 1) ? stage0 : stage1);
#pragma nounroll
  for (j += kAhead; j < ntiles; ++j) {  // (copies for the others)
    publish();
    if (j + 1 < ntiles) copy(j + 1, (j & 1) ? stage0 : stage1);
  }

  // register r of block db is d = 32 db + 8 (r >> 2) + 4 hi + (r & 3)
#pragma unroll
  for (int c = 0; c < CG; ++c) {
    uint32_t a = __builtin_bit_cast(uint32_t, l_run[c]), b = a;
    half_swap(a, b);
    const float l = __builtin_bit_cast(float, a) + __builtin_bit_cast(float, b);
    const float inv = l > 0.f ? __fdividef(1.f, l) : 0.f;
    if (last[c] < 0) continue;
    S* row = (S*)p.out + (int64_t)(qbeg + t0 + c * TQ + cq) * p.out_stride + (int64_t)(head0 + ch) * kDenseHead;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        u32x2_t o;
        o.x = pack2<T>(acc[c][db][4 * rq + 0] * inv, acc[c][db][4 * rq + 1] * inv);
        o.y = pack2<T>(acc[c][db][4 * rq + 2] * inv, acc[c][db][4 * rq + 3] * inv);
        *reinterpret_cast<u32x2_t*>(row + 32 * db + 8 * rq + 4 * hi) = o;
      }
  }
}

// What dense_mfma32_takes takes (block_tables = seq_lens = null: context == chunk), 128 or 256 columns a workgroup
template <typename T>
static int launch_dense_attention(const PrefillParams& p0, int num_seqs, int max_query_len, int columns, hipStream_t stream) {
  PrefillParams p = p0;
  const int G = p.num_heads / p.num_kv_heads, HG = (G + 31) / 32;
  p.gp_shift = G == 1 ? 0 : G == 2 ? 1 : G <= 4 ? 2 : G <= 8 ? 3 : G <= 16 ? 4 : 5;
  auto grid_of = [&](int columns) {
    const int tokens = columns >> p.gp_shift;
    return dim3(p.num_kv_heads * HG, num_seqs, (max_query_len + tokens - 1) / tokens);
  };
  if (columns == 128) hipLaunchKernelGGL((dense_attention_kernel<T, 1>), grid_of(128), dim3(256), 0, stream, p);
  else hipLaunchKernelGGL((dense_attention_kernel<T, 2>), grid_of(256), dim3(256), 0, stream, p);
  return 0;
}

}  // namespace lvllm
