// ln w [rows, channels] from a low-rank projection (log_decay.h), as exact bf16 parts on bf16 MFMAs.
//
// A float is the sum of three bf16 numbers (8 bits each), and the products of such parts are exact in fp32: with bf16 inputs as
// they are (f = identity) three MFMAs of 32 k stand for eight fp32 ones of 4 k, 48 clocks for 256.  Other inputs are split as
// well; of their nine products the six that reach fp32's last bit are taken.
// The error against 64 bits is 0.55 (logsigmoid) and 0.77 (exponential of tanh) of that of fp32 MFMAs and log1pf.  us alone, 8192 rows, rank 64, 2048 channels,
// logsigmoid: 29; exponentials of tanh: 31; rank 128, 4096 channels, softplus: 76.  Writing the results is 14 (28) of these, the rest
// the logarithms' vector instructions.
#pragma once
#include <type_traits>

#include "log_decay.h"

namespace lvllm {

typedef __bf16 d_bf16x8_t __attribute__((ext_vector_type(8)));
typedef unsigned int d_u32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ r_f32x4_t mfma_parts(d_u32x4_t a, d_u32x4_t b, r_f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(d_bf16x8_t, a), __builtin_bit_cast(d_bf16x8_t, b), c, 0, 0, 0);
}

// two floats as three pairs of bf16; `odd` becomes NaN of what has no such parts (infinities, NaN, what rounds to infinity)
__device__ __forceinline__ void split2(float x, float y, uint32_t (&part)[3], float& odd) {
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    part[i] = pack2<BF16>(x, y);
    const float hx = __builtin_bit_cast(float, part[i] << 16), hy = __builtin_bit_cast(float, part[i] & 0xffff0000u);
    if (i == 0) odd = fmaf(hx, 0.f, fmaf(hy, 0.f, odd));
    x -= hx;
    y -= hy;
  }
}

// A workgroup per 16 RT rows x 64 CT channels.  64 of f(u)'s k at a time through LDS; a wave splits the weights of its CT tiles of 16 channels in
// registers and takes them against all row tiles; the weights of the next step are on their way meanwhile.  A lane's results are 4 channels of
// a row.
template <typename T, bool SPLIT, int RT, int CT>  // SPLIT: f(u) is not a bf16 number
static __global__ __launch_bounds__(256) void log_decay_kernel(float* __restrict__ out, const typename T::store_t* __restrict__ u,
                                                        const int64_t u_stride, const float* __restrict__ a_t,  // [rank, channels]
                                                        const float* __restrict__ bias, const int kind,
                                                        const float inv_tau, const float* __restrict__ scale,
                                                        const int rows, const int rank, const int channels) {
  constexpr int P = SPLIT ? 3 : 1, K = 64, kRows = 16 * RT, kPairs = K / 2, kSide = 256 / kPairs;  // kSide: rows that are staged at once
  __shared__ __attribute__((aligned(16))) uint16_t su[P][kRows][K + 8];
  const int row0 = blockIdx.y * kRows, nr = min(kRows, rows - row0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int ch0 = (blockIdx.x * 4 + wave) * 16 * CT;
  auto input = [&](int row, int k) { return T::to_float(u[(int64_t)(row0 + min(row, nr - 1)) * u_stride + min(k, rank - 1)]); };
  auto f_of = [&](float x) { return kind == kDecayNegExp ? tanhf(x) : x; };
  r_f32x4_t z[CT][RT];
#pragma unroll
  for (int j = 0; j < CT; ++j)
#pragma unroll
    for (int i = 0; i < RT; ++i) z[j][i] = r_f32x4_t{0.f, 0.f, 0.f, 0.f};
  float odd = 0.f;  // of this wave's weights and of the inputs that this thread brings
  float v[CT][8];   // the next step's weights
  auto weights = [&](int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < CT; ++j) {
      const float* at = a_t + min(ch0 + 16 * j + c, channels - 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) v[j][i] = at[(int64_t)min(k0 + 8 * g + i, rank - 1) * channels];  // (beyond the rank: f(u) is zero)
    }
  };
  for (int kc = 0; kc < rank; kc += K) {
    if (kc > 0) __syncthreads();
    {  // two k a thread of every kSide-th row
      constexpr int N = (kRows + kSide - 1) / kSide;
      float x[N][2];  // (all of a thread's loads in flight at once)
      const int pair = threadIdx.x % kPairs, side = threadIdx.x / kPairs, k = kc + 2 * pair;
#pragma unroll
      for (int i = 0; i < N; ++i) { x[i][0] = input(side + kSide * i, k); x[i][1] = input(side + kSide * i, k + 1); }
      weights(kc);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        uint32_t part[3];
        split2(k < rank ? f_of(x[i][0]) : 0.f, k + 1 < rank ? f_of(x[i][1]) : 0.f, part, odd);
#pragma unroll
        for (int s = 0; s < P; ++s) *reinterpret_cast<uint32_t*>(&su[s][side + kSide * i][2 * pair]) = part[s];
      }
    }
    __syncthreads();
    const int steps = (min(rank - kc, K) + 31) / 32;
    for (int t = 0; t < steps; ++t) {
      d_u32x4_t a[CT][3];
#pragma unroll
      for (int j = 0; j < CT; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t part[3];
          split2(v[j][2 * i], v[j][2 * i + 1], part, odd);
#pragma unroll
          for (int s = 0; s < 3; ++s) a[j][s][i] = part[s];
        }
      if (t + 1 < steps) weights(kc + 32 * (t + 1));
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        d_u32x4_t b[P];
#pragma unroll
        for (int s = 0; s < P; ++s) b[s] = *reinterpret_cast<const d_u32x4_t*>(&su[s][16 * i + c][32 * t + 8 * g]);
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int s = 2; s >= 0; --s)  // (the small ones first)
#pragma unroll
            for (int q = P - 1; q >= 0; --q)
              if (s + q < 3) z[j][i] = mfma_parts(a[j][s], b[q], z[j][i]);
      }
    }
  }
  if (__syncthreads_or(odd != 0.f)) {  // by themselves, in fp32
    for (int j = 0; j < CT; ++j)
      for (int i = 0; i < RT; ++i)
        for (int r = 0; r < 4; ++r) {
          const int ch = min(ch0 + 16 * j + 4 * g + r, channels - 1);
          float sum = 0.f;
          for (int k = 0; k < rank; ++k) sum = fmaf(a_t[(int64_t)k * channels + ch], f_of(input(16 * i + c, k)), sum);
#pragma unroll
          for (int jj = 0; jj < CT; ++jj)
#pragma unroll
            for (int ii = 0; ii < RT; ++ii)
#pragma unroll
              for (int rr = 0; rr < 4; ++rr)
                if (jj == j && ii == i && rr == r) z[jj][ii][rr] = sum;
        }
  }
  const bool vec = (channels & 3) == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
  for (int j = 0; j < CT; ++j) {
    const int ch = ch0 + 16 * j + 4 * g;
    float bb[4], f[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      bb[r] = bias[min(ch + r, channels - 1)];
      f[r] = scale != nullptr ? scale[min(ch + r, channels - 1)] : inv_tau;
    }
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int row = 16 * i + c;
      if (row >= nr || ch >= channels) continue;
      float* o = out + (int64_t)(row0 + row) * channels + ch;
      r_f32x4_t y;
#pragma unroll
      for (int r = 0; r < 4; ++r) y[r] = log_decay_of(z[j][i][r] + bb[r], kind, f[r]);
      if (vec) {
        *reinterpret_cast<r_f32x4_t*>(o) = y;
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (ch + r < channels) o[r] = y[r];
      }
    }
  }
}

template <typename T, bool SPLIT, int RT, int CT>
static void launch_log_decay_tiles(float* out, const void* u, int64_t u_stride, const float* a_t, const float* bias, int kind, float inv_tau,
                                   const float* scale, int rows, int rank, int channels, hipStream_t s) {
  hipLaunchKernelGGL((log_decay_kernel<T, SPLIT, RT, CT>), dim3((channels + 64 * CT - 1) / (64 * CT), (rows + 16 * RT - 1) / (16 * RT)),
                     dim3(256), 0, s, out, (const typename T::store_t*)u, u_stride, a_t, bias, kind, inv_tau, scale, rows, rank, channels);
}

// `scale` [channels] of softplus decays, or null: inv_tau
static int launch_log_decay(float* out, const void* u, int64_t u_stride, const float* a_t, const float* bias, int kind,
                            float inv_tau, const float* scale, int rows, int rank, int channels, int dtype, hipStream_t s) {
  if (rows == 0) return 0;
  LV_CHECK(rank > 0 && rank <= 512 && channels > 0, "rank must be in 1 .. 512");
  LV_CHECK((rows + 63) / 64 <= 65535, "too many rows");
  // Few tiles leave the chip idle and a workgroup's own chain is all there is; many bring f(u) and split the weights again in each of them.  us,
  // exponentials of tanh, rank 64, 2048 channels, tiles of 16 x 64, 32 x 64 and 64 x 128: 100 rows 4.2, 4.9, 8.8 (64 x 128 with 128 k at once and no
  // loads ahead: 13.0); 300 rows 5.5, 5.9, 9.1; 1000 rows 10.2, 8.9, 10.3; 2000 rows 17.0, 13.8, 12.7; 4096 rows 28.5, 22.1, 18.5 (26.0).
  const int64_t tiles = (int64_t)((rows + 15) / 16) * ((channels + 63) / 64);
  LV_DISPATCH_DTYPE(dtype, {
    auto with = [&](auto split) {
      constexpr bool S = decltype(split)::value;
      const auto launch = tiles <= 700    ? launch_log_decay_tiles<scalar_t, S, 1, 1>
                          : tiles <= 3800 ? launch_log_decay_tiles<scalar_t, S, 2, 1>
                                          : launch_log_decay_tiles<scalar_t, S, 4, 2>;
      launch(out, u, u_stride, a_t, bias, kind, inv_tau, scale, rows, rank, channels, s);
    };
    if (dtype == LVLLM_BF16 && kind != kDecayNegExp) with(std::false_type());
    else with(std::true_type());
  });
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm
