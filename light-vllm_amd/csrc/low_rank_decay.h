// ln w [rows, channels] from a low-rank projection (log_decay.h), as exact bf16 parts on bf16 MFMAs.
//
// A float is the sum of three bf16 numbers (8 bits each), and the products of such parts are exact in fp32: with bf16 inputs as
// they are (f = identity) three MFMAs of 32 k stand for eight fp32 ones of 4 k, 48 clocks for 256.  Other inputs are split as
// well; of their nine products the six that reach fp32's last bit are taken.
// The error against 64 bits is 0.55 (logsigmoid) and 0.77 (exponential of tanh) of that of fp32 MFMAs and log1pf.  us alone, 8192 rows, rank 128, 2048 channels, logsigmoid: 107,
// now 45; exponentials of tanh: 78, 56; 4096 rows, rank 64: 45, 20 and 28, 26.  Writing the results is 14 of the 45, the rest
// the logarithms' vector instructions.
#pragma once
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

// A workgroup per 64 rows x 128 channels.  128 k of f(u) at a time through LDS; a wave splits the weights of its two tiles of 16
// channels in registers and takes them against all four row tiles.  A lane's results are 4 channels of a row.
constexpr int kDecayRows = 64, kDecayCols = 128, kDecayK = 128, kDecayLd = kDecayK + 8;
template <typename T, bool SPLIT>  // SPLIT: f(u) is not a bf16 number
static __global__ __launch_bounds__(256) void log_decay_kernel(float* __restrict__ out, const typename T::store_t* __restrict__ u,
                                                        const int64_t u_stride, const float* __restrict__ a_t,  // [rank, channels]
                                                        const float* __restrict__ bias, const int kind,
                                                        const float inv_tau, const float* __restrict__ scale,
                                                        const int rows, const int rank, const int channels) {
  constexpr int P = SPLIT ? 3 : 1;
  __shared__ __attribute__((aligned(16))) uint16_t su[P][kDecayRows][kDecayLd];
  const int row0 = blockIdx.y * kDecayRows, nr = min(kDecayRows, rows - row0);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), g = lane >> 4, c = lane & 15;
  const int ch0 = blockIdx.x * kDecayCols + wave * 32;
  auto input = [&](int row, int k) { return T::to_float(u[(int64_t)(row0 + min(row, nr - 1)) * u_stride + min(k, rank - 1)]); };
  auto f_of = [&](float x) { return kind == kDecayNegExp ? tanhf(x) : x; };
  r_f32x4_t z[2][4];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int i = 0; i < 4; ++i) z[j][i] = r_f32x4_t{0.f, 0.f, 0.f, 0.f};
  float odd = 0.f;  // of this wave's weights and of the inputs that this thread brings
  for (int kc = 0; kc < rank; kc += kDecayK) {
    if (kc > 0) __syncthreads();
    {  // two k of 16 rows a thread
      constexpr int N = kDecayRows / 4;
      float x[N][2];  // (all of a thread's loads in flight at once)
      const int k = kc + 2 * lane;
#pragma unroll
      for (int i = 0; i < N; ++i) { x[i][0] = input(wave + 4 * i, k); x[i][1] = input(wave + 4 * i, k + 1); }
#pragma unroll
      for (int i = 0; i < N; ++i) {
        uint32_t part[3];
        split2(k < rank ? f_of(x[i][0]) : 0.f, k + 1 < rank ? f_of(x[i][1]) : 0.f, part, odd);
#pragma unroll
        for (int s = 0; s < P; ++s) *reinterpret_cast<uint32_t*>(&su[s][wave + 4 * i][2 * lane]) = part[s];
      }
    }
    __syncthreads();
    const int steps = (min(rank - kc, kDecayK) + 31) / 32;
    for (int t = 0; t < steps; ++t) {
      d_u32x4_t a[2][3];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const float* at = a_t + min(ch0 + 16 * j + c, channels - 1);
        const int k = kc + 32 * t + 8 * g;
        float v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = at[(int64_t)min(k + i, rank - 1) * channels];  // (beyond the rank: f(u) is zero)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          uint32_t part[3];
          split2(v[2 * i], v[2 * i + 1], part, odd);
#pragma unroll
          for (int s = 0; s < 3; ++s) a[j][s][i] = part[s];
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        d_u32x4_t b[P];
#pragma unroll
        for (int s = 0; s < P; ++s) b[s] = *reinterpret_cast<const d_u32x4_t*>(&su[s][16 * i + c][32 * t + 8 * g]);
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int s = 2; s >= 0; --s)  // (the small ones first)
#pragma unroll
            for (int q = P - 1; q >= 0; --q)
              if (s + q < 3) z[j][i] = mfma_parts(a[j][s], b[q], z[j][i]);
      }
    }
  }
  if (__syncthreads_or(odd != 0.f)) {  // by themselves, in fp32
    for (int j = 0; j < 2; ++j)
      for (int i = 0; i < 4; ++i)
        for (int r = 0; r < 4; ++r) {
          const int ch = min(ch0 + 16 * j + 4 * g + r, channels - 1);
          float sum = 0.f;
          for (int k = 0; k < rank; ++k) sum = fmaf(a_t[(int64_t)k * channels + ch], f_of(input(16 * i + c, k)), sum);
#pragma unroll
          for (int jj = 0; jj < 2; ++jj)
#pragma unroll
            for (int ii = 0; ii < 4; ++ii)
#pragma unroll
              for (int rr = 0; rr < 4; ++rr)
                if (jj == j && ii == i && rr == r) z[jj][ii][rr] = sum;
        }
  }
  const bool vec = (channels & 3) == 0 && ((uintptr_t)out & 15) == 0;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int ch = ch0 + 16 * j + 4 * g;
    float bb[4], f[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      bb[r] = bias[min(ch + r, channels - 1)];
      f[r] = scale != nullptr ? scale[min(ch + r, channels - 1)] : inv_tau;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
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

// `scale` [channels] of softplus decays, or null: inv_tau
static int launch_log_decay(float* out, const void* u, int64_t u_stride, const float* a_t, const float* bias, int kind,
                            float inv_tau, const float* scale, int rows, int rank, int channels, int dtype, hipStream_t s) {
  if (rows == 0) return 0;
  LV_CHECK(rank > 0 && rank <= 512 && channels > 0, "rank must be in 1 .. 512");
  const int ny = (rows + kDecayRows - 1) / kDecayRows;
  LV_CHECK(ny <= 65535, "too many rows");
  const dim3 grid((channels + kDecayCols - 1) / kDecayCols, ny);
  LV_DISPATCH_DTYPE(dtype, {
    using S = scalar_t::store_t;
    if (dtype == LVLLM_BF16 && kind != kDecayNegExp)
      hipLaunchKernelGGL((log_decay_kernel<scalar_t, false>), grid, dim3(256), 0, s, out, (const S*)u, u_stride, a_t, bias, kind,
                         inv_tau, scale, rows, rank, channels);
    else
      hipLaunchKernelGGL((log_decay_kernel<scalar_t, true>), grid, dim3(256), 0, s, out, (const S*)u, u_stride, a_t, bias, kind,
                         inv_tau, scale, rows, rank, channels);
  });
  LV_LAUNCH_CHECK();
  return 0;
}

}  // namespace lvllm
