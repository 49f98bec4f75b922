// Which body reads the rows of whole sequences in place (lvllm_varlen_attention), in whole numbers.
#pragma once
#include <stdint.h>

namespace lvllm {

// kDenseWaves: prefill_mfma32.h, DENSE, 32 columns a wave in workgroups of 128 or 256 that have a CU's registers to themselves in pairs or alone.
// kDense128, kDense256: dense_attention.h, three workgroups of 128 columns a CU or two of 256.
enum DenseBody { kDenseWaves, kDense128, kDense256 };

// The lengths are on the device, and a launch has as many blocks of columns for each sequence as the longest takes.  Where they differ, most of its
// workgroups end at once, and those of a long sequence lie two and three on a part of the CUs: with few of them, their walks beside each other are the
// launch.  `work`: workgroups of 128 columns if the tokens were one sequence.  16 heads, us in the three bodies:
//   * long walks that fill the chip several times over: 256 columns.  32 x 512 71, 67, 61; 8 x 2048 174, 151, 144.  Causal walks differ by themselves:
//     2 x 4096 92, 86, 98; 16 of 8000 down to nothing 985, 945, 876;
//   * lengths alike, or enough of them: 128 columns.  4 x 512 18.5, 15.0, 19.6; 1 x 2048 42, 36.6, 48; 24 x 400 47, 43, 43; 16 of 2000 down to nothing,
//     causal, 100, 83, 87.  But of 257 to 400 workgroups some CUs have two and others one (3 x 1000 26.8, 28.4, 31.9), and causal walks of up to eight
//     tiles are no shorter here (8 x 512 18.2, 19.5, 23.5);
//   * the rest: one of 2000 and 8 of 100 44, 54, 70; one of 4000 and 20 of 50, causal, 70, 75, 112; 16 of 512 down to nothing 23.2, 25.3, 30.8.
// 824 launches of 1 to 128 sequences, seven shapes of heads and lengths alike, halving, falling, random and single: 0.70 to 1.05 of the first body,
// mean 0.937.
inline DenseBody dense_body(int num_seqs, int num_tokens, int longest, int heads, int kv_heads, bool causal) {
  const int group = heads / kv_heads, head_groups = (group + 31) / 32;
  int padded = 1;  // heads a query token has among 32 columns
  while (padded < group && padded < 32) padded *= 2;
  const int64_t work = (int64_t)num_tokens * padded * kv_heads * head_groups / 128;
  if (causal ? longest >= 3000 && work >= 4096 : longest >= 512 && work >= 1024) return kDense256;
  if (causal ? longest > 256 && longest <= 512 && work <= 512 : work > 256 && work <= 400) return kDenseWaves;
  const bool alike = (int64_t)num_tokens * 5 >= (int64_t)num_seqs * longest * 3;
  return alike || work >= 1536 ? kDense128 : kDenseWaves;
}

}  // namespace lvllm
