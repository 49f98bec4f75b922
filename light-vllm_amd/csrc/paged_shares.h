// Shares that paged decode attention cuts each context into, in whole numbers.
#pragma once
#include <stdint.h>

#include <algorithm>

namespace lvllm {

// The reference always cuts at 512 tokens; here the cut exists only to fill the GPU: with >= 8 waves per CU from (sequence, kv head) pairs
// alone there is no cut at all (one pass, no merge), otherwise just enough shares, bounded by the caller's scratch (slots per head) and by a
// minimum of 4 tiles of 16 tokens per share.  The lengths are on the device: a batch of `max_seq_len` may hold one such context and many short
// ones, whose longest walk is the launch, or equal ones, whose workgroups are.
//   * Two shares of more than 128 pairs are more workgroups than CUs: equal contexts pay a second turn, which the last of them waits for, and
//     the merge.  Up to 1024 tokens the walk of a whole context is no longer than that of its half and the merge, so that there is no cut, whatever
//     the other lengths.  One layer of 8 kv heads of 128, us in two shares and whole: 17 of 1000 27.1, 19.4; 24 of 700 26.5, 17.6; 31 of 1000 down to
//     nothing 23.4, 20.0; 17 and 24 of which one has 1000 and the others 100 16.2, 16.2 and 16.8, 16.5.
//   * Beyond, a long context among short ones would take up to twice as long (17, one of 2000 and the others of 200: 20.3, 25.7; one of 16000: 85,
//     154), where equal ones would gain a fifth (20 of 2000 42.4, 33.1).
//   * One share fewer than fills the CUs, where that is a part of a second turn, is the same exchange (12 of 2000 32.9, 25.0 with two; one of 16000
//     and 11 of 200 61, 84).
// Contexts of an fp8 cache are cut as they were: 24 of 1024 27.1, would be 24.2 whole, but behind such a cache projections are most often of 8 bits
// too, and there the last bit of a merge moves logits by 0.11 (relative, four layers): neither cut is the more exact one.
inline int paged_shares(int num_seqs, int num_heads, int num_kv_heads, int max_seq_len, int slots, bool mfma, bool fp8) {
  const int G = num_heads / num_kv_heads;
  const int64_t pairs = mfma ? (int64_t)num_seqs * num_kv_heads * ((G + 15) / 16) : (int64_t)num_seqs * num_heads;
  const int64_t want = mfma ? (2048 + 8 * pairs - 1) / (8 * pairs) : (1024 + pairs - 1) / pairs;
  if (mfma && !fp8 && pairs > 128 && max_seq_len <= 1024) return 1;
  const int n = (int)std::min<int64_t>({want, slots, ((int64_t)max_seq_len + 15) / 16 / 4});
  return n < 1 ? 1 : n;
}

}  // namespace lvllm
