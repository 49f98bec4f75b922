// Which workgroup of the grouped products' launches takes which piece of work, in whole numbers that the host counts as well.
//
// A unit is a block of W rows of one tile of slots; a workgroup takes one.  An XCD gets an eighth of the last expert's units, which come
// first (the shared expert may be larger), and an eighth of all others'.
#pragma once
#include <math.h>
#include <stdint.h>

namespace lvllm {

struct TurnUnit {
  int unit;   // among the last expert's, or among all others'
  bool last;  // the last expert's
  bool any;
};
// Workgroup `cu` of an XCD; units_first, units_last: of all XCDs.
__host__ __device__ inline TurnUnit turn_unit(int units_first, int units_last, int xcd, int cu) {
  const int per_first = (units_first + 7) / 8, per_last = (units_last + 7) / 8;
  if (cu < per_last) {
    const int unit = xcd * per_last + cu;
    return {unit, true, unit < units_last};
  }
  const int mine = cu - per_last, unit = xcd * per_first + mine;
  return {unit, false, mine < per_first && unit < units_first};
}

// Their workgroups: an eighth of both kinds, rounded up, eight times.
inline int64_t unit_workgroups(int64_t units_first, int64_t units_last) {
  return 8 * ((units_first + 7) / 8 + (units_last + 7) / 8);
}

// Blocks of W rows of the other experts and of the last one.
struct BlockCounts {
  int first, last;
};

// Workgroups that slots spread evenly over all experts make.
inline int64_t even_workgroups(int rows, int64_t slots, int experts, int tile, const BlockCounts& b) {
  const int64_t even = (slots + (int64_t)experts * tile - 1) / ((int64_t)experts * tile), last = ((int64_t)rows + tile - 1) / tile;
  return experts * even * b.first + last * b.last;
}

// Whether whole blocks have a body for each height of a tile: more workgroups than two a CU, which power bounds.  With bodies of 4, 6 and 8 groups of 16
// slots, then of every height, us going up: 4096 rows, 6 of 64 experts of 2816, 2048 wide 612, 594; 3000 rows, 6 of 64 of 1408 and a shared one of
// 2816 312, 301; 8192 rows, 2 of 32 of 1408 and a shared one 294, 285.  Fewer workgroups wait for memory, and a launch with more code takes longer:
// 2500 rows, 2 of 16 of 512, 1024 wide (192) 28.3, 30.0; 1300 rows, 2 of 8 of 1024 (192) 27.9, 29.5; 1500 rows, 4 of 32 of 512 (256) 31.1, 31.9.
inline bool takes_every_height(int rows, int64_t slots, int experts, int tile, const BlockCounts& whole) {
  return even_workgroups(rows, slots, experts, tile, whole) > 512;
}

// Whether a prompt's products take half blocks (128 W rows) or whole ones, by the workgroups with work that slots spread evenly over
// the experts make.  `larger_last`: the last expert is larger, a shared one then, which has every row.  A half block's walk takes three
// quarters of a whole one's where a workgroup has a CU to itself, and where two share one no less than a whole one that has none beside
// it:
//   * half blocks where they fit a CU each.  Down, 2 of 16 experts of 1408, 2048 wide, 500 rows (128 of whole blocks, 256 of half), us
//     whole and half: 28.6, 21.5;
//   * whole ones where those fit: 4 of 32 experts of 512, 1024 wide (256), down, 1500 rows 17.3, 23.2; 2 of 16 of 2816 and a shared one
//     as large (136), 300 rows 53.4, 61.2;
//   * half ones for up to one and a half whole ones a CU: 2 of 32 of 1408 and a shared one of 2816, down, 300 rows (288) 68.6, 46.6;
//     2 of 16 of 1408, up, 1000 rows 75, 56 (tiles of 125 slots on the average: every expert may have one more, 352 for 176);
//   * going down, a larger expert's walks are the longest, and the launch waits for them: half ones for up to as many in any case.  2 of
//     8 of 1408 and a shared one of 2816, 1000 rows (256) 45.7, 43.0.
inline bool takes_half_blocks(int rows, int64_t slots, int experts, int tile, const BlockCounts& whole, const BlockCounts& half, bool up,
                              bool larger_last) {
  const int64_t last_tiles = ((int64_t)rows + tile - 1) / tile;
  auto workgroups = [&](const BlockCounts& b, bool shared) {  // shared: one that has every row, and the others what is left
    const double mean = shared ? (double)(slots > rows ? slots - rows : 0) / (experts > 1 ? experts - 1 : 1) : (double)slots / experts;
    const int64_t each = mean > 1 ? (int64_t)ceil((shared ? mean : mean + sqrt(mean)) / tile) : 1;  // (of all, who may have more)
    return unit_workgroups((experts - 1) * each * b.first, (shared ? last_tiles : each) * b.last);
  };
  if (workgroups(half, true) <= 256 || (!larger_last && workgroups(half, false) <= 256)) return true;
  if (even_workgroups(rows, slots, experts, tile, whole) > 384) return false;
  return (!up && larger_last) || workgroups(whole, larger_last) > 256;
}

}  // namespace lvllm
