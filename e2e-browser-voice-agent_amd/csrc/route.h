// route.h -- which kernel takes a call: rules on sizes, types and positions, every candidate giving the
// same bits.  Host code without HIP, so that a test can compile it alone.  The figures beside each rule
// are MI355X times of the two sides.
#pragma once
#include <stddef.h>

namespace q4 {

// ---- one-token projections

// k_matvec_split takes rows of kSplitMinBlocks .. kSplitMaxBlocks blocks.
constexpr int kSplitMinBlocks = 64;
constexpr int kSplitMaxBlocks = 480;

// Whether a matvec on device buffers (N rows of nb blocks, y not over x) quantizes x in the projection's
// own workgroups, or in a launch before them.  One launch costs about 2 us, whatever N; each workgroup's
// own quantize costs nothing where all workgroups run at once or each takes many row groups, and adds up
// where they come in many rounds:
//   rows of up to 63 blocks  any N (microseconds two launches / one: 896 x 896 6.0 / 4.3, 151936 rows of
//                            28 blocks 15.6 / 13.9, of 4 7.3 / 5.9, of 63 33.2 / 32.1)
//   wider (k_matvec_split,   up to 1792 workgroups and as many as leave the blocks quantized in all within
//   a workgroup per 16 rows) 440000: 896 x 4864 8.7 / 6.2, 28672 x 3200 24.2 / 23.1, 24576 x 8960 62.4 /
//                            61.9, 16384 x 12800 59.0 / 57.3; beyond, 151936 x 2048 69 / 81, 80000 x 8960
//                            195 / 203, 24576 x 15360 99.7 / 101.2
inline bool mv_quantizes_itself(int N, int nb) {
  if (nb > kSplitMaxBlocks) return false;
  if (nb < kSplitMinBlocks) return true;
  const long wgs = ((long)N + 63) / 64 * 4;
  return wgs <= 1792 && wgs * nb <= 440000;
}

// ---- attention

// Shared memory of k_attn_head, whose workgroup takes one row and head: the K stages and V slots, the row
// of scores (exponentials, probabilities) of up to `end` positions -- every position, the +0 past them
// for ordered_sum_wave and the rest of the last P.V chunk -- and the waves' q and reductions.  `end` is
// one past the last position that any row of the call looks at, not the context's size: two workgroups
// fit a CU up to about 3,600 positions (head_dim 64; 3,300 with 128), one beyond.
constexpr int kHeadStageBytes = 64 * 1024;
constexpr int head_row(int end) { return ((end + 31) & ~31) + 128 + (end >> 6); }
constexpr size_t attn_head_lds(int HD, int end) {
  return (size_t)kHeadStageBytes + (size_t)(head_row(end) + 16 + 4 * HD) * sizeof(float);
}

}  // namespace q4
