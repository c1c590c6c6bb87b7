// route.h -- which kernel takes a call: rules on sizes, types and positions, every candidate giving the
// same bits.  Host code without HIP, so that a test can compile it alone.  The figures beside each rule
// are MI355X times of the two sides.
#pragma once
#include <stddef.h>

namespace q4 {

constexpr int kXcds = 8, kCus = 256;

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

// ---- projections of prompt passes

// Whether k_gemm_tile (64 tokens x 32 rows, three workgroups on a CU) takes a projection of nrg groups of 32
// rows, against k_gemm_sk; qkv: the q|k|v projection, whose epilogue is RoPE and the cache append.  Its
// time steps up with every round of 256 workgroups (down of the 0.5B shape 47 us in one round, 59 in two),
// where k_gemm_sk's grows with every 16 tokens, so it takes the sizes that nearly fill their last round: a
// single round by the 16-token groups it holds, more by the workgroups.  Whole passes, ms by k_gemm_sk / with
// o and down by k_gemm_tile:
//   one round     1.5B shape 288 tokens 7.25 / 7.50, 304 7.57 / 7.57, 320 7.68 / 7.67; 0.5B 512 4.21 / 4.30,
//                 544 4.75 / 4.73
//   two, three..  1.5B 512 9.72 / 10.31, 608 12.03 / 11.65, 672 13.2 / 13.7, 768 14.83 / 14.79, 1,024 19.3 /
//                 18.4; 0.5B 640 4.97 / 5.33, 864 6.35 / 6.69, 992 7.55 / 7.38
// q|k|v in one or two rounds is slower with its registers' RoPE epilogue (0.5B 448 tokens 4.13 / 4.18, 832
// 6.10 / 6.18, 1.5B 400 8.85 / 8.90) and level from there (1.5B 576 11.56 / 11.61, 1,024 19.26 / 19.10).
constexpr int kTileMinTokens = 256;   // below, half of a 64-token tile may be idle
inline bool tile_takes(int nrg, int M, bool qkv) {
  if (M < kTileMinTokens) return false;
  const int wgs = nrg * ((M + 63) / 64), rounds = (wgs + kCus - 1) / kCus;
  if (rounds <= 2 && qkv) return false;
  if (rounds == 1) return nrg * ((M + 15) / 16) * 100 >= 88 * 4 * kCus;
  return wgs * 100 >= (rounds == 2 ? 85 : 75) * kCus * rounds;
}

// Whether it takes the fused gate|up projection (64 tokens x one 32-value block) of nrg blocks: from nearly
// two workgroups per CU on (456: 152 blocks by three tiles was the least that paid, 304 the most that did
// not), up to three token tiles only where the last one is well filled.  Whole passes, ms by k_gemm_sk / by
// it: 0.5B shape 128 tokens 1.84 / 1.91, 160 2.15 / 2.14, 176 2.31 / 2.23, 193 2.42 / 2.40, 208 2.44 / 2.42,
// 224 2.73 / 2.64, 257 3.03 / 2.82; 1.5B 112 3.83 / 3.90, 120 4.15 / 4.10, 160 4.99 / 5.18, 176 5.63 / 5.61, 193
// 6.08 / 5.92, 224 6.72 / 6.43, 288 8.02 / 7.49.
inline bool tile_takes_gu(int nrg, int M) {
  const int nt = (M + 63) / 64, last = M - 64 * (nt - 1);
  return nrg * nt >= 456 && last > (nt <= 2 ? 48 : nt == 3 ? 32 : 0);
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

// The positions a call's rows look at: one past the last of any row, and the mean of the rows on the XCD
// that has most of them.
struct AttnSpan {
  int end, mean;
};

// M tokens of a pass from pos on.
constexpr AttnSpan pass_span(int pos, int M) { return {pos + M, pos + (M + 1) / 2}; }

// k_attn_head's workgroups: units (row, kv head) dealt to the 8 XCDs, the G heads of a unit 8 apart.
constexpr int attn_head_grid(int rows, int KVH, int G) { return (rows * KVH + kXcds - 1) / kXcds * kXcds * G; }

// `steps` steps of B sequences at pos[]: sequences of different lengths may meet on an XCD (k_attn_head
// deals its units from the last sequence on).
inline AttnSpan batch_span(const int* pos, int B, int KVH, int steps) {
  long load[kXcds] = {}, most = 0;
  int last = 0;
  for (int b = 0; b < B; b++) {
    if (pos[b] > last) last = pos[b];
    for (int g = 0; g < KVH; g++) {
      long& l = load[((B - 1 - b) * KVH + g) % kXcds];
      l += pos[b] + (steps + 1) / 2;
      if (l > most) most = l;
    }
  }
  const int per = (B * KVH + kXcds - 1) / kXcds;
  return {last + steps, (int)((most + per - 1) / per)};
}

// How many of its workgroups run at once.
constexpr int head_slots(int HD, int end) { return kCus * (attn_head_lds(HD, end) <= 80 * 1024 ? 2 : 1); }

// Whether k_attn_head takes a prompt pass of `rows` rows, against k_attn_rows (head_dim 64) or three
// launches (128), which read a K row once for the heads of a group.  Both sides timed as whole passes, ms
// theirs / its (0.5B shape: 14 heads of 64 in groups of 7; 1.5B shape: 12 of 128 in groups of 6):
//   head_dim 64   while its workgroups run at once, any group and position (0.5B, 36 rows at 0 1.44 / 1.23,
//     at 3,000 3.09 / 2.19).  A second round costs as much again, where k_attn_rows' time grows with the
//     group: groups of 3 to 5 leave nothing (40 rows of groups of 4 at 600 1.68 / 1.72), larger ones half
//     of it (0.5B, 48 rows at 3,000 3.11 / 2.88) and all of it while positions are few (72 rows at 220 1.73 /
//     1.66, 600 1.94 / 1.93, 1,500 2.45 / 2.51), groups of two half (40 rows at 1,500 2.48 / 2.29, 62 at
//     600 1.96 / 1.99).  No group: faster at any size measured, to 1,024 heads.
//   head_dim 128  two rounds (1.5B, fp16, 64 rows at 3,000 5.93 / 5.21), with fp32 rows up to some 1,400
//     positions (64 rows at 1,000 4.16 / 3.98, 72 at 1,500 4.84 / 4.90, 48 at 3,000 5.72 / 5.81); more where
//     positions are few (fp32, 128 rows at 220 4.54 / 4.46, at 400 4.73 / 4.77, 256 at 0 6.89 / 6.79, at 220
//     7.28 / 7.57); groups of one or two at any size measured, to 3,072 heads.
inline bool head_takes_pass(int rows, int H, int KVH, int HD, bool kv16, AttnSpan sp) {
  const int G = H / KVH, slots = head_slots(HD, sp.end), grid = attn_head_grid(rows, KVH, G);
  const int rounds = (grid + slots - 1) / slots;
  if (rows * H > (HD == 64 ? 1024 : 3072)) return false;
  if (rounds == 1 || G == 1) return true;
  if (HD == 64) {
    if (slots == kCus) return G >= 6 && rounds == 2;       // 0.5B, 32 rows at 3,600: 79 / 65 us a layer
    return G == 2 ? grid <= 768 : G >= 6 && (grid <= 768 || (rounds == 2 && sp.mean <= 704));
  }
  if (G == 2) return true;
  return rounds == 2 ? kv16 || sp.mean <= 1400 : (long)rounds * sp.mean <= (kv16 ? 1700 : 1350);
}

// Whether it takes one token, or one of each sequence of a batch, against k_attn_scores_list and
// k_attn_pv_list, which spread a row's positions over workgroups and read a cache row once for the heads
// of a group.  ms of a whole step, theirs / its (32 sequences of 300, 0.5B 1.63 / 1.40).  Not:
//   * rows of 128 fp32 columns past some positions.  The heads of a group read the rows one after the
//     other, and from there on the rows leave the L2 in between.  1.5B, 2 sequences of 700 2.47 / 2.39, of
//     1,024 2.59 / 2.68; 32 of 700 2.83 / 2.75, of 3,000 4.09 / 4.83; one token of 12 layers at 700 0.71 /
//     0.67, at 1,500 0.83 / 0.91; the smaller the group, the sooner (16 heads in groups of 4, 2 sequences of
//     600 1.007 times as fast, of 1,024 0.94; in groups of 1 300 1.00, 1,024 0.86).  One long row is enough
//     (16 sequences of 200 and one of 1,500 0.93 times as fast).  Large batches of small groups read enough on
//     either side to hide it (groups of 4, 24 sequences of 3,000 1.05; groups of 2, 16 sequences 1.05).
//   * large groups in more workgroups than run at once, where the list kernels' two workgroups fit a CU or
//     head_dim is 64, past some 300 to 700 positions (0.5B, 64 sequences of 500 1.92 / 1.88, of 700 2.00 /
//     2.06, 48 of 700 1.85 / 1.83; 1.5B fp16, 48 of 900 in a context of 940 0.97, of 4,352 1.09), and past some
//     3,500 positions, where one of its own does (32 sequences of 3,800 83 / 91 us a layer).  Rows of unequal
//     length run at once if their positions do while the longest runs (0.5B, 64 sequences of 16 to 900 1.07
//     times as fast, of 900 0.95, every other one of 900 0.91: those meet on half the XCDs).
inline bool head_takes_rows(int rows, int H, int KVH, int HD, bool kv16, int ctx, AttnSpan sp) {
  if (rows == 1) sp.end = sp.mean;         // a captured step is launched for all of the context
  const int G = H / KVH, slots = head_slots(HD, sp.end), grid = attn_head_grid(rows, KVH, G);
  const long work = (long)grid * sp.mean, once = (long)slots * sp.end;
  const bool one_round = work <= once || (4L * sp.mean <= 3L * sp.end && 4 * work <= 5 * once);
  const bool list_pairs = 34 * 1024 + 4L * G * ctx <= 80 * 1024;       // two k_attn_pv_list workgroups fit a CU
  if (HD == 128 && !kv16) {
    if (slots == 2 * kCus && 3L * sp.mean >= 2L * sp.end &&
        (G <= 2 ? grid >= 128 * G : G == 4 && grid >= 384 && !list_pairs))
      return true;
    if (G >= 5 && grid > 2 * kCus && one_round) return sp.end <= 1024;
    int most;                              // positions up to which it is the faster one
    if (G >= 5) most = one_round ? 832 : list_pairs ? 288 : 640;
    else most = G >= 3 ? (!one_round && list_pairs ? 400 : 704) : G == 2 ? 512 : 384;
    if (sp.mean > most || sp.end > most + 64) return false;
  }
  if (one_round || G <= 2) return true;
  if (slots == kCus) return false;
  if (HD == 128) return sp.end <= 512 || !list_pairs;
  return G == 4 || (G == 3 && !list_pairs) || sp.end <= (grid <= 768 ? 704 : 576);
}

}  // namespace q4
