// attn_head.h -- attention of one query row and one head per workgroup.
//
// Scores, softmax, P.V and the quantize of the head's output in one launch, every step in the
// reference's per-output order (engine/kernels.c:355-377): four lane sums over i = j mod 4 per score,
// the maximum, e_t = fast_exp(s_t - max), the sum in position order, p_t = e_t / sum, then out[c] =
// sum_t p_t * v_t[c] in position order.
//
// What bounds it is latency: two chains of T dependent additions (the sum; each column of P.V) and
// the round trips to the cache in front of them.  So the workgroup is one (row, head), the smallest
// unit with chains of its own, which spreads few rows over many CUs, and inside it
//   * the waves share the positions of the scores.  K rows come as 64-row stages of 128 bytes a row
//     by asynchronous global -> LDS loads, coalesced (8 lanes a row), each wave through two
//     stages of its own, with no barrier.  The 16-byte pieces of a row are rotated by the row's
//     number, so the 64 rows a wave reads piece by piece fall on distinct banks.
//   * P.V keeps all waves at work on the columns' chains.  A single wave issues an instruction about
//     every 5 cycles, so a chain costs what its wave issues per position.  With 64 columns, waves 1..3
//     form the products p_t * v_t[c] (each rounded, as in the reference's acc + p*v) of 128-position
//     chunks in shared memory and wave 0 only reads and adds them, one lane per column.  With 128
//     columns those products are twice the shared-memory traffic with half the waves to form them, so
//     waves 0 and 1 form and add theirs and waves 2 and 3 only load V to shared memory, ahead.
// Workgroups of one (row, kv head) run on one XCD (workgroup L runs on XCD L mod 8), so the heads of
// a group read their K and V rows from one L2.
#pragma once
#include <type_traits>

#include "gemm_sk.h"
#include "kernels.h"
#include "route.h"

namespace q4 {

constexpr int kHeadThreads = 256;
constexpr int kHeadStage = 8192;        // bytes of a K stage: 64 rows x 128 bytes
constexpr int kHeadMaxLds = 160 * 1024;
static_assert(kHeadStageBytes == kHeadThreads / 64 * 2 * kHeadStage, "two K stages per wave (three were no faster)");

// Four neighbouring cache values, and a product with one: rounded once to fp32.  An fp16 value is
// widened inside the instruction (v_fma_mix with an addend of +0, which can only turn a product of
// -0 into +0: every sum here starts at +0, where both add the same).
template <class KT> struct HeadVec { typedef float4 T; };
typedef _Float16 head_h2 __attribute__((ext_vector_type(2)));
typedef _Float16 head_h4 __attribute__((ext_vector_type(4)));
template <> struct HeadVec<kvhalf> { typedef head_h4 T; };
__device__ __forceinline__ float head_mul(float a, float v) { return a * v; }
__device__ __forceinline__ float head_mul(float a, _Float16 v) { return __builtin_fmaf(a, (float)v, 0.0f); }

// Asynchronous global -> LDS load of 16 bytes per lane (sk_dma16) from a wave-uniform base and a
// 32-bit offset per lane.
__device__ __forceinline__ void head_dma16(const void* base, uint32_t off, const void* lds) {
  const uint32_t a = (uint32_t)(uintptr_t)(SkLds*)lds;
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "{m0}"(a) : "memory");
}

// Value K of a register that holds 16 of them in each 16-lane row, in every lane (a DPP broadcast,
// folded into the product that uses it).
template <int K>
__device__ __forceinline__ float head_bcast(float v) {
  return __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x150 + K, 0xF, 0xF, true));
}
// The four lane sums of a score over elements 4 u .. 4 u + 3 of a K row, u = U .. U + N - 1 (q: 16
// values per register).
template <class KT, int U, int N>
struct head_dot {
  static __device__ __forceinline__ void run(float (&s)[4], const float* q, const typename HeadVec<KT>::T* k) {
    const float qv = q[U >> 2];
    constexpr int o = (U & 3) * 4;
    s[0] = s[0] + head_mul(head_bcast<o>(qv), k->x);
    s[1] = s[1] + head_mul(head_bcast<o + 1>(qv), k->y);
    s[2] = s[2] + head_mul(head_bcast<o + 2>(qv), k->z);
    s[3] = s[3] + head_mul(head_bcast<o + 3>(qv), k->w);
    head_dot<KT, U + 1, N - 1>::run(s, q, k + 1);
  }
};
template <class KT, int U>
struct head_dot<KT, U, 0> {
  static __device__ __forceinline__ void run(float (&)[4], const float*, const typename HeadVec<KT>::T*) {}
};

// P.V of one head: out[c] = sum_t p_t * v_t[c] in position order, p in shared memory at p (positions
// past T - 1 within the last chunk are readable), 64 KB of shared memory at `area`.  Every wave of
// the workgroup calls start() and run(); waves 0 .. HD / 64 - 1 return the sum of column().
// Chunk c is added after run()'s c-th barrier.  Positions past T - 1 add +0: a sum that began at +0
// stays as it is (it is never -0).
template <int HD, class KT>
struct HeadPv;

template <class KT>
struct HeadPv<64, KT> {
  // chunk c's products are formed by the waves 1..3 (a lane takes the VN columns of a 16-byte load, an
  // instruction RPI rows) in buffer c & 1, from register set c mod NS, which loads NS chunks ahead
  static constexpr int HD = 64, CH = 128, VN = 16 / (int)sizeof(KT), LPR = HD / VN, RPI = 64 / LPR;
  static constexpr int NGT = CH / RPI, NG = (NGT + 2) / 3, NS = sizeof(KT) == 2 ? 3 : 2;
  const int wave, lane, T, nch, vrow, vcol;
  const unsigned char* const vb;
  float* const prod;                       // [2][position of the chunk][HD]
  const float* const p;
  uint4 vset[NS][NG];
  __device__ __forceinline__ HeadPv(int wave, int lane, int T, const unsigned char* vb, void* area, const float* p)
      : wave(wave), lane(lane), T(T), nch((T + CH - 1) / CH), vrow(lane / LPR), vcol(VN * (lane % LPR)), vb(vb),
        prod((float*)area), p(p) {}
  __device__ __forceinline__ int column() const { return lane; }
  __device__ __forceinline__ void load(int c, uint4 (&r)[NG]) const {
#pragma unroll
    for (int n = 0; n < NG; n++) {
      const int t = min(CH * c + RPI * (wave - 1 + 3 * n) + vrow, T - 1);
      r[n] = *reinterpret_cast<const uint4*>(vb + (uint32_t)(t * HD + vcol) * (uint32_t)sizeof(KT));
    }
  }
  template <bool WHOLE>
  __device__ __forceinline__ void form(int c, const uint4 (&r)[NG]) const {
    float* const d = prod + (c & 1) * CH * HD + vcol;
    float pr[NG];                          // all read ahead of the first store: the accesses are served in order
#pragma unroll
    for (int n = 0; n < NG; n++) pr[n] = p[CH * c + min(RPI * (wave - 1 + 3 * n) + vrow, CH - 1)];
#pragma unroll
    for (int n = 0; n < NG; n++) {
      __builtin_amdgcn_sched_barrier(0);   // one group's products in registers at a time
      const int row = RPI * (wave - 1 + 3 * n) + vrow;
      if (3 * (n + 1) <= NGT || wave - 1 + 3 * n < NGT) {
        const bool in = WHOLE || CH * c + row < T;
        const float* f = reinterpret_cast<const float*>(&r[n]);
        const _Float16* hf = reinterpret_cast<const _Float16*>(&r[n]);
        float v[VN];
#pragma unroll
        for (int k = 0; k < VN; k++) {
          if constexpr (sizeof(KT) == 2) v[k] = head_mul(pr[n], hf[k]);
          else v[k] = pr[n] * f[k];
          if constexpr (!WHOLE) v[k] = in ? v[k] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < VN; k += 4)
          *reinterpret_cast<float4*>(d + row * HD + k) = make_float4(v[k], v[k + 1], v[k + 2], v[k + 3]);
      }
    }
  }
  __device__ __forceinline__ void start() {
    if (wave > 0) {
#pragma unroll
      for (int k = 0; k < NS; k++) load(k, vset[k]);
    }
  }
  __device__ __forceinline__ float run() {
    float acc = 0.0f;
    if (wave > 0) {
      // whole rounds of NS chunks without a branch, so that no register is copied (and no load
      // waited for) where paths meet; the last chunks are loaded already
      int c = 0;
      for (; c + NS < nch; c += NS)
#pragma unroll
        for (int k = 0; k < NS; k++) {
          form<true>(c + k, vset[k]);
          load(c + k + NS, vset[k]);
          lds_barrier();
        }
#pragma unroll
      for (int k = 0; k < NS; k++)
        if (c + k < nch) {
          form<false>(c + k, vset[k]);
          lds_barrier();
        }
    } else {
      constexpr int BT = 32;               // positions read ahead of the additions
      for (int c = 0; c < nch; c++) {
        lds_barrier();
        const float* const col = prod + (c & 1) * CH * HD + lane;
        // the last chunk stops at the batch that holds position T - 1
        const int nb = min(CH / BT, (T - CH * c + BT - 1) / BT);
        float d[2][BT];
        auto read = [&](int j, float (&r)[BT]) {
#pragma unroll
          for (int k = 0; k < BT; k++) r[k] = col[(BT * j + k) * HD];
        };
        read(0, d[0]);
#pragma unroll
        for (int j = 0; j < CH / BT; j++) {
          if (j < nb) {
            if (j + 1 < CH / BT) read(j + 1, d[(j + 1) & 1]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < BT; k++) acc = acc + d[j & 1][k];
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    }
    lds_barrier();
    return acc;
  }
};

template <class KT>
struct HeadPv<128, KT> {
  // V chunk c (64 positions) comes to slot c mod SL, half of it by each of the waves 2 and 3.  An fp16
  // row's columns 2 l and 2 l + 1 are read as one word by lane l of wave 0 (which takes the first) and
  // of wave 1 (the second), so that one instruction reads two positions, as with fp32.
  static constexpr int HD = 128, CH = 64, RB = HD * (int)sizeof(KT), SL = 65536 / (CH * RB), VI = CH * RB / 2048;
  static constexpr int RPI = 1024 / RB;    // rows of a load instruction
  const int wave, lane, T, nch;
  const unsigned char* const vb;
  unsigned char* const area;
  const float* const p;
  __device__ __forceinline__ HeadPv(int wave, int lane, int T, const unsigned char* vb, void* area, const float* p)
      : wave(wave), lane(lane), T(T), nch((T + CH - 1) / CH), vb(vb), area((unsigned char*)area), p(p) {}
  __device__ __forceinline__ int column() const { return sizeof(KT) == 2 ? 2 * lane + wave : 64 * wave + lane; }
  __device__ __forceinline__ void issue(int c) const {
    const int t0 = CH * min(c, nch - 1) + RPI * VI * (wave - 2) + lane / (RB / 16);
    unsigned char* const d = area + (c % SL) * (CH * RB) + 1024 * VI * (wave - 2);
#pragma unroll
    for (int k = 0; k < VI; k++)           // rows past T - 1 repeat it and are never added
      head_dma16(vb, (uint32_t)min(t0 + RPI * k, T - 1) * RB + 16 * (lane % (RB / 16)), d + 1024 * k);
  }
  template <bool WHOLE, int HALF>
  __device__ __forceinline__ void add(int c, float& acc) const {
    typedef typename std::conditional<sizeof(KT) == 2, uint32_t, float>::type W;
    const W* const v = reinterpret_cast<const W*>(area + (c % SL) * (CH * RB)) + (sizeof(KT) == 2 ? lane : 64 * wave + lane);
    const float* const pc = p + CH * c;
    constexpr int BT = 16, RS = RB / 4;    // positions of a batch, read one batch ahead of the additions
    float4 pb[2][BT / 4];
    W vb2[2][BT];
    auto read = [&](int j, int st) {
#pragma unroll
      for (int k = 0; k < BT; k++) vb2[st][k] = v[(BT * j + k) * RS];
#pragma unroll
      for (int k = 0; k < BT / 4; k++) pb[st][k] = *reinterpret_cast<const float4*>(pc + BT * j + 4 * k);
    };
    read(0, 0);
#pragma unroll
    for (int j = 0; j < CH / BT; j++) {
      if (j + 1 < CH / BT) read(j + 1, (j + 1) & 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int k = 0; k < BT; k++) {
        const float4& p4 = pb[j & 1][k >> 2];
        const float pk = (k & 3) == 0 ? p4.x : (k & 3) == 1 ? p4.y : (k & 3) == 2 ? p4.z : p4.w;
        float d;
        if constexpr (sizeof(KT) == 2) {
          const head_h2 h = __builtin_bit_cast(head_h2, vb2[j & 1][k]);
          d = head_mul(pk, h[HALF]);
        } else {
          d = pk * vb2[j & 1][k];
        }
        if constexpr (!WHOLE) d = CH * c + BT * j + k < T ? d : 0.0f;
        acc = acc + d;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  template <int HALF>
  __device__ __forceinline__ float sum() const {
    float acc = 0.0f;
    for (int c = 0; c + 1 < nch; c++) {
      lds_barrier();
      add<true, HALF>(c, acc);
    }
    lds_barrier();
    add<false, HALF>(nch - 1, acc);
    return acc;
  }
  __device__ __forceinline__ void start() const {
    if (wave >= 2) {
#pragma unroll
      for (int c = 0; c < SL - 1; c++) issue(c);
    }
  }
  __device__ __forceinline__ float run() const {
    float acc = 0.0f;
    if (wave >= 2) {
      // the barrier also frees the slot of chunk c - 1, which chunk c + SL - 1 takes
      for (int c = 0; c < nch; c++) {
        sk_sync<VI * (SL - 2)>();
        issue(c + SL - 1);
      }
      sk_wait<0>();
    } else if (sizeof(KT) == 2 && wave == 1) {
      acc = sum<1>();
    } else {
      acc = sum<0>();
    }
    lds_barrier();
    return acc;
  }
};

template <int HD, class KT>
__global__ __launch_bounds__(kHeadThreads, 2) void k_attn_head(const float* __restrict__ qkv, int QKV, int H, int KVH,
                                                               const KT* __restrict__ kc, const KT* __restrict__ vc,
                                                               int ctx, int end, int layer,
                                                               const int* __restrict__ pos, int B,
                                                               size_t seq_stride, uint4* __restrict__ xq, int xstride,
                                                               uint4* __restrict__ xh) {
  constexpr int NW = kHeadThreads / 64, RB = HD * (int)sizeof(KT), NP = RB / 128;   // bytes, 128-byte pieces of a row
  extern __shared__ __attribute__((aligned(16))) float lsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int G = H / KVH;
  const int L = blockIdx.x, unit = (L / kXcds / G) * kXcds + L % kXcds;
  if (unit >= B * KVH) return;
  // the rows of a prompt pass end later the higher they are: longest first
  const int g = unit % KVH, b = B - 1 - unit / KVH, h = g * G + (L / kXcds) % G;
  const int T = pos[b] + 1;
  unsigned char* const stage = reinterpret_cast<unsigned char*>(lsm);
  float* const e = lsm + kHeadStageBytes / 4;      // scores, then exponentials, then probabilities
  float* const red = e + head_row(end);
  const size_t cb = (size_t)b * seq_stride + ((size_t)layer * KVH + g) * ctx * HD;

  // ---- scores: wave w takes positions 64 c .. 64 c + 63 of the chunks c = w mod 4
  const unsigned char* const kb = reinterpret_cast<const unsigned char*>(kc + cb);
  unsigned char* const ring = stage + wave * 2 * kHeadStage;
  const int nch = (T + 63) >> 6, mine = nch > wave ? (nch - wave + NW - 1) / NW : 0;
  // lane l of a load instruction fills slot l & 7 of row l >> 3 (of 8), which holds piece (slot - row) mod 8
  const uint32_t kpiece = 16 * (((lane & 7) - (lane >> 3)) & 7);
  const int stages = mine * NP;
  auto issue = [&](int n) {                // stage n: piece n mod NP of the wave's chunk n / NP, 8 instructions
    const int t0 = 64 * (wave + NW * (n / NP)) + (lane >> 3);
    unsigned char* const d = ring + (n & 1) * kHeadStage;
    const unsigned char* const src = kb + 128 * (n % NP);
#pragma unroll
    for (int k = 0; k < 8; k++)            // rows past T - 1 repeat it and are never used
      head_dma16(src, (uint32_t)min(t0 + 8 * k, T - 1) * RB + kpiece, d + 1024 * k);
  };
  // q comes the same way, a copy for each wave: a plain load's wait inside the loop would wait for the
  // stage in flight as well
  float* const ql = red + 16 + wave * HD;
  const float* const qg = qkv + (size_t)b * QKV + h * HD;
#pragma unroll
  for (int u = 0; u < HD / 64; u++) sk_dma4(qg + 64 * u + lane, ql + 64 * u);
  float mx = -1e30f;
  const float scale = 1.0f / __builtin_sqrtf((float)HD);
  if (stages > 0) {
    issue(0);
    sk_wait<8>();
  } else {
    sk_wait<0>();
  }
  float qr[HD / 16];
#pragma unroll
  for (int u = 0; u < HD / 16; u++) qr[u] = ql[16 * u + (lane & 15)];
  for (int i = 0; i < mine; i++) {
    float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    auto piece = [&](auto stc) {
      constexpr int st = decltype(stc)::value, E = 128 / (int)sizeof(KT);   // elements of a row in a piece
      const int n = i * NP + st;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // the stage that is loaded next has been read
      if (n + 1 < stages) {
        issue(n + 1);
        sk_wait<8>();
      } else {
        sk_wait<0>();
      }
      const unsigned char* const row = ring + (n & 1) * kHeadStage + 128 * lane;
      typedef typename HeadVec<KT>::T V4;
      V4 k[E / 4];
#pragma unroll
      for (int p = 0; p < 8; p++) {
        const V4* v = reinterpret_cast<const V4*>(row + 16 * ((p + lane) & 7));
        if constexpr (sizeof(KT) == 2) {
          k[2 * p] = v[0];
          k[2 * p + 1] = v[1];
        } else {
          k[p] = v[0];
        }
      }
      head_dot<KT, st * E / 4, E / 4>::run(s, qr, k);
    };
    piece(std::integral_constant<int, 0>());
    if constexpr (NP > 1) piece(std::integral_constant<int, 1>());
    if constexpr (NP > 2) {
      piece(std::integral_constant<int, 2>());
      piece(std::integral_constant<int, 3>());
    }
    const int t = 64 * (wave + NW * i) + lane;
    const float sv = (s[0] + s[1] + s[2] + s[3]) * scale;
    if (t < T) {
      e[t] = sv;
      mx = __builtin_fmaxf(mx, sv);
    }
  }

  // ---- softmax
  mx = max64(mx);
  if (lane == 0) red[wave] = mx;
  lds_barrier();                           // every wave has read its last K stage

  HeadPv<HD, KT> pv(wave, lane, T, reinterpret_cast<const unsigned char*>(vc + cb), stage, e);
  pv.start();                              // V's first chunks load while the softmax runs
  mx = __builtin_fmaxf(__builtin_fmaxf(red[0], red[1]), __builtin_fmaxf(red[2], red[3]));
  for (int t = tid; t < T + ordered_run(T); t += kHeadThreads) e[t] = t < T ? fast_exp(e[t] - mx) : 0.0f;
  lds_barrier();
  if (wave == 0) {
    const float s = ordered_sum_wave(e, T);
    if (lane == 0) red[8] = s;
  }
  lds_barrier();
  const float sum = red[8];
  for (int t = tid; t < T; t += kHeadThreads) e[t] = e[t] / sum;
  lds_barrier();

  // ---- P.V
  const float acc = pv.run();

  // ---- the o projection's activation: the head's HD outputs as HD / 32 quantize_row blocks of row b
  float* const out = lsm;                  // the last barrier freed the slots
  if (wave < HD / 64) out[pv.column()] = acc;
  lds_barrier();
  if (tid < HD / 8) {
    const int blk = tid >> 2, j = tid & 3, base = 32 * blk + 2 * j;
    const float v[8] = {out[base],      out[base + 1],  out[base + 8],  out[base + 9],
                        out[base + 16], out[base + 17], out[base + 24], out[base + 25]};
    quantize_item(v, h * HD / 32 + blk, j, xq + (size_t)b * xstride * 4, xh ? xh + xh_tile(b, xstride) : nullptr, b & 15);
  }
}

}  // namespace q4
