// gemm_tile.h -- the Q4_0 projection of a prompt pass: 32 x 32 matrix-core tiles.
//
// Every output is accumulated exactly as matmul_q4 does (engine/kernels.c:200-229; gemm_sk.h states the
// arithmetic): four lane chains acc_j += f32(p_j) * (dw * dx) over the blocks in order, then ((a0 + a1) +
// a2) + a3.  What bounds a pass of many tokens is vector-ALU issue: a product and an addition per block,
// chain, row and token are the reference's rounding points (32 instructions per 16 x 16 tile and block
// with the four chains), the block scales dw * dx another 4; everything else is overhead.  gemm_sk.h's
// 16 x 16 tiles add 14: the weight operands (12) and scale conversions serve 16 tokens only.  Here p_j
// of 32 rows x 32 tokens is one v_mfma_f32_32x32x8_f16, whose k = 0..7 are just the 8 values of the
// chain: k = 0..3 (lanes 0..31) x_0..3 against n - 8, k = 4..7 (lanes 32..63) x_4..7 / 16 against
// 16 (n - 8); a nibble becomes fp16 1024 + n (1024 + 16 n, masked in place) by a byte permute, and a
// packed fp16 addition takes the 1032 (1152) off.  Products and partial sums are integers below 2^21.
// An operand costs 5 instructions per lane and serves 32 tokens: 5.4 per 16 x 16 tile and block instead
// of 13.5.  The operands are the first two quarters of each chain in the tiled layout of quantize_item;
// the offset quarters of the 16 x 16 encoding are not read.
#pragma once
#include "gemm_sk.h"
#include "kernels.h"

namespace q4 {

typedef _Float16 tile_h2 __attribute__((ext_vector_type(2)));
typedef float tile_f16 __attribute__((ext_vector_type(16)));

// The B operand of one weight word (8 nibbles of a block and chain) for lanes kg = 0 (low nibbles) and
// kg = 1 (high nibbles, times 16).
struct TileB {
  uint32_t mask;
  tile_h2 off;
  __device__ __forceinline__ explicit TileB(int kg) {
    mask = kg ? 0xF0F0F0F0u : 0x0F0F0F0Fu;
    off = __builtin_bit_cast(tile_h2, kg ? 0xE480E480u : 0xE408E408u);     // -1152, -1032
  }
  __device__ __forceinline__ sk_h4 operator()(uint32_t wv) const {
    const uint32_t v = wv & mask;
    const tile_h2 a = __builtin_bit_cast(tile_h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04010400u)) + off;
    const tile_h2 b = __builtin_bit_cast(tile_h2, __builtin_amdgcn_perm(0x64646464u, v, 0x04030402u)) + off;
    return (sk_h4){a[0], a[1], b[0], b[1]};
  }
};

// Register r of a 32 x 32 product holds token tile_token(r, kg) of weight row lane % 32.
__device__ __forceinline__ constexpr int tile_token(int r, int kg) { return (r & 3) + 8 * (r >> 2) + 4 * kg; }

// A workgroup takes 64 tokens and 64 / CS rows, wave (c, t) with CS = 1: rows 32 c.. and tokens 32 t..
// with all four chains; with CS = 2: all 32 rows, tokens 32 t.. and chains 2 c and 2 c + 1 (the chains
// meet in shared memory at the end).  A slot of the two-slot ring holds a group of 4 blocks: the 4 token
// tiles' operands (wave w loads tile w; 128 bytes of padding between tiles put the two tiles a wave
// reads together on different banks), their dx, the weight words and scales.  Computing a group takes
// longer than loading its successor, so two slots are enough.
template <int CS>
struct TileSlot {
  static constexpr int ROWS = 64 / CS, TILE = 4 * 1024 + 128, oDX = 4 * TILE, oQS = oDX + 1024, oSC = oQS + 64 * ROWS,
                       BYTES = oSC + 8 * ROWS;
};

template <int OP, int CS, int EPI>
__global__ __launch_bounds__(256, 3) void k_gemm_tile(Q4Mat W, const uint4* __restrict__ xt, int xstride,
                                                                   int M, float* __restrict__ y, int ldy,
                                                                   const float* __restrict__ bias, bool by_tile,
                                                                   uint4* __restrict__ xq_out,
                                                                   uint4* __restrict__ xh_out, int ffn, SkRope rp) {
  static_assert(EPI != 1 || CS == 1, "the SwiGLU epilogue needs gate and up rows in one workgroup");
  static_assert(EPI != 2 || (CS == 2 && OP == 1), "the RoPE epilogue is the 32-row bias projection");
  using S = TileSlot<CS>;
  constexpr int NC = 4 / CS, ROWS = S::ROWS;
  __shared__ __align__(16) unsigned char ring[2][S::BYTES];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int li = lane & 31, kg = lane >> 5, wc = wave & 1, wt = wave >> 1;
  const int wr = CS == 1 ? wc : 0, c0 = CS == 1 ? 0 : 2 * wc;
  const int nrg = EPI == 1 ? ffn / 32 : W.Np / ROWS;
  int rgi, T;
  if (!sk_place(blockIdx.x, nrg, (M + 63) / 64, by_tile, rgi, T)) return;
  const int R0 = EPI == 1 ? rgi * 32 : rgi * ROWS, ng = W.ng;
  // this wave's loads: token tile 4 T + wave (past the last one: the last), weight chain `wave`, the
  // scales of ROWS / 4 rows
  const uint4* const act = xt + (size_t)min(4 * T + wave, (M - 1) >> 4) * xstride * kXhBlock;
  const uint4* const asrc = act + (lane >> 4) * 32 + (lane & 15);          // chain lane / 16, its first 256 bytes
  const float* const dsrc = reinterpret_cast<const float*>(act + 128) + (size_t)(lane >> 4) * kXhBlock * 4 + (lane & 15);
  // local row -> matrix row; with the RoPE epilogue, rows 16 p .. 16 p + 15 of a head's first half and
  // the matching rows of its second half, so that a pair meets in lanes l and l ^ 16 of a wave
  auto row_of = [&](int l) {
    if constexpr (EPI == 2) {
      const int gpr = rp.hd >> 5, head = rgi / gpr, p = rgi - head * gpr;
      return head * rp.hd + (l < 16 ? 16 * p + l : (rp.hd >> 1) + 16 * p + l - 16);
    } else {
      return SkSrc<1>::row_of(R0, EPI == 1 ? ffn : 0, l);
    }
  };
  const int rq = row_of(lane & (ROWS - 1)), rs = row_of(ROWS / 4 * wave + ((lane >> 1) & (ROWS / 4 - 1)));
  const uint4* const qsrc = W.qs + ((size_t)(rq >> 6) * ng * 64 + (rq & 63)) * 4 + wave;
  const uint32_t* const ssrc =
      reinterpret_cast<const uint32_t*>(W.d + (size_t)(rs >> 6) * W.nb8 * 64 + (rs & 63)) + (lane & 1);
  auto issue = [&](unsigned char* slot, int g) {
#pragma unroll
    for (int k = 0; k < 4; k++)
      sk_dma16(asrc + (size_t)(4 * g + k) * kXhBlock, slot + wave * S::TILE + 1024 * k);
    sk_dma4(dsrc + (size_t)(4 * g) * kXhBlock * 4, slot + S::oDX + 256 * wave);
    if (lane < ROWS) sk_dma16(qsrc + (size_t)g * 256, slot + S::oQS + 16 * ROWS * wave);
    if (lane < ROWS / 2) sk_dma4(ssrc + (size_t)(g >> 1) * 256 + ((g & 1) << 1), slot + S::oSC + 2 * ROWS * wave);
  };
  const TileB bop(kg);
  float acc[NC][16];
#pragma unroll
  for (int c = 0; c < NC; c++)
#pragma unroll
    for (int r = 0; r < 16; r++) acc[c][r] = 0.0f;
  const bool work = 64 * T + 32 * wt < M;                     // a wave past the last token only loads
  // where the lane's operands lie in a slot
  const int oA = (2 * wt + (li >> 4)) * S::TILE + 256 * c0 + kg * 128 + (li & 15) * 8;
  const int oD = S::oDX + 512 * wt + 16 * kg, oW = S::oQS + 16 * (ROWS * c0 + 32 * wr + li), oS = S::oSC + 8 * (32 * wr + li);
  // A group's 4 NC products in order (block, chain), each formed one ahead of its update, its token
  // operand read two ahead; a block's token scales are read one block ahead.
  auto group = [&](const unsigned char* slot) {
    uint4 w[NC];
#pragma unroll
    for (int c = 0; c < NC; c++) w[c] = *reinterpret_cast<const uint4*>(slot + oW + 16 * ROWS * c);
    const uint2 sc = *reinterpret_cast<const uint2*>(slot + oS);
    constexpr int NI = 4 * NC;
    sk_h4 a[2];
    tile_f16 d[2];
    float4 dx[4];
    auto reada = [&](int i) { a[i & 1] = *reinterpret_cast<const sk_h4*>(slot + oA + 1024 * (i / NC) + 256 * (i % NC)); };
    auto readd = [&](int k) {
#pragma unroll
      for (int q = 0; q < 4; q++) dx[q] = *reinterpret_cast<const float4*>(slot + oD + 256 * (q >> 1) + 64 * k + 32 * (q & 1));
    };
    auto product = [&](int i) {
      const int k = i / NC;
      const uint4& wc4 = w[i % NC];
      const uint32_t wv = k == 0 ? wc4.x : k == 1 ? wc4.y : k == 2 ? wc4.z : wc4.w;
      d[i & 1] = __builtin_amdgcn_mfma_f32_32x32x8f16(a[i & 1], bop(wv), (tile_f16){}, 0, 0, 0);
    };
    float s[16];
    reada(0);
    readd(0);
    reada(1);
    product(0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < NI; i++) {
      const int k = i / NC, c = i % NC;
      if (c == 0) {
        const uint32_t sw = (k >> 1) == 0 ? sc.x : sc.y;
        const float dw = half_bits_to_float((k & 1) ? (sw >> 16) : (sw & 0xffffu));
#pragma unroll
        for (int q = 0; q < 4; q++) {
          s[4 * q] = dw * dx[q].x;
          s[4 * q + 1] = dw * dx[q].y;
          s[4 * q + 2] = dw * dx[q].z;
          s[4 * q + 3] = dw * dx[q].w;
        }
        if (k < 3) readd(k + 1);
      }
      if (i + 1 < NI) product(i + 1);
      if (i + 2 < NI) reada(i + 2);
#pragma unroll
      for (int r = 0; r < 16; r++) acc[c][r] = acc[c][r] + d[i & 1][r] * s[r];
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  issue(ring[0], 0);
  for (int g0 = 0; g0 < ng; g0 += 2) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int g = g0 + u;
      if (g < ng) {
        sk_sync<0>();                      // group g has landed; every wave has read group g - 1
        if (g + 1 < ng) issue(ring[u ^ 1], g + 1);
        if (work) group(ring[u]);
      }
    }
  }
  float v[16];                             // the four chains in the reference's order
  if constexpr (CS == 1) {
#pragma unroll
    for (int r = 0; r < 16; r++) v[r] = ((acc[0][r] + acc[1][r]) + acc[2][r]) + acc[3][r];
  } else {
    __syncthreads();
    float2* const red = reinterpret_cast<float2*>(ring) + wt * 1024 + lane;   // [wt][register][lane]: chains 2 and 3
    if (wc == 1) {
#pragma unroll
      for (int r = 0; r < 16; r++) red[64 * r] = make_float2(acc[0][r], acc[1][r]);
    }
    __syncthreads();
    if (wc == 1) return;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const float2 h = red[64 * r];
      v[r] = ((acc[0][r] + acc[1][r]) + h.x) + h.y;
    }
  }
  if constexpr (EPI == 1) {
    __syncthreads();
    constexpr int GS = 66;
    float* const gus = reinterpret_cast<float*>(ring);        // [token 64][local row 64]: gate 0..31, up 32..63
#pragma unroll
    for (int r = 0; r < 16; r++) gus[(32 * wt + tile_token(r, kg)) * GS + 32 * wr + li] = v[r];
    __syncthreads();
    const int t = tid >> 2, j = tid & 3, m = T * 64 + t;      // thread (token t, reference lane j)
    const int e[8] = {2 * j, 2 * j + 1, 8 + 2 * j, 9 + 2 * j, 16 + 2 * j, 17 + 2 * j, 24 + 2 * j, 25 + 2 * j};
    float g[8], u[8], act8[8];
#pragma unroll
    for (int k = 0; k < 8; k++) {
      g[k] = gus[t * GS + e[k]];
      u[k] = gus[t * GS + 32 + e[k]];
    }
    swiglu8(g, u, act8);
    if (m < M) quantize_item(act8, rgi, j, xq_out + (size_t)m * xstride * 4, xh_out + xh_tile(m, xstride), m & 15);
  } else if constexpr (EPI == 2) {
    // bias, RoPE at the token's position, q to y, k and v to the cache (kernels.c:337-352)
    const int row = row_of(li), hd = rp.hd, half = hd >> 1;
    const int head = row / hd, e = row - head * hd, i = e < half ? e : e - half;
    const float b = row < W.N ? bias[row] : 0.0f;
    const bool isv = head >= rp.H + rp.KVH;
    const size_t kvrow = ((size_t)rp.layer * rp.KVH + (head - rp.H - (isv ? rp.KVH : 0))) * rp.ctx;
#pragma unroll
    for (int r = 0; r < 16; r++) {
      const int m = T * 64 + 32 * wt + tile_token(r, kg);
      const float x = v[r] + b;
      const float xo = __shfl_xor(x, 16);                    // the pair's other value, same token
      if (m < M && row < W.N) {
        const int p = rp.pos[m];
        float out = x;
        if (!isv) {
          const float c = rp.rope[(size_t)p * hd + 2 * i], sn = rp.rope[(size_t)p * hd + 2 * i + 1];
          out = e < half ? x * c - xo * sn : x * c + xo * sn;
        }
        if (head < rp.H) {
          y[(size_t)m * ldy + row] = out;
        } else {
          const size_t off = (size_t)m * rp.seq_stride + (kvrow + p) * hd + e;
          void* cache = isv ? rp.vc : rp.kc;
          if (rp.kv16) reinterpret_cast<_Float16*>(cache)[off] = (_Float16)out;
          else reinterpret_cast<float*>(cache)[off] = out;
        }
      }
    }
  } else {
#pragma unroll
    for (int r = 0; r < 16; r++)
      sk_put<OP>(y, ldy, bias, M, W.N, T * 64 + 32 * wt + tile_token(r, kg), R0 + 32 * wr + li, v[r]);
  }
}

}  // namespace q4
