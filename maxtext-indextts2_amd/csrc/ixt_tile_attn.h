// ixt_tile_attn.h -- prefill attention on the f32 matrix units, for pages of 32 tokens.
//
// v_mfma_f32_16x16x4_f32 (and v_mfma_f32_16x16x1_4b_f32, four blocks of one product) adds its four products to the accumulator one after the other, k ascending, each step one IEEE fma (subnormals kept): on
// 10^6 cells of random bf16 and f32 operands, down to subnormal sums, its result is the chain of four fmaf bit for bit.  So the contract's chains --
// a score is one fma chain over d, an output one fma chain over the tokens of a page -- run on it unchanged, at 140 TFLOP/s where the vector units'
// chains (k_attn_tile) reached 17.
#pragma once
#include "ixt_kernels.h"

#include <type_traits>

typedef float ixt_f32x4 __attribute__((ext_vector_type(4)));
typedef float ixt_f32x16 __attribute__((ext_vector_type(16)));

// rows 1 and 3 of `a` (16 lanes each) against rows 0 and 2 of `b` / the upper half of `a` against the lower half of `b`
__device__ __forceinline__ void ixt_swap16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0]; b = r[1];
}
__device__ __forceinline__ void ixt_swap32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0]; b = r[1];
}

// The scores of a super-block: 128 keys against 16 query vectors.  kp: token 4 lg + i16 % 4 of page i16 / 4 of it; q: the lane's vector in LDS.  Register 4 (t % 4) + r of half t / 4: token
// 4 t + r of the lane's page (page lg), vector i16.
template <int HD>
__device__ __forceinline__ void mtile_scores(const bf16_t* kp, const float* q, ixt_f32x16& S0, ixt_f32x16& S1) {
  constexpr int NB = HD / 32;
  u32x4 kr[2][8];
  auto fetch = [&](int k, int b) {
#pragma unroll
    for (int t = 0; t < 8; ++t) kr[k][t] = *reinterpret_cast<const u32x4*>(kp + b * 1024 + (t >> 1) * 256 + (t & 1) * 128);
  };
  auto products = [&](int k, int b) {              // 32 d of 128 keys, eight d's operands at a time: the scores need the registers
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float* qp = q + b * 32 + c * 8;
      const float4 q0 = *reinterpret_cast<const float4*>(qp), q1 = *reinterpret_cast<const float4*>(qp + 4);
      const float q8[8] = {q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w};
      float x[8], y[8];
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        x[s] = s & 1 ? bfhi(kr[k][2 * c][s >> 1]) : bflo(kr[k][2 * c][s >> 1]);
        y[s] = s & 1 ? bfhi(kr[k][2 * c + 1][s >> 1]) : bflo(kr[k][2 * c + 1][s >> 1]);
        asm volatile("" : "+v"(x[s]), "+v"(y[s]));
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < 8; ++s) {
        S0 = __builtin_amdgcn_mfma_f32_16x16x1f32(x[s], q8[s], S0, 0, 0, 0);
        S1 = __builtin_amdgcn_mfma_f32_16x16x1f32(y[s], q8[s], S1, 0, 0, 0);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  fetch(0, 0);
  fetch(1, 1);
#pragma unroll 1
  for (int b = 2; b < NB; b += 2) {                // the next 32 d fly while these are multiplied
    products(0, b - 2);
    fetch(0, b);
    products(1, b - 1);
    fetch(1, b + 1);
  }
  products(0, NB - 2);
  products(1, NB - 1);
}
// the soft cap of a super-block's scores
__device__ __forceinline__ void mtile_cap(ixt_f32x16& S0, ixt_f32x16& S1, float cap) {
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    S0[k] = ixt_tanh(S0[k] / cap) * cap;
    S1[k] = ixt_tanh(S1[k] / cap) * cap;
    if ((k & 1) == 1) __builtin_amdgcn_sched_barrier(0);
  }
}
// Where a launch's (kv head, tile) blocks leave half of the CUs idle, the scores go ahead of it in a launch of their own, a tile's super-blocks dealt among gridDim.z blocks, and
// k_attn_mtile<.., GIVEN> finds them in memory, 8 KiB a super-block, as its lanes hold them: two blocks that share a value's columns no longer take every score both (Gemma-2 2B, 3000
// tokens by 256: 22.1 ms of attention launches of more than 512 keys, now 7.2 of scores and 10.4 of values).  The rows of a tile are of one page group (the caller's promise: one segment), idle ones among them.
__device__ __forceinline__ size_t mscores_at(const TileAttnArgs& a, int tile, int kvh, int sb) {
  return (((size_t)tile * a.g.nkv + kvh) * ((a.lmax + 127) >> 7) + sb) * 2048;
}
template <int HD, int GQ>
__global__ __launch_bounds__(512, 2) void k_attn_mscores(TileAttnArgs a) {
  constexpr int TQ = 16 / GQ, QP = HD + 4, NW = 8;
  __shared__ __attribute__((aligned(16))) float qs[16 * QP];
  __shared__ int s_pos[TQ], s_slot[TQ];
  const AttnGeom& g = a.g;
  const int kvh = blockIdx.x, r0 = (gridDim.y - 1 - blockIdx.y) * TQ;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, i16 = lane & 15, lg = lane >> 4;
  if (tid < TQ) {
    const int r = r0 + tid;
    const bool ok = r < a.R && a.row_active[r] != 0;
    s_pos[tid] = ok ? a.row_pos[r] : -1;
    s_slot[tid] = ok ? a.row_slot[r] : -1;
  }
  for (int it = tid; it < 16 * (HD / 8); it += NW * 64) {
    const int v = it & 15, c = it >> 4;
    const u32x4 w = *reinterpret_cast<const u32x4*>(a.qbuf + ((size_t)min(r0 + v / GQ, a.R - 1) * g.nq + kvh * GQ + v % GQ) * HD + c * 8);
    float4* q = reinterpret_cast<float4*>(qs + v * QP + c * 8);
    q[0] = make_float4(bflo(w[0]), bfhi(w[0]), bflo(w[1]), bfhi(w[1]));
    q[1] = make_float4(bflo(w[2]), bfhi(w[2]), bflo(w[3]), bfhi(w[3]));
  }
  __syncthreads();
  int posmax = -1, slot = 0;
#pragma unroll
  for (int i = 0; i < TQ; ++i) {
    const int ps = __builtin_amdgcn_readfirstlane(s_pos[i]);
    if (ps >= 0 && ps < a.lmax && ps > posmax) { posmax = ps; slot = __builtin_amdgcn_readfirstlane(s_slot[i]); }
  }
  if (posmax < 0) return;
  const int pages_all = (posmax + 32) >> 5, nsb = (pages_all + IXT_SB - 1) / IXT_SB;
  const int32_t* prow = a.page_map + (size_t)slot * g.mpg;
  for (int sb = wave * gridDim.z + blockIdx.z; sb < nsb; sb += NW * gridDim.z) {
    ixt_f32x16 S0 = ixt_f32x16(0.0f), S1 = ixt_f32x16(0.0f);
    mtile_scores<HD>(a.kpages + kpage_off(g, prow[min(4 * sb + (i16 >> 2), pages_all - 1)], kvh, 0, 4 * lg + (i16 & 3)), qs + i16 * QP, S0, S1);
    if (a.cap > 0.0f) mtile_cap(S0, S1, a.cap);
    float4* sp = reinterpret_cast<float4*>(a.scores + mscores_at(a, r0 / TQ, kvh, sb)) + lane;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      sp[k * 64] = make_float4(S0[4 * k], S0[4 * k + 1], S0[4 * k + 2], S0[4 * k + 3]);
      sp[(4 + k) * 64] = make_float4(S1[4 * k], S1[4 * k + 1], S1[4 * k + 2], S1[4 * k + 3]);
    }
  }
}
// Buffers of the exchange: with two a round has one barrier (another one's sums are read while the next is written); one where there is one round, or where two
// would take a CU's second block away.
constexpr int mtile_buffers(int hd, int nw, int nr) { return nr > 1 && (nw == 8 || hd <= 128) ? 2 : 1; }
constexpr int mtile_width(int hd) { return hd >= 128 ? 128 : hd; }        // value columns of one output pass
constexpr size_t mtile_lds(int hd, int nw, int nr, int vw) { return (size_t)mtile_buffers(hd, nw, nr) * nw * 16 * (vw + 4) * 4; }
// block = (kv head, 16 query vectors = 16 / GQ consecutive rows x GQ heads), NW waves.  Super-block (4 pages, 128 keys) n NW + w belongs to wave w in
// round n; its 128 x 16 scores stay in that wave's registers from the score products to the output products, so the keys one block holds are
// 128 NW NR and nothing of them goes through LDS or memory.
//   Scores: matrix rows = keys, columns = query vectors, one d a step (16x16x1: four blocks of 16 keys, each with the operand of its own lane group).  Row i
//   of block b is token 4 t + i % 4 of page i / 4, t = b and 4 + b: a lane then holds the 32 tokens of ONE page (its 16-lane group) for one query vector, and
//   the page's sum of exponentials is a sum over its own registers, in order.  K is read once, 16 bytes a lane: eight d of the lane's own key, operands as they are
//   (with four d a step, 16x16x4, they had to change lanes first, 18 vector instructions for eight products instead of 8: 33.7 us of a block's 103 in <8, 4>, now 28, which is
//   the products' own time).  The query operand comes from LDS, 16 bytes for four steps.
//   Softmax: max over lanes and waves; page sums meet in LDS and every lane adds its vector's in page order.  e / l with one reciprocal per lane:
//   two corrections of the quotient give the correctly rounded one where no remainder is subnormal (e >= 2^-96); otherwise the divide itself.
//   Outputs: matrix rows = value columns, P as the other operand after a 4 x 4 transpose of lane groups and registers.  A lane's 16 bytes of V are 8
//   columns of one token: column 8 i + x belongs to row i of tile x.  Page chains start from zero, four pages add up in order; the super-blocks of a
//   round meet in LDS, where the thread that owns (vector, column) adds them in order: with two buffers there, one barrier a round (four, half of the columns at
//   a time, took 3 us more of the 103).
// A key that a row does not see has P = +0 (k_attn_tile says why that is exact); tokens past the end are re-reads of the last one.
// Rows of other page groups in the tile are worked off group by group, dealt among `shares` blocks.  grid = (kv heads, tiles, parts x shares): parts = 1 or
// the number of 128-column parts of a value (the two halves of head_dim 256 in two blocks, each taking the scores anew), shares = 1 or more, both for
// launches that leave CUs idle otherwise.
// Bound by the matrix units and the vector units TOGETHER: an f32 product and a vector instruction of the same SIMD take turns, whichever waves they belong to (products
// alone 150 TFLOP/s; one bf16 -> f32 conversion in front of each 116, eight in front of eight 129).  So what counts is vector instructions: operands of a
// step converted together, no mask where every row sees every key (sees_all; the selects of a score were a branch each), weights rounded and packed two at a time ahead
// of the transpose.  A block of <8, 4> at 3072 to 3900 keys: 4.1 us until the first scores, 28 scores, 12 maxima and exponentials, 5 weights, 43 outputs (their products: 27 and 27); the
// clock stays at 2.2 to 2.4 GHz.  Tried without gain: a priority for half of the waves; values by 16x16x1 products, too, four pages at a time from weights as they lie (286
// against 293 us at <= 3072 keys, but 403 against 375 at <= 3900 and 118 against 117 with heads of 256: the sums of four pages leave no registers); a whole page of values
// ahead (spills: 316 us).  Keys and values widened to f32 by a launch ahead: level up to 2048 keys.
// What the bound of two or three blocks a CU leaves no register for goes through scratch.  Registers spilled, heads of 128: <2, 1> 32, <8, 3> 23, <8, 4> 76; heads of 256: <8, 3> 33.
// Measured against k_attn_tile, 16 heads of 128, 1024 rows at <= 1024 / 2048 / 3072 keys 282 / 860 / 1143 us, before the scores' 16x16x1 products and the exchange with one barrier
// 92 / 212 / 310, now 87 / 198 / 293.  828 rows at <= 3900 keys 1496, 408, 375 us (63 TFLOP/s).  8 heads of 256 on 4, 256 rows at <= 1756 / 2756 keys: 88 / 131, 79 / 117 us.
// Prompts of <= 256 keys: two waves per block; with four, two of them had nothing to do (eight packed ones, 1525 rows: 90.2 us against 67.6).
// GIVEN: the scores are in memory (k_attn_mscores, the same rows)
template <int HD, int GQ, int NW, int NR, bool GIVEN = false, int VW = mtile_width(HD)>
__global__ __launch_bounds__(NW * 64, NR == 1 && NW <= 4 ? 3 : 2) void k_attn_mtile(TileAttnArgs a) {
  constexpr int TQ = 16 / GQ;
  constexpr int NE = VW / 16;                  // matrix tiles of them
  constexpr int OP = VW + 4, NTOT = 16 * VW / (NW * 64);       // a vector's pitch of the exchange; (vector, column) totals per thread
  constexpr int NBUF = mtile_buffers(HD, NW, NR);
  static_assert(16 % GQ == 0 && HD % VW == 0 && VW % 64 == 0 && VW <= 128, "tile geometry");
  constexpr int QP = HD + 4;                                             // a vector's pitch: 16 lanes read 16 bytes of 16 vectors without a bank conflict
  __shared__ __attribute__((aligned(16))) float qs[16 * QP];
  __shared__ float psum[NW * NR * 4 * 16];                               // [page][vector]
  __shared__ float wmax[NW * 16];
  extern __shared__ __attribute__((aligned(16))) float ob[];             // [buffer][wave][vector][columns]
  __shared__ int s_pos[TQ], s_slot[TQ];
  const AttnGeom& g = a.g;
  const int kvh = blockIdx.x, r0 = (gridDim.y - 1 - blockIdx.y) * TQ;    // the rows with the most keys first
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, i16 = lane & 15, lg = lane >> 4;
  const int part0 = blockIdx.z % a.parts, share = blockIdx.z / a.parts, shares = gridDim.z / a.parts;
  const int n_out = g.nq * HD;
  if (tid < TQ) {
    const int r = r0 + tid;
    const bool ok = r < a.R && a.row_active[r] != 0;
    s_pos[tid] = ok ? a.row_pos[r] : -1;
    s_slot[tid] = ok ? a.row_slot[r] : -1;
  }
  for (int it = GIVEN ? 16 * (HD / 8) : tid; it < 16 * (HD / 8); it += NW * 64) {
    const int v = it & 15, c = it >> 4;
    const u32x4 w = *reinterpret_cast<const u32x4*>(a.qbuf + ((size_t)min(r0 + v / GQ, a.R - 1) * g.nq + kvh * GQ + v % GQ) * HD + c * 8);
    float4* q = reinterpret_cast<float4*>(qs + v * QP + c * 8);
    q[0] = make_float4(bflo(w[0]), bfhi(w[0]), bflo(w[1]), bfhi(w[1]));
    q[1] = make_float4(bflo(w[2]), bfhi(w[2]), bflo(w[3]), bfhi(w[3]));
  }
  __syncthreads();
  unsigned pending = 0;
#pragma unroll
  for (int i = 0; i < TQ; ++i) {
    const bool act = __builtin_amdgcn_readfirstlane(s_pos[i]) >= 0;
    if (act) pending |= 1u << i;
    else if (r0 + i < a.R && blockIdx.z == 0) {          // idle row: zeros, as the per-row kernel writes
      for (int idx = tid; idx < GQ * HD; idx += NW * 64) a.out[xidx(r0 + i, kvh * GQ * HD + idx, n_out)] = 0;
    }
  }
  int turn = 0;                                          // whose group comes next
  while (pending != 0) {
    // the rows of the leader's page group
    const int lead = __builtin_ctz(pending);
    const int slot = __builtin_amdgcn_readfirstlane(s_slot[lead]);
    unsigned grp = 0;
    int posmax = -1, posmin = a.lmax;
#pragma unroll
    for (int i = 0; i < TQ; ++i) {
      const int ps_ = __builtin_amdgcn_readfirstlane(s_pos[i]), sl_ = __builtin_amdgcn_readfirstlane(s_slot[i]);
      const bool in = ((pending >> i) & 1u) && sl_ == slot && ps_ < a.lmax;
      if (in) { grp |= 1u << i; posmax = max(posmax, ps_); posmin = min(posmin, ps_); }
    }
    if (((grp >> lead) & 1u) == 0) {                     // the leader reaches beyond the keys a block holds (the caller's max_len guard prevents it): zeros
      if (blockIdx.z == 0)
        for (int idx = tid; idx < GQ * HD; idx += NW * 64) a.out[xidx(r0 + lead, kvh * GQ * HD + idx, n_out)] = 0;
      pending &= ~(1u << lead);
      continue;
    }
    pending &= ~grp;
    const bool mine = turn == share;
    turn = turn + 1 == shares ? 0 : turn + 1;
    if (!mine) continue;
    const int kv_all = posmax + 1, pages_all = (kv_all + 31) >> 5, nsb = (pages_all + IXT_SB - 1) / IXT_SB;
    const int32_t* prow = a.page_map + (size_t)slot * g.mpg;
    const int mypos = ((grp >> (i16 / GQ)) & 1u) ? s_pos[i16 / GQ] : -1;

    // every row of the group sees every key of the super-block (a vector of another group may see any: it is not stored)
    auto sees_all = [&](int sb) { return sb * 128 + 127 <= posmin && (a.window <= 0 || posmax - a.window < sb * 128); };

    // ---- scores
    ixt_f32x16 S[NR][2];                                 // register 4 (t % 4) + r of half t / 4: token 4 t + r of the lane's page
    float mx = -INFINITY, mn = INFINITY;
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      const int sb = n * NW + wave;
      S[n][0] = S[n][1] = ixt_f32x16(0.0f);
      if (sb < nsb) {
        if constexpr (GIVEN) {
          const float4* sp = reinterpret_cast<const float4*>(a.scores + mscores_at(a, r0 / TQ, kvh, sb)) + lane;
#pragma unroll
          for (int k = 0; k < 8; ++k) {
            const float4 v = sp[k * 64];
            S[n][k >> 2][4 * (k & 3)] = v.x; S[n][k >> 2][4 * (k & 3) + 1] = v.y; S[n][k >> 2][4 * (k & 3) + 2] = v.z; S[n][k >> 2][4 * (k & 3) + 3] = v.w;
          }
        } else {
          mtile_scores<HD>(a.kpages + kpage_off(g, prow[min(4 * sb + (i16 >> 2), pages_all - 1)], kvh, 0, 4 * lg + (i16 & 3)), qs + i16 * QP, S[n][0], S[n][1]);
          if (a.cap > 0.0f) mtile_cap(S[n][0], S[n][1], a.cap);
        }
        // lane (vector i16, group lg): register r of tile t is token 4 t + r of page 4 sb + lg
        const int lim = mypos - sb * 128 - lg * 32, lo = a.window > 0 ? lim - a.window : -1;
        auto range = [&](auto masked) {
#pragma unroll
          for (int t = 0; t < 8; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int k = 4 * t + r;
              mn = fminf(mn, S[n][t >> 2][4 * (t & 3) + r]);
              mx = fmaxf(mx, !masked.value || (k <= lim && k > lo) ? S[n][t >> 2][4 * (t & 3) + r] : -INFINITY);
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        };
        if (sees_all(sb)) range(std::false_type());
        else range(std::true_type());
      }
    }
    // ---- softmax
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    if (lane < 16) wmax[wave * 16 + lane] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < NW; ++w) mx = fmaxf(mx, wmax[w * 16 + i16]);
#pragma unroll
    for (int n = 0; n < NR; ++n) {
      const int sb = n * NW + wave;
      if (sb < nsb) {
        const int lim = mypos - sb * 128 - lg * 32, lo = a.window > 0 ? lim - a.window : -1;
        float sacc = 0.0f;
        auto exps = [&](auto masked) {
#pragma unroll
          for (int t = 0; t < 8; ++t) {
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int k = 4 * t + r;
              const float e = ixt_exp(S[n][t >> 2][4 * (t & 3) + r] - mx);
              S[n][t >> 2][4 * (t & 3) + r] = !masked.value || (k <= lim && k > lo) ? e : 0.0f;
              sacc = sacc + S[n][t >> 2][4 * (t & 3) + r];
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        };
        if (sees_all(sb)) exps(std::false_type());
        else exps(std::true_type());
        psum[(4 * sb + lg) * 16 + i16] = sacc;
      }
    }
    __syncthreads();
    float l = 0.0f;
    for (int p = 0; p < nsb * 4; p += 4) {
      const float s0 = psum[p * 16 + i16], s1 = psum[p * 16 + 16 + i16], s2 = psum[p * 16 + 32 + i16], s3 = psum[p * 16 + 48 + i16];
      l = l + s0; l = l + s1; l = l + s2; l = l + s3;
    }
    if (!(l > 0.0f)) l = 1.0f;                           // a vector of another group
    const float rl = 1.0f / l;
    uint32_t P[NR][8][2];                                // bf16 pairs: pages 2 k (low half) and 2 k + 1 of the super-block, token 4 t + lg
    const uint32_t half = (lg & 1) ? 0x07060302u : 0x05040100u;      // the lane group's token of either page
    auto weights = [&](auto quotient) {
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        if (n * NW + wave < nsb) {
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            // bf16 pairs of tokens of the lane's page -> pairs of pages, lane group = token
            uint32_t u = pack2(f2bf(quotient(S[n][t >> 2][4 * (t & 3) + 0])), f2bf(quotient(S[n][t >> 2][4 * (t & 3) + 1]))), v = pack2(f2bf(quotient(S[n][t >> 2][4 * (t & 3) + 2])), f2bf(quotient(S[n][t >> 2][4 * (t & 3) + 3])));
            ixt_swap32(u, v);                            // u: pages 0, 1, v: pages 2, 3; lane groups 0, 1: tokens 0 and 1, 2, 3: tokens 2 and 3
            uint32_t u1 = u, v1 = v;
            ixt_swap16(u, u1);
            ixt_swap16(v, v1);
            P[n][t][0] = __builtin_amdgcn_perm(u1, u, half);
            P[n][t][1] = __builtin_amdgcn_perm(v1, v, half);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
    };
    if (__any(mypos >= 0 && mn - mx < -66.0f)) weights([&](float e) { return e / l; });
    else weights([&](float e) {
      float q = e * rl;
      q = __builtin_fmaf(__builtin_fmaf(-q, l, e), rl, q);
      return __builtin_fmaf(__builtin_fmaf(-q, l, e), rl, q);
    });
    // ---- outputs
    for (int part = part0; part < HD / VW; part += a.parts) {
      float tot[NTOT];
      int nsb_t[NTOT];                                   // super-blocks of the total's row
#pragma unroll
      for (int k = 0; k < NTOT; ++k) {
        const int v = (tid + k * NW * 64) / VW;
        tot[k] = 0.0f;
        nsb_t[k] = ((grp >> (v / GQ)) & 1u) ? (((s_pos[v / GQ] + 32) >> 5) + IXT_SB - 1) / IXT_SB : 0;
      }
      const int nsb_min = (((posmin + 32) >> 5) + IXT_SB - 1) / IXT_SB;
#pragma unroll
      for (int n = 0; n < NR; ++n) {
        if (n * NW >= nsb) break;
        const int sb = n * NW + wave;
        ixt_f32x4 ss[NE];
#pragma unroll
        for (int x = 0; x < NE; ++x) ss[x] = ixt_f32x4(0.0f);
        if (sb < nsb) {
          const int np = min(IXT_SB, pages_all - sb * IXT_SB);
#pragma unroll
          for (int t = 0; t < 8; ++t) asm volatile("" : "+v"(P[n][t][0]), "+v"(P[n][t][1]));   // unpacked here, a step at a time, and not ahead of the loops
          u32x4 va[4], vb[4];
          auto fetch = [&](u32x4 (&v)[4], int p, int t0) {
            const char* vp = reinterpret_cast<const char*>(a.vpages + vpage_off(g, prow[p], kvh, 0) + part * VW);
            const int last = min(32, kv_all - p * 32) - 1;
            int at = lg;
            asm volatile("" : "+v"(at));                 // the addresses of this fetch only: ahead of the loops they would take the scores' registers
#pragma unroll
            for (int t = 0; t < 4; ++t) {
              const char* q = vp + (uint32_t)((min(4 * (t0 + t) + at, last) * HD + i16 * NE) * 2);
              if constexpr (NE == 8) v[t] = *reinterpret_cast<const u32x4*>(q);
              else { const uint2 w = *reinterpret_cast<const uint2*>(q); v[t].x = w.x; v[t].y = w.y; }
            }
          };
          fetch(va, sb * IXT_SB, 0);
#pragma unroll
          for (int pg = 0; pg < IXT_SB; ++pg) {
            if (pg < np) {
              const int p = sb * IXT_SB + pg;
              ixt_f32x4 acc[NE];
#pragma unroll
              for (int x = 0; x < NE; ++x) acc[x] = ixt_f32x4(0.0f);
              // a step's operands all ahead of its products: one right in front of its own takes two empty cycles more
              auto values = [&](const u32x4& v, float pv) {
                float f[NE];
#pragma unroll
                for (int x = 0; x < NE; ++x) {
                  f[x] = (x & 1) ? bfhi(v[x >> 1]) : bflo(v[x >> 1]);
                  asm volatile("" : "+v"(f[x]));
                }
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int x = 0; x < NE; ++x) acc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[x], pv, acc[x], 0, 0, 0);
              };
              fetch(vb, p, 4);
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const float pv = (pg & 1) ? bfhi(P[n][t][pg >> 1]) : bflo(P[n][t][pg >> 1]);
                values(va[t], pv);
                __builtin_amdgcn_sched_barrier(0);
              }
              if (pg + 1 < np) fetch(va, p + 1, 0);
              __builtin_amdgcn_sched_barrier(0);
#pragma unroll
              for (int t = 0; t < 4; ++t) {
                const float pv = (pg & 1) ? bfhi(P[n][4 + t][pg >> 1]) : bflo(P[n][4 + t][pg >> 1]);
                values(vb[t], pv);
                __builtin_amdgcn_sched_barrier(0);
              }
#pragma unroll
              for (int x = 0; x < NE; ++x)
#pragma unroll
                for (int r = 0; r < 4; ++r) ss[x][r] = ss[x][r] + acc[x][r];
            }
          }
        }
        // lane: vector i16, columns NE (4 lg + r) + x
        float* const buf = ob + (NBUF == 2 ? n & 1 : 0) * NW * 16 * OP;
        if (NBUF == 1) __syncthreads();
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
          for (int x = 0; x < NE; x += 4) *reinterpret_cast<float4*>(buf + (wave * 16 + i16) * OP + (4 * lg + r) * NE + x) = make_float4(ss[x][r], ss[x + 1][r], ss[x + 2][r], ss[x + 3][r]);
        __syncthreads();
        if ((n + 1) * NW <= nsb_min) {                   // every row has all of the round
#pragma unroll
          for (int k = 0; k < NTOT; ++k) {
            const int idx = tid + k * NW * 64, at = idx / VW * OP + idx % VW;
#pragma unroll
            for (int w = 0; w < NW; ++w) tot[k] = tot[k] + buf[w * 16 * OP + at];
          }
        } else {
#pragma unroll
          for (int k = 0; k < NTOT; ++k) {
            const int idx = tid + k * NW * 64, at = idx / VW * OP + idx % VW;
#pragma unroll
            for (int w = 0; w < NW; ++w)
              if (n * NW + w < nsb_t[k]) tot[k] = tot[k] + buf[w * 16 * OP + at];
          }
        }
      }
#pragma unroll
      for (int k = 0; k < NTOT; ++k) {
        const int idx = tid + k * NW * 64, v = idx / VW, c = idx % VW;
        if ((grp >> (v / GQ)) & 1u) a.out[xidx(r0 + v / GQ, (kvh * GQ + v % GQ) * HD + part * VW + c, n_out)] = f2bf(tot[k]);
      }
      if (NBUF == 2 && part + a.parts < HD / VW) __syncthreads();      // (the next part's first buffer may be this one's last)
    }
    __syncthreads();                                     // the LDS arrays are reused by the next group
  }
}
