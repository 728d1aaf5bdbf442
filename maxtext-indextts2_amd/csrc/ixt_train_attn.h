// ixt_train_attn.h -- causal attention of the training step, heads of 64 and 128: scores, softmax and products in one launch forward, two backward.
//
// With a query head a kv head every number is the one that products and softmax through memory give (k_tgemm, k_t_softmax_*), bit for bit: the same products of 32 features or rows in the same
// order, the same exponentials, row sums in the same order, the same quotients.  (16 layers of bf16 carry any other last bit on to every gradient: with weights and sums rounded elsewhere, as precise, a
// step's gradients differed by as much as either is from 64 bits.)  With groups of query heads that holds for the outputs and the queries' gradients; dK and dV of a group are one chain of f32 sums
// over its heads here, a sum a head, added up in f32, there.
// Forward: a wave has 16 queries in registers and walks the keys, 64 at a time: S^T = K Q^T, so that a lane holds the scores of ONE query (four keys a register quad) and hands its
// weights to O^T += V^T P^T as they are.  Three walks: maxima; sums of exponentials; weights, which go to memory for the way back, and outputs.  Rows of at most 512 tokens are held and walked once.
// Backward: k_t_attn_dq is the same walk over P and dP = dO V^T, twice: the rows' sums, then dS, to memory, and dQ; k_t_attn_dkv the transposed one, a wave 16 N keys, of P and dS.
// What a walk need not look at: tiles beyond the diagonal, tiles in front of and behind the block's segments (ta_range; `reach` keeps them), and for a wave of one segment those of others: rows of
// padding see none of the tokens.
// What bounds it: forward, vector instructions: 17 a score for its exponential and the sum, 23 for the exponential, the least one and the quotient.  k_t_attn_dq: 0.35 GB of P twice and of dS once beside three
// products; k_t_attn_dkv the two of them once and two products.  LDS: stages of images of 64 (32) rows, filled by LDS-DMA a stage ahead, a barrier a stage.
// Measured (us a layer, forward / dP, softmax's gradient, dQ / dK, dV; a fifth of the rows padding), through memory, before, and now: 128 heads of 128 x 2048 tokens 1018 / 1035 / 382, 462 / 392 / 250 (the
// forward 449 before it looked for weights to divide); 48 heads of 64 x 512 43 / 37 / 17, 21 / 19 / 12.  In whole steps, whose rows
// are half to all tokens, 464 / 430 / 258 and 22 / 20 / 13.
//
// Image: 16-byte pieces, piece c of row r at c ^ ta_swizzle(r): 16 rows at one piece (ds_read_b128), and 8 rows at one pair of pieces (ds_read_tr16_b64, columns to
// lanes), lie on disjoint banks.  (Lanes step along a row by an exclusive or of addresses: the images lie at a multiple of 256 bytes, in front of everything else in LDS.)
#pragma once
#include "ixt_device.h"
#include "ixt_train_gemm.h"

struct TAttn {
  const bf16_t *q, *k, *v;                              // [B S][H D], [B S][KVH D]; features of q and k in the order of ta_place4
  const int32_t* seg;                                   // [B][S]: a query sees the keys of its segment up to itself
  bf16_t *P, *o;                                        // [B][H][S][ld], keys of 32 in the order of ta_place4; [B S][H D]
  int2* reach;                                          // [B][64]: the tiles of 64 keys whose weights the rows of a tile of 64 queries have in P and dS, first and last
  const bf16_t* d_o;
  bf16_t *dS, *dq, *dk, *dv;                            // as P, as q, k and v
  int B, S, H, KVH;
  long ld;
};
#define TA_MOST 4096                                    // tokens of a row (a word of 64 tiles)
#define TA_LDS_IMAGES(D, N) ((N) * 64 * (D) * 2)        // images of 64 rows
#define TA_LDS(D, N) (TA_LDS_IMAGES(D, N) + 32)         // behind them ta_range's words
#define TA_LDS_DKV(D, N) (2 * (2 * 32 * (D) * 2 + 2 * 32 * 64 * (N) * 2))   // two stages of 32 rows: queries, dO, P, dS
template <int D>
__device__ __forceinline__ int ta_swizzle(int row) {    // D / 8 pieces a row; of rows that share their low four bits it is the same
  return D == 128 ? (row & 7) << 1 | (row >> 3 & 1) : (row >> 1 & 3) << 1 | (row >> 3 & 1);
}
// Two images of 64 rows side by side, filled with rows of two tensors of one stride (elements); rows past S repeat the last one.  A wave fetches pieces 64 NJ wave + 64 j + lane: from
// one j to the next 4 (D 128) or 8 rows on, where the swizzle changes by a constant.
template <int D>
struct TaStage {
  static constexpr int IMG = 64 * D, PIECES = D / 8, NJ = 64 * PIECES / 256;
  const bf16_t *a, *b;
  int S, ld, row;
  uint32_t in, dst;
  __device__ __forceinline__ TaStage(const bf16_t* a_, const bf16_t* b_, int S_, int ld_, int wave, int lane, uint32_t lds0) : a(a_), b(b_), S(S_), ld(ld_) {
    row = (wave * NJ * 64 + lane) / PIECES;
    in = (uint32_t)((lane % PIECES) ^ ta_swizzle<D>(row)) << 4;
    dst = lds0 + (uint32_t)(wave * NJ * 1024);
  }
  __device__ __forceinline__ void fetch(int image, int row0) const {              // rows row0 .. of a, to one of the four images
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const uint32_t c = in ^ (D == 128 ? (uint32_t)((j & 1) << 7 | (j >> 1) << 4) : (uint32_t)(j << 4));
      lds_dma16(__builtin_amdgcn_readfirstlane(dst + (uint32_t)(image * IMG * 2 + j * 1024)), a, (uint32_t)min(row0 + row + j * (64 / PIECES), S - 1) * (uint32_t)(ld * 2) + c);
    }
  }
  __device__ __forceinline__ void fetch(int buf, int row0, int row1) const {      // rows row0 .. of a, row1 .. of b
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int r = row + j * (64 / PIECES);
      const uint32_t c = in ^ (D == 128 ? (uint32_t)((j & 1) << 7 | (j >> 1) << 4) : (uint32_t)(j << 4));
      const uint32_t to = __builtin_amdgcn_readfirstlane(dst + (uint32_t)(buf * 2 * IMG * 2 + j * 1024));
      lds_dma16(to, a, (uint32_t)min(row0 + r, S - 1) * (uint32_t)(ld * 2) + c);
      lds_dma16(to + IMG * 2, b, (uint32_t)min(row1 + r, S - 1) * (uint32_t)(ld * 2) + c);
    }
  }
};
// everything this wave has asked for is there, and it has read what it wanted of the other stage; then everyone's
__device__ __forceinline__ void ta_turn() {
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  lds_barrier();
}
// A value loaded in front of the turn, used behind the next fetches: the compiler, which counts its own loads only, would wait for it there, and with it for the fetches.
template <typename T> __device__ __forceinline__ void ta_here(T& v) { asm volatile("" : "+v"(v)); }
// Where a lane reads an image: its row's swizzled first piece as an operand row (lane r16, features 8 q .. of 32), and of an operand column (lane = column; reduction rows 4 q .. and 16 + 4 q ..,
// the order in which a lane holds two accumulator tiles).  Steps along a row are an exclusive or, made anew for each read (asm): kept, they are a dozen registers.
template <int D>
struct TaLane {
  uint32_t rows, rows4, cols;                           // bytes
  __device__ __forceinline__ TaLane(uint32_t lds0, int r16, int q) {
    const int row = 4 * q + (r16 >> 2), p = r16 & 3;
    rows = lds0 + (uint32_t)(r16 * D * 2 + ((q ^ ta_swizzle<D>(r16)) << 4));
    rows4 = lds0 + (uint32_t)(r16 * D * 2 + (((q >> 1) ^ ta_swizzle<D>(r16)) << 4) + (q & 1) * 8);
    cols = lds0 + (uint32_t)(row * D * 2 + (((p >> 1) ^ ta_swizzle<D>(row)) << 4) + (p & 1) * 8);
  }
};
typedef __attribute__((address_space(3))) tbf16x8* ta_p8;
typedef __attribute__((address_space(3))) tbf16x4* ta_p4;
template <typename P> __device__ __forceinline__ P ta_at(uint32_t a) { return (P)(uintptr_t)a; }
// 16 rows from 16 t on, features 32 ks ..; `at` TaLane's word, plus the image's
template <int D>
__device__ __forceinline__ tbf16x8 ta_rows(uint32_t at, int t, int ks) {
  uint32_t a = at;
  asm("" : "+v"(a));
  a ^= (uint32_t)(ks << 6);
  return *ta_at<ta_p8>(a + t * 16 * D * 2);
}
// the same with features 4 q .. and 16 + 4 q .. on a lane, as k_tgemm's products have them (at: TaLane's rows4)
template <int D>
__device__ __forceinline__ tbf16x8 ta_rows4(uint32_t at, int t, int ks) {
  uint32_t a = at;
  asm("" : "+v"(a));
  a ^= (uint32_t)(ks << 6);
  const tbf16x4 lo = *ta_at<ta_p4>(a + t * 16 * D * 2), hi = *ta_at<ta_p4>((a ^ 32u) + t * 16 * D * 2);
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// 16 columns from 16 t on, rows 32 s ..
template <int D>
__device__ __forceinline__ tbf16x8 ta_cols(uint32_t at, int t, int s) {
  uint32_t a = at;
  asm("" : "+v"(a));
  a ^= (uint32_t)(t << 5);
  const tbf16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(ta_at<ta_p4>(a + s * 32 * D * 2)), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(ta_at<ta_p4>(a + (s * 32 + 16) * D * 2));
  return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
}
// 16 rows in registers, as ta_rows gives them
template <int D>
__device__ __forceinline__ void ta_load(const bf16_t* p, long ld, int row, int S, int q, tbf16x8 (&f)[D / 32]) {
  const bf16_t* at = p + (long)min(row, S - 1) * ld + q * 8;
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks) f[ks] = *reinterpret_cast<const tbf16x8*>(at + ks * 32);
}
template <int D>
__device__ __forceinline__ void ta_load4(const bf16_t* p, long ld, int row, int S, int q, tbf16x8 (&f)[D / 32]) {      // (ta_rows4)
  const bf16_t* at = p + (long)min(row, S - 1) * ld + q * 4;
#pragma unroll
  for (int ks = 0; ks < D / 32; ++ks)
    f[ks] = __builtin_shufflevector(*reinterpret_cast<const tbf16x4*>(at + ks * 32), *reinterpret_cast<const tbf16x4*>(at + ks * 32 + 16), 0, 1, 2, 3, 4, 5, 6, 7);
}
__device__ __forceinline__ tf32x4 ta_mfma(const tbf16x8& a, const tbf16x8& b, const tf32x4& c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
__device__ __forceinline__ uint32_t ta_pack2(float lo, float hi) {      // one v_cvt_pk_bf16_f32
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef __bf16 b2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f2{lo, hi}, b2));
}
__device__ __forceinline__ tbf16x8 ta_pack(const tf32x4& a, const tf32x4& b) {
  return __builtin_bit_cast(tbf16x8, u32x4{ta_pack2(a[0], a[1]), ta_pack2(a[2], a[3]), ta_pack2(b[0], b[1]), ta_pack2(b[2], b[3])});
}
// ixt_exp of a number that is not positive: the same value by an instruction less (the whole number out of the sum's last bits instead of a conversion and a scaling)
__device__ __forceinline__ float ta_exp(float x) {
  x = fmaxf(x, -80.0f);
  const float u = x * 1.44269504088896340736f + 12582912.0f, n = u - 12582912.0f;     // 1.5 2^23: rounds to a whole number (no contraction: the product is rounded first)
  float r = __builtin_fmaf(n, -0.693145751953125f, x), p = 1.98412698412698412698e-4f;
  r = __builtin_fmaf(n, -1.42860682030941723212e-6f, r);
  p = __builtin_fmaf(p, r, 1.38888888888888888889e-3f);
  p = __builtin_fmaf(p, r, 8.33333333333333333333e-3f);
  p = __builtin_fmaf(p, r, 4.16666666666666666667e-2f);
  p = __builtin_fmaf(p, r, 1.66666666666666666667e-1f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  return __uint_as_float(__float_as_uint(p) + (__float_as_uint(u) << 23));
}
__device__ __forceinline__ void ta_store(bf16_t* to, const tf32x4& v) { *reinterpret_cast<uint2*>(to) = make_uint2(ta_pack2(v[0], v[1]), ta_pack2(v[2], v[3])); }
// over the four lane groups
__device__ __forceinline__ float ta_max4(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
// A row's sum in the order of the kernels that have a row of 256 threads (k_t_softmax_fwd): columns 256 apart one behind the other, those 32, 16, 8, 4, 2, 1 apart in turn, then the four runs
// of 64.  So tiles are taken four apart, one place of the four after the other (TaFour), a sum for each place of a tile (l); ta_run: one place's, over the lanes.
__device__ __forceinline__ float ta_run(const tf32x4& l0, const tf32x4& l1, const tf32x4& l2, const tf32x4& l3) {
  const tf32x4 a = (l0 + l2) + (l1 + l3);
  float d[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const auto x = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[i]), __float_as_uint(a[i]), false, false);
    const float y = __uint_as_float(x[0]) + __uint_as_float(x[1]);
    const auto z = __builtin_amdgcn_permlane16_swap(__float_as_uint(y), __float_as_uint(y), false, false);
    d[i] = __uint_as_float(z[0]) + __uint_as_float(z[1]);
  }
  return (d[0] + d[2]) + (d[1] + d[3]);
}
struct TaFour {
  int first, last, w, j;                                // tiles; the next one's place of the four, the next one (> last: none)
  __device__ __forceinline__ TaFour(int first_, int last_) : first(first_), last(last_), w(-1), j(last_ + 1) { step(); }
  __device__ __forceinline__ void step() {
    j += 4;
    while (j > last && w < 3) { ++w; j = first + ((w - first) & 3); }
  }
};
// Which tiles of 64 rows a block has to look at: of the rows [from, end), those between the first and the last whose segment is one of its own 64 rows' (own ..), or between two of them.
// Rows of padding, and packed rows, see little of what the causal mask leaves.  word: LDS, 8 words.
struct TaRange { int first, last; };                    // first > last: none
__device__ __forceinline__ TaRange ta_range(const int32_t* __restrict__ seg, int S, int own, int from, int end, int32_t* word) {
  const int tid = threadIdx.x, lane = tid & 63;
  int lo = seg[min(own + lane, S - 1)], hi = lo;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) { lo = min(lo, __shfl_xor(lo, off, 64)); hi = max(hi, __shfl_xor(hi, off, 64)); }
  int first = 0x7fffffff, last = -1;
#pragma unroll 8
  for (int r = from + tid; r < end; r += 256) {
    const int s = seg[r];
    if (s >= lo && s <= hi) { first = min(first, r); last = r; }
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) { first = min(first, __shfl_xor(first, off, 64)); last = max(last, __shfl_xor(last, off, 64)); }
  if (lane == 0) { word[tid >> 6] = first; word[4 + (tid >> 6)] = last; }
  __syncthreads();
  first = __builtin_amdgcn_readfirstlane(min(min(word[0], word[1]), min(word[2], word[3])));
  last = __builtin_amdgcn_readfirstlane(max(max(word[4], word[5]), max(word[6], word[7])));
  return TaRange{first >> 6, last >> 6};
}
// Block -> (head, tile): the tiles of a head on one XCD, whose L2 holds its keys and values; the longest walk first.  grid = 8 ceil(heads / 8) tiles
__device__ __forceinline__ bool ta_place(int heads, int tiles, int& head, int& nth) {
  const int y = blockIdx.x >> 3;
  const int every = (heads + 7) >> 3;
  head = y % every * 8 + (blockIdx.x & 7);
  nth = y / every;
  return head < heads;
}

#define TA_HELD 8                // tiles of keys whose scores a wave of 16 queries holds
enum { TA_NONE, TA_SOME, TA_ALL };
template <int D, bool HELD>
__global__ __launch_bounds__(256, HELD ? 2 : D == 64 ? 4 : 3) void k_t_attn_fwd(TAttn t) {
  constexpr int KS = D / 32, DT = D / 16, IMG = 64 * D;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];            // four images (HELD) or three, 8 words of ta_range
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, q = lane >> 4, S = t.S;
  int bh, nth;
  const int tiles = (S + 63) >> 6;
  if (!ta_place(t.B * t.H, tiles, bh, nth)) return;                       // whole block
  const int b = bh / t.H, h = bh - b * t.H, q0 = (tiles - 1 - nth) * 64, qw = q0 + wave * 16;
  const long ldq = (long)t.H * D, ldk = (long)t.KVH * D;
  const int32_t* seg = t.seg + (long)b * S;
  const long kv = (long)b * S * ldk + h / (t.H / t.KVH) * D;
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) bf16_t*)lds);
  const TaLane<D> at(lds0, r16, q);
  const int row = min(qw + r16, S - 1);
  tbf16x8 qf[KS];
  ta_load<D>(t.q + (long)b * S * ldq + h * D, ldq, row, S, q, qf);
  const int sq = seg[row], s0 = __builtin_amdgcn_readfirstlane(sq);
  const bool one = __all(sq == s0);                 // the wave's queries are of one segment
  const TaRange in = ta_range(seg, S, q0, 0, min(S, q0 + 64), reinterpret_cast<int32_t*>(lds + (HELD ? 4 : 3) * IMG));     // (a query's own key is one of them)
  // scores of the 64 keys from k0 on (`img`: their image), a segment a key a lane; who sees them, TA_SOME: bit 4 kt + i of `see` the lane's
  auto scores = [&](tf32x4 (&s)[4], uint32_t& see, uint32_t img, int k0, int sk) __attribute__((always_inline)) -> int {
    if (k0 > qw + 15 || (one && !__any(sk == s0))) return TA_NONE;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
      s[kt] = tf32x4(0.0f);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) s[kt] = ta_mfma(ta_rows<D>(at.rows + img, kt, ks), qf[ks], s[kt]);
    }
    if (one && __all(sk == s0) && k0 + 63 <= qw) return TA_ALL;
    see = 0;
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int key = kt * 16 + 4 * q + i, sg = __shfl(sk, key, 64);
        see |= k0 + key <= qw + r16 && sg == sq ? 1u << (kt * 4 + i) : 0u;
      }
    return TA_SOME;
  };
  auto unseen = [&](tf32x4 (&s)[4], uint32_t see, float with) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[kt][i] = see >> (kt * 4 + i) & 1u ? s[kt][i] : with;
  };
  float m = -INFINITY, sum = 0.0f, rsum;
  auto highest = [&](const tf32x4 (&s)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) m = fmaxf(fmaxf(fmaxf(fmaxf(m, s[kt][0]), s[kt][1]), s[kt][2]), s[kt][3]);      // (two instructions)
  };
  // least: a lane's least one (of keys that are not seen, too) as a word, whose order is that of numbers that are not negative
  auto exps = [&](tf32x4 (&s)[4], int& least) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[kt][i] = ta_exp(s[kt][i] - m);
        least = min(least, __float_as_int(s[kt][i]));
      }
  };
  const int most = 0x7fffffff;
  auto small = [](int least) __attribute__((always_inline)) { return __any(least < __float_as_int(0x1p-96f)); };
  tf32x4 o[DT];
#pragma unroll
  for (int d = 0; d < DT; ++d) o[d] = tf32x4(0.0f);
  bf16_t* const prow = t.P + ((long)bh * S + row) * t.ld + 8 * q;         // (to the end of the tile: zeros past the last key)
  const bool real = qw + r16 < S;
  // with a weight below 2^-96 among them they are divided, as k_t_softmax_fwd_wave has it (the quotient by 1 that follows changes nothing)
  auto divide = [&](tf32x4 (&s)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt)
#pragma unroll
      for (int i = 0; i < 4; ++i) s[kt][i] = s[kt][i] / sum;
  };
  auto zeros = [&](int k0) __attribute__((always_inline)) {
    if (real) *reinterpret_cast<u32x4*>(prow + k0) = *reinterpret_cast<u32x4*>(prow + k0 + 32) = u32x4(0u);
  };
  // weights of the tile of the keys from k0 on, and their product with its values.  The quotient by the reciprocal and two corrections, the last of which rounds as a division does where no residue
  // is lost below the normal numbers
  auto values = [&](tf32x4 (&s)[4], float by, float rby, uint32_t img, int k0) __attribute__((always_inline)) {
#pragma unroll
    for (int st = 0; st < 2; ++st) {
#pragma unroll
      for (int kt = 2 * st; kt < 2 * st + 2; ++kt)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float e = s[kt][i];
          float x = e * rby;
          x = __builtin_fmaf(__builtin_fmaf(-x, by, e), rby, x);
          s[kt][i] = __builtin_fmaf(__builtin_fmaf(-x, by, e), rby, x);
        }
      const tbf16x8 p = ta_pack(s[2 * st], s[2 * st + 1]);
      if (real) *reinterpret_cast<u32x4*>(prow + k0 + st * 32) = __builtin_bit_cast(u32x4, p);
#pragma unroll
      for (int d = 0; d < DT; ++d) o[d] = ta_mfma(ta_cols<D>(at.cols + img, d, st), p, o[d]);
    }
  };
  const TaStage<D> keys(t.k + kv, t.k + kv, S, (int)ldk, wave, lane, lds0);
  const int from = in.first & ~3;
  if constexpr (HELD) {
    {
      // all scores of the wave's rows at once, two tiles a stage
      const TaStage<D> vals(t.v + kv, t.v + kv, S, (int)ldk, wave, lane, lds0);
      tf32x4 s[TA_HELD][4];
      uint32_t see[TA_HELD];
      int who[TA_HELD];
      auto segs = [&](int j) __attribute__((always_inline)) { return seg[min(j * 64 + lane, S - 1)]; };
      int sa = segs(from), sb = segs(from + 1);
      keys.fetch(0, from * 64, from * 64 + 64);
#pragma unroll
      for (int p = 0; p < TA_HELD / 2; ++p) {
        const int j = from + p * 2;
        who[2 * p] = who[2 * p + 1] = TA_NONE;
        if (j > in.last) continue;
        ta_turn();
        int na = sa, nb = sb;
        ta_here(na); ta_here(nb);
        if (j + 2 <= in.last) {
          sa = segs(j + 2); sb = segs(j + 3);
          keys.fetch((p + 1) & 1, j * 64 + 128, j * 64 + 192);
        } else {
          vals.fetch((p + 1) & 1, from * 64, from * 64 + 64);
        }
        who[2 * p] = scores(s[2 * p], see[2 * p], (uint32_t)((p & 1) * 2 * IMG * 2), j * 64, na);
        who[2 * p + 1] = scores(s[2 * p + 1], see[2 * p + 1], (uint32_t)(((p & 1) * 2 + 1) * IMG * 2), j * 64 + 64, nb);
      }
#pragma unroll
      for (int j = 0; j < TA_HELD; ++j) {
        if (who[j] == TA_ALL) highest(s[j]);
        if (who[j] != TA_SOME) continue;
        tf32x4 seen[4] = {s[j][0], s[j][1], s[j][2], s[j][3]};           // (the scores stay: least would be that of -INFINITY)
        unseen(seen, see[j], -INFINITY);
        highest(seen);
      }
      m = ta_max4(m);
      int least = most;
#pragma unroll
      for (int j = 0; j < TA_HELD; ++j) {
        if (who[j] == TA_NONE) {
#pragma unroll
          for (int kt = 0; kt < 4; ++kt) s[j][kt] = tf32x4(0.0f);
        } else {
          exps(s[j], least);
          if (who[j] == TA_SOME) unseen(s[j], see[j], 0.0f);
        }
      }
      float run[4];
#pragma unroll
      for (int w = 0; w < 4; ++w) run[w] = ta_run(s[w][0] + s[w + 4][0], s[w][1] + s[w + 4][1], s[w][2] + s[w + 4][2], s[w][3] + s[w + 4][3]);
      sum = run[0] + run[1] + run[2] + run[3];
      if (__builtin_expect(small(least), false)) {
#pragma unroll
        for (int j = 0; j < TA_HELD; ++j) divide(s[j]);
        sum = 1.0f;
      }
      rsum = 1.0f / sum;
      const int vbuf = ((in.last - from) / 2 + 1) & 1;                    // the stage that the first values came to
#pragma unroll
      for (int p = 0; p < TA_HELD / 2; ++p) {
        const int j = from + p * 2, buf = (vbuf + p) & 1;
        if (j > in.last) continue;
        ta_turn();
        if (j + 2 <= in.last) vals.fetch(buf ^ 1, j * 64 + 128, j * 64 + 192);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          if (j + u < in.first || j + u > in.last) continue;              // (in front of and behind what is kept)
          if (who[2 * p + u] == TA_NONE) zeros(j * 64 + u * 64);
          else values(s[2 * p + u], sum, rsum, (uint32_t)((buf * 2 + u) * IMG * 2), j * 64 + u * 64);
        }
      }
    }
  } else {
    tf32x4 s[4];
    uint32_t see;
    int sk = seg[min(in.first * 64 + lane, S - 1)];
    keys.fetch(0, in.first * 64);
    for (int j = in.first; j <= in.last; ++j) {                           // maxima
      const int img = (j - in.first) & 1;
      ta_turn();
      int now = sk;
      ta_here(now);
      if (j < in.last) {
        sk = seg[min(j * 64 + 64 + lane, S - 1)];
        keys.fetch(img ^ 1, j * 64 + 64);
      }
      const int who = scores(s, see, (uint32_t)(img * IMG * 2), j * 64, now);
      if (who == TA_SOME) unseen(s, see, -INFINITY);
      if (who != TA_NONE) highest(s);
    }
    m = ta_max4(m);
    ta_turn();                                                            // (the last stage is read out)
    tf32x4 l[4] = {tf32x4(0.0f), tf32x4(0.0f), tf32x4(0.0f), tf32x4(0.0f)};
    TaFour ask(in.first, in.last), now = ask;                             // sums
    sk = seg[min(ask.j * 64 + lane, S - 1)];
    keys.fetch(0, ask.j * 64);
    for (int img = 0; now.j <= in.last; img ^= 1) {
      ta_turn();
      const int k0 = now.j * 64, w = now.w;
      int skj = sk;
      ta_here(skj);
      ask.step();
      if (ask.j <= in.last) {
        sk = seg[min(ask.j * 64 + lane, S - 1)];
        keys.fetch(img ^ 1, ask.j * 64);
      }
      const int who = scores(s, see, (uint32_t)(img * IMG * 2), k0, skj);
      if (who != TA_NONE) {
        int least;
        exps(s, least = most);
        if (who == TA_SOME) unseen(s, see, 0.0f);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) l[kt] += s[kt];
      }
      now = ask;
      if (now.w != w || now.j > in.last) {
        sum += ta_run(l[0], l[1], l[2], l[3]);
#pragma unroll
        for (int kt = 0; kt < 4; ++kt) l[kt] = tf32x4(0.0f);
      }
    }
    ta_turn();
    rsum = 1.0f / sum;
    // weights: keys and values one behind the other through three images, the next but one on its way
    const TaStage<D> vals(t.v + kv, t.v + kv, S, (int)ldk, wave, lane, lds0);
    sk = seg[min(in.first * 64 + lane, S - 1)];
    keys.fetch(0, in.first * 64);
    vals.fetch(1, in.first * 64);
    int img = 0;
    for (int j = in.first; j <= in.last; ++j) {
      const int k0 = j * 64;
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(TaStage<D>::NJ) : "memory");     // the keys (the values behind them are on their way)
      lds_barrier();
      const int v = img == 2 ? 0 : img + 1, next = v == 2 ? 0 : v + 1;
      int skj = sk;
      ta_here(skj);
      if (j < in.last) keys.fetch(next, k0 + 64);
      const int who = scores(s, see, (uint32_t)(img * IMG * 2), k0, skj);
      int least = most;
      if (who != TA_NONE) exps(s, least);
      if (who == TA_SOME) unseen(s, see, 0.0f);
      const bool divided = small(least);
      if (__builtin_expect(divided, false)) divide(s);
      if (j < in.last) {
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(TaStage<D>::NJ) : "memory");   // the values
        lds_barrier();
        sk = seg[min(k0 + 64 + lane, S - 1)];
        vals.fetch(img, k0 + 64);
      } else {
        ta_turn();
      }
      if (who == TA_NONE) zeros(k0);
      else values(s, divided ? 1.0f : sum, divided ? 1.0f : rsum, (uint32_t)(v * IMG * 2), k0);
      img = next;
    }
  }
  if (h == 0 && tid == 0) t.reach[b * 64 + q0 / 64] = make_int2(in.first, in.last);
  if (!real) return;
  bf16_t* const to = t.o + ((long)b * S + row) * ldq + h * D + 4 * q;
#pragma unroll
  for (int d = 0; d < DT; ++d) ta_store(to + d * 16, o[d]);
}

// dS = P o (dP - sum over the row of dP o P), dP = dO V^T, and dQ = dS K.  Two walks: the rows' sums, then dS.
template <int D, int N>
__global__ __launch_bounds__(256, 2) void k_t_attn_dq(TAttn t) {
  constexpr int KS = D / 32, DT = D / 16, IMG = 64 * D;
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];            // four images
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, q = lane >> 4, S = t.S;
  int bh, nth;
  const int tiles = (S + 64 * N - 1) / (64 * N);
  if (!ta_place(t.B * t.H, tiles, bh, nth)) return;                       // whole block
  const int b = bh / t.H, h = bh - b * t.H, q0 = (tiles - 1 - nth) * (64 * N), qw = q0 + wave * 16 * N;
  const long ldq = (long)t.H * D, ldk = (long)t.KVH * D, qat = (long)b * S * ldq + h * D;
  const int32_t* seg = t.seg + (long)b * S;
  const long kv = (long)b * S * ldk + h / (t.H / t.KVH) * D;
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) bf16_t*)lds);
  const TaLane<D> at(lds0, r16, q);
  tbf16x8 gf[N][KS];
  int sq[N];
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int row = min(qw + n * 16 + r16, S - 1);
    ta_load4<D>(t.d_o + qat, ldq, row, S, q, gf[n]);
    sq[n] = seg[row];
  }
  const int s0 = __builtin_amdgcn_readfirstlane(sq[0]);
  const bool one = __all(sq[0] == s0 && sq[N - 1] == s0);
  // what the rows have: of the wave's 64 queries, and of the block's
  const int2* const reach = t.reach + b * 64 + q0 / 64;
  const int2 first = reach[0], second = N == 2 && q0 + 64 < S ? reach[1] : first, own = N == 2 && wave >= 2 ? second : first;
  const TaRange in{min(first.x, second.x), max(first.y, second.y)};
  const long at_row = (long)bh * S * t.ld + 8 * q;
  struct Tile { int seg; u32x4 p[N][2]; };                                // a key's segment a lane, the lane's weights
  auto ask = [&](int k0) __attribute__((always_inline)) -> Tile {
    Tile x;
    x.seg = seg[min(k0 + lane, S - 1)];
#pragma unroll
    for (int n = 0; n < N; ++n)
#pragma unroll
      for (int st = 0; st < 2; ++st) x.p[n][st] = *reinterpret_cast<const u32x4*>(t.P + at_row + min(qw + n * 16 + r16, S - 1) * t.ld + k0 + st * 32);
    return x;
  };
  auto here = [&](Tile& x) __attribute__((always_inline)) {
    ta_here(x.seg);
#pragma unroll
    for (int n = 0; n < N; ++n) { ta_here(x.p[n][0]); ta_here(x.p[n][1]); }
  };
  // do the rows have the tile, and do queries of the wave see a key of it
  auto has = [&](int j) __attribute__((always_inline)) -> bool { return j >= own.x && j <= own.y; };
  auto sees = [&](const Tile& x, int j) __attribute__((always_inline)) -> bool { return has(j) && j * 64 <= qw + 16 * N - 1 && !(one && !__any(x.seg == s0)); };
  auto put = [&](int n, int col, const u32x4& w) __attribute__((always_inline)) {
    const int row = qw + n * 16 + r16;
    if (row < S) *reinterpret_cast<u32x4*>(t.dS + at_row + row * t.ld + col) = w;
  };
  tf32x4 g[4][N];
  auto grads = [&](uint32_t img) __attribute__((always_inline)) {
#pragma unroll
    for (int kt = 0; kt < 4; ++kt) {
#pragma unroll
      for (int n = 0; n < N; ++n) g[kt][n] = tf32x4(0.0f);
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const tbf16x8 f = ta_rows4<D>(at.rows4 + img, kt, ks);
#pragma unroll
        for (int n = 0; n < N; ++n) g[kt][n] = ta_mfma(f, gf[n][ks], g[kt][n]);
      }
    }
  };
  float dot[N];
#pragma unroll
  for (int n = 0; n < N; ++n) dot[n] = 0.0f;
  {
    tf32x4 l[4][N];
    auto clear = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int kt = 0; kt < 4; ++kt)
#pragma unroll
        for (int n = 0; n < N; ++n) l[kt][n] = tf32x4(0.0f);
    };
    clear();
    const TaStage<D> vals(t.v + kv, t.v + kv, S, (int)ldk, wave, lane, lds0);
    TaFour next(in.first, in.last), now = next;
    Tile x = ask(next.j * 64);
    vals.fetch(0, next.j * 64);
    for (int img = 0; now.j <= in.last; img ^= 1) {
      ta_turn();
      Tile y = x;
      here(y);
      const int j = now.j, w = now.w;
      next.step();
      if (next.j <= in.last) {
        x = ask(next.j * 64);
        vals.fetch(img ^ 1, next.j * 64);
      }
      if (sees(y, j)) {
        grads((uint32_t)(img * IMG * 2));
#pragma unroll
        for (int kt = 0; kt < 4; ++kt)
#pragma unroll
          for (int n = 0; n < N; ++n) {
            const uint32_t lo = y.p[n][kt >> 1][2 * (kt & 1)], hi = y.p[n][kt >> 1][2 * (kt & 1) + 1];
            l[kt][n] += g[kt][n] * tf32x4{bflo(lo), bfhi(lo), bflo(hi), bfhi(hi)};
          }
      }
      now = next;
      if (now.w != w || now.j > in.last) {
#pragma unroll
        for (int n = 0; n < N; ++n) dot[n] += ta_run(l[0][n], l[1][n], l[2][n], l[3][n]);
        clear();
      }
    }
    ta_turn();                                                            // (the last stage is read out)
  }
  tf32x4 dq[DT][N];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int n = 0; n < N; ++n) dq[d][n] = tf32x4(0.0f);
  const TaStage<D> both(t.k + kv, t.v + kv, S, (int)ldk, wave, lane, lds0);
  Tile x = ask(in.first * 64);
  both.fetch(0, in.first * 64, in.first * 64);
  for (int j = in.first; j <= in.last; ++j) {
    const int k0 = j * 64, buf = (j - in.first) & 1;
    ta_turn();
    Tile y = x;
    here(y);
    if (j < in.last) {
      x = ask(k0 + 64);
      both.fetch(buf ^ 1, k0 + 64, k0 + 64);
    }
    const uint32_t img = (uint32_t)(buf * 2 * IMG * 2);
    if (!sees(y, j)) {
      if (has(j)) {
#pragma unroll
        for (int n = 0; n < N; ++n) { put(n, k0, u32x4(0u)); put(n, k0 + 32, u32x4(0u)); }
      }
      continue;
    }
    grads(img + IMG * 2);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      u32x4 w[N];
#pragma unroll
      for (int n = 0; n < N; ++n) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {                                     // (two keys a word)
          const uint32_t p = y.p[n][st][i];
          const tf32x4& x = g[2 * st + (i >> 1)][n];
          w[n][i] = ta_pack2(bflo(p) * (x[2 * (i & 1)] - dot[n]), bfhi(p) * (x[2 * (i & 1) + 1] - dot[n]));
        }
        put(n, k0 + st * 32, w[n]);
      }
#pragma unroll
      for (int d = 0; d < DT; ++d) {
        const tbf16x8 f = ta_cols<D>(at.cols + img, d, st);
#pragma unroll
        for (int n = 0; n < N; ++n) dq[d][n] = ta_mfma(f, __builtin_bit_cast(tbf16x8, w[n]), dq[d][n]);
      }
    }
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int row = qw + n * 16 + r16;
    if (row >= S) continue;
    bf16_t* const to = t.dq + qat + (long)row * ldq + 4 * q;
#pragma unroll
    for (int d = 0; d < DT; ++d) ta_store(to + d * 16, dq[d][n]);
  }
}

// dV = P^T dO and dK = dS^T Q, a wave 16 N keys: both of a tile's operands by columns (ds_read_tr16).  Stages of 32 queries, from the diagonal on, of the tiles that the rows have; the query heads
// of a group one behind the other.
template <int D, int N>
__global__ __launch_bounds__(256, 2) void k_t_attn_dkv(TAttn t) {
  constexpr int DT = D / 16, IMG = 32 * D * 2, KEYS = 64 * N, PIMG = 32 * KEYS * 2, STAGE = 2 * IMG + 2 * PIMG;      // bytes
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];            // [2 stages][queries | dO | P | dS], 32 rows each
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, q = lane >> 4, S = t.S;
  int bh, nth;
  if (!ta_place(t.B * t.KVH, (S + KEYS - 1) / KEYS, bh, nth)) return;     // whole block
  const int G = t.H / t.KVH, b = bh / t.KVH, kvh = bh - b * t.KVH, k0 = nth * KEYS;
  const long ldq = (long)t.H * D, ldk = (long)t.KVH * D;
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) bf16_t*)lds);
  const uint32_t cols = TaLane<D>(lds0, r16, q).cols, pcols = TaLane<KEYS>(lds0, r16, q).cols;
  // query tiles whose rows have one of the block's key tiles, and those that have the wave's
  const int2 has = t.reach[b * 64 + lane];
  const int nt = (S + 63) >> 6, mine = N == 2 ? nth * 2 + (wave >> 1) : nth;
  const bool in = lane < nt;
  unsigned long long every = __ballot(in && lane >= nth * N && has.y >= nth * N && has.x <= nth * N + N - 1);
  const unsigned long long own = __ballot(in && lane >= mine && has.y >= mine && has.x <= mine);
  tf32x4 dk[DT][N], dv[DT][N];
#pragma unroll
  for (int d = 0; d < DT; ++d)
#pragma unroll
    for (int n = 0; n < N; ++n) dk[d][n] = dv[d][n] = tf32x4(0.0f);
  // 32 rows of four tensors: 16-byte pieces as in TaStage
  constexpr int PC = D / 8, NJ = 32 * PC / 256, PP = KEYS / 8, PJ = 32 * PP / 256;
  const int row = (wave * NJ * 64 + lane) / PC, prow = (wave * PJ * 64 + lane) / PP;
  const uint32_t piece = (uint32_t)((lane % PC) ^ ta_swizzle<D>(row)) << 4, ppiece = (uint32_t)((lane % PP) ^ ta_swizzle<KEYS>(prow)) << 4;
  const uint32_t keep = (uint32_t)(min(k0 + KEYS, (int)t.ld) - k0) * 2 - 16;      // the last piece of a row of P (past it: this one, for keys past the end)
  auto fetch = [&](int buf, int row0, int h) __attribute__((always_inline)) {
    const bf16_t *fq = t.q + (long)b * S * ldq + h * D, *fg = t.d_o + (long)b * S * ldq + h * D;
    const long at = ((long)b * t.H + h) * S * t.ld + k0;
    const uint32_t to = lds0 + (uint32_t)(buf * STAGE);
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const uint32_t off = (uint32_t)min(row0 + row + j * (64 / PC), S - 1) * (uint32_t)(ldq * 2) + (piece ^ (uint32_t)(j << 7));
      const uint32_t dst = __builtin_amdgcn_readfirstlane(to + (uint32_t)((wave * NJ + j) * 1024));
      lds_dma16(dst, fq, off);
      lds_dma16(dst + IMG, fg, off);
    }
#pragma unroll
    for (int j = 0; j < PJ; ++j) {
      const uint32_t off = (uint32_t)min(row0 + prow + j * (64 / PP), S - 1) * (uint32_t)(t.ld * 2) + min(ppiece ^ (uint32_t)(j << 7), keep);
      const uint32_t dst = __builtin_amdgcn_readfirstlane(to + (uint32_t)(2 * IMG + (wave * PJ + j) * 1024));
      lds_dma16(dst, t.P + at, off);
      lds_dma16(dst + PIMG, t.dS + at, off);
    }
  };
  for (int g = 0; g < G && every != 0; ++g) {
    const int h = kvh * G + g;
    unsigned long long left = every;
    int next = __builtin_ctzll(left), buf = 0;
    fetch(0, next * 64, h);
    while (left != 0) {
      const int tile = next;
      left &= left - 1;
#pragma unroll
      for (int half = 0; half < 2; ++half) {
        const int row0 = tile * 64 + half * 32;
        ta_turn();
        if (half == 0) {
          fetch(buf ^ 1, row0 + 32, h);
        } else if (left != 0) {
          next = __builtin_ctzll(left);
          fetch(buf ^ 1, next * 64, h);
        }
        if (own >> tile & 1) {
          const uint32_t img = (uint32_t)(buf * STAGE);
          tbf16x8 p[N], ds[N];
#pragma unroll
          for (int n = 0; n < N; ++n) {
            p[n] = ta_cols<KEYS>(pcols + img + 2 * IMG, wave * N + n, 0);
            ds[n] = ta_cols<KEYS>(pcols + img + 2 * IMG + PIMG, wave * N + n, 0);
            if (row0 + 32 > S) {                                          // rows past the end weigh nothing
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (row0 + (i >> 2) * 16 + 4 * q + (i & 3) >= S) p[n][i] = ds[n][i] = 0;
            }
          }
#pragma unroll
          for (int d = 0; d < DT; ++d) {
            const tbf16x8 f = ta_cols<D>(cols + img + IMG, d, 0), u = ta_cols<D>(cols + img, d, 0);
#pragma unroll
            for (int n = 0; n < N; ++n) { dv[d][n] = ta_mfma(f, p[n], dv[d][n]); dk[d][n] = ta_mfma(u, ds[n], dk[d][n]); }
          }
        }
        buf ^= 1;
      }
    }
    ta_turn();                                                            // (the last stage is read out)
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    const int at = (wave * N + n) * 16 + r16, key = k0 + (at & ~31) + ((at >> 3 & 3) + 4 * (at >> 2 & 1)) * 4 + (at & 3);      // (P's order of keys)
    if (key >= S) continue;
    const long to = ((long)b * S + key) * ldk + kvh * D + 4 * q;
#pragma unroll
    for (int d = 0; d < DT; ++d) { ta_store(t.dk + to + d * 16, dk[d][n]); ta_store(t.dv + to + d * 16, dv[d][n]); }
  }
}
