// ixt_train_gemm.h -- the matrix products of the training step: C[m][n] (+)= sum_k A(m, k) B(k, n), bf16 operands of which either index may be the
// contiguous one, f32 accumulation.
//
// Block = (16 MI WM) x (16 NI WN), waves WM x WN, 32 k at a time through a ring of NS LDS slots (one more for pairs, below) filled by LDS-DMA; a wave's tile is 16 MI x 16 NI.
// What bounds it: the matrix units at the clock that the card's power leaves them.  Random operands, 256 x 256 blocks: 1068 cycles of products per 32 k, 1136 with the
// LDS reads and the fetches beside them and nothing else (1.55 PFLOP/s at 1.64 GHz), 1340 to 1450 here at 1.5 to 1.8 GHz.  Per 32 k a wave reads MI + NI KiB for MI NI products of
// 16 cycles, which is why the largest block is taken wherever its tiles fill the chip.  With few tiles a wave is alone on its SIMD and bound by its own instructions: smaller tiles,
// more waves (gemm_launch has the rule).  So what counts is what stands between the products:
//   the next 32 k are read from LDS and fetched from memory between the rows of products, not in front of them;
//   the steps that fetch whole chunks are a loop of their own without a branch (a branch a fetch: 1515 cycles instead of 1400);
//   the block's barrier stands behind a step's first products, which cover the last reads and the waves' skew (2 to 4 % of long reductions);
//   a row of 32 k is half a line of 128 bytes: where an operand's k is contiguous (PAIR), both halves are fetched one behind the other, every second step, so that the second comes
//   from the L1 (fetches alone 593 cycles per 32 KiB, 1110 with the halves a step apart; five slots instead of four).
// Measured (us, with a launch's start and end), before these three and the stores of 16 bytes / now: 4096 x 4096, K 8192, k contiguous 232 / 205, of one operand 243 / 229, by columns 231 / 216;
// 16384 x 8192, K 2048 531 / 477; 128 x 128 blocks, 4096 x 2048, K 4096 86 / 68; 64 x 64, 2048 x 768, K 4096 31.8 / 26.8.
//   k contiguous:   slot image [row][32 k], four 16-byte pieces a row, piece c of row r at c ^ ((r >> 2) & 3): the 16 rows a half wave reads lie on
//                   disjoint banks
//   row contiguous: slot image [k][row], 32-byte pieces, piece u of row k at u ^ (k & 7) (64 rows: u ^ (k / 2 & 3)); ds_read_tr16 hands a 4 x 16 block to 16 lanes column-wise, so
//                   the transpose costs nothing; the eight k rows a half wave touches lie on disjoint banks
// Both put k = 4 q .. 4 q + 3 and 16 + 4 q .. on lane group q, 32 k after 32 k into one accumulator .  A piece past
// K comes from a zeroed word instead, a row past M or N is a re-read of a valid one (its results are not stored), so dimensions need only be
// multiples of 8.
// One launch takes up to three products of the same M (`nprob`: the q, k and v projections, their gradients); `parts` > 1 cuts the reduction, part p
// writing its own f32 C.  The attention's products run as batches, with the tiles and the reduction that the causal mask leaves: what it takes away is
// zero, and a product of zeros leaves the accumulator as it is.  Blocks of one XCD take neighbouring tiles.
// FOLD: where the tiles fill the chip without cutting the reduction, its parts, and products that are added up (the gradients of q, k and v), follow one
// another in the block and join a second set of accumulators, in the same order: no partial C in memory, no kernel that adds them, one launch.
#pragma once
#include "ixt_device.h"

#include <type_traits>

typedef float tf32x4 __attribute__((ext_vector_type(4)));
typedef short tbf16x8 __attribute__((ext_vector_type(8)));
typedef short tbf16x4 __attribute__((ext_vector_type(4)));

enum { TG_F32 = 0, TG_F32_ADD = 1, TG_BF16 = 2, TG_BF16_RES = 3 };   // C = acc, C += acc, C = bf16(acc), C = bf16(R + bf16(acc))

struct TGemm {
  const bf16_t* A[3]; long lda[3];       // stride of the index that is not contiguous
  const bf16_t* B[3]; long ldb[3];
  void* C[3]; long ldc[3];
  const bf16_t* R;                       // TG_BF16_RES: as C[0]
  int M, N[3], K[3];
  int nprob, parts, kpart;               // parts > 1: part p covers k in [p kpart, (p + 1) kpart) and writes C + p * cpart
  long cpart[3];
  int out;
  int mt, nt[3];                         // tiles
  // attention: nb1 x nb2 products of the same shape (nprob = parts = 1), element strides between them; `causal`: what the mask leaves
  int nb1, nb2, causal;
  long sa1, sa2, sb1, sb2, sc1, sc2;
  // FOLD: C[0] = the sum of `nsum` products of the same K and strides (nprob = 1 then); product 0, or each of nprob, adds up `fold` chunks of 32 k at a time (0: all)
  int nsum, fold;
};
enum { TC_NONE = 0, TC_LOWER = 1, TC_K_TO_ROW = 2, TC_K_FROM_ROW = 3 };   // C's tiles on and below the diagonal; k up to the tile's last row; k from its first row

static __device__ const uint32_t tg_zero[4] = {0u, 0u, 0u, 0u};

template <bool TA, bool TB, int MI, int NI, int WM, int WN, int NS, bool FOLD = false>
__global__ __launch_bounds__(WM * WN * 64, 2) void k_tgemm(TGemm g) {
  constexpr bool PAIR = !TA || !TB;
  constexpr int SLOTS = PAIR ? NS + 1 : NS;                               // pairs: two chunks being read, three ahead
  constexpr int BM = 16 * MI * WM, BN = 16 * NI * WN, NW = WM * WN;
  constexpr int NA = BM / 16, NB = BN / 16, NJ = (NA + NB) / NW;          // KiB of a chunk; a wave fetches NJ of them
  constexpr int SLOT = (BM + BN) * 32;                                    // elements
  static_assert(NA % NW == 0 && NB % NW == 0 && NS == 4, "a fetch is of one operand; the counts of the waits");
  extern __shared__ __attribute__((aligned(16))) bf16_t lds[];            // [SLOTS][A image | B image]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, r16 = lane & 15, q = lane >> 4;
  const int wm = wave / WN, wn = wave % WN;
  // XCD x takes a run of tiles (part by part); eight row tiles share their columns' operand
  const int ntn = g.nt[0] + g.nt[1] + g.nt[2], total = g.mt * ntn, every = total * g.parts * g.nb1 * g.nb2, per = (every + 7) >> 3;
  const int id = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (id >= every) return;                                                // whole block
  const int z = id / total, tile = id - z * total, part = g.parts > 1 ? z : 0, z1 = z / g.nb2, z2 = z - z1 * g.nb2;
  const int grp = tile / (8 * ntn), rows = min(8, g.mt - grp * 8), in = tile - grp * 8 * ntn;
  int tn = in / rows;
  const int tm = grp * 8 + in % rows;
  int prob = 0;
  while (prob < g.nprob - 1 && tn >= g.nt[prob]) tn -= g.nt[prob++];
  const int m0 = tm * BM, n0 = tn * BN, N = g.N[prob];
  if (g.causal == TC_LOWER && n0 > m0 + BM - 1) return;                   // whole block
  const long za = z1 * g.sa1 + z2 * g.sa2, zb = z1 * g.sb1 + z2 * g.sb2, zc = z1 * g.sc1 + z2 * g.sc2;

  int segk, segend;                                                       // k: next to fetch, end
  const char *pa, *pb;                                                    // the tile's first row at segk; bytes between chunks
  long adva, advb;
  uint32_t off[NJ];                                                       // the lane's place in a chunk, in bytes
  // piece f of a chunk's image (KiB): the k of this lane's 16 bytes, and row
  auto place = [&](bool tr, int bx, int f, int& k, int& x) {
    if (tr) {
      const int pr = bx / 8, sl = lane % pr;
      k = f * (64 / pr) + lane / pr;
      x = (((sl >> 1) ^ (bx == 64 ? k >> 1 & 3 : k & 7)) << 4) + (sl & 1) * 8;
    } else {
      x = f * 16 + (lane >> 2);
      k = ((lane & 3) ^ ((x >> 2) & 3)) * 8;
    }
  };
  {
    const long la = g.lda[prob], lb = g.ldb[prob];
    segk = g.parts > 1 ? part * g.kpart : 0;
    segend = g.parts > 1 ? min(g.K[prob], segk + g.kpart) : g.K[prob];
    if (g.causal == TC_K_TO_ROW) segend = min(segend, m0 + BM);
    if (g.causal == TC_K_FROM_ROW) segk = m0;
    pa = reinterpret_cast<const char*>(g.A[prob] + za + (TA ? (long)segk * la + m0 : (long)m0 * la + segk));
    pb = reinterpret_cast<const char*>(g.B[prob] + zb + (TB ? (long)segk * lb + n0 : (long)n0 * lb + segk));
    adva = TA ? 64 * la : 64; advb = TB ? 64 * lb : 64;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const int f = wave + NW * j;
      const bool isa = j * NW < NA;
      int k, x;
      place(isa ? TA : TB, isa ? BM : BN, isa ? f : f - NA, k, x);
      const int lim = (isa ? g.M - m0 : N - n0) - ((isa ? TA : TB) ? 8 : 1);
      x = min(x, lim);
      off[j] = (uint32_t)((isa ? TA : TB) ? k * (int)(isa ? la : lb) + x : x * (int)(isa ? la : lb) + k) * 2u;
    }
  }
  const int chunks1 = (segend - segk + 31) >> 5, chunks = FOLD ? g.nsum * chunks1 : chunks1;
  const int whole = !FOLD ? (segend - segk) >> 5 : (segend & 31) == 0 ? chunks : 0;      // chunks from the first on that end within K
  int sum = 0;                                                            // FOLD: the product that is fetched
  const uint32_t lds0 = (uint32_t)(uintptr_t)((__attribute__((address_space(3))) bf16_t*)lds);
  struct Chunk { const char *a, *b; int k; };                             // a chunk to fetch: its first row of either operand, its first k
  // piece j of this wave's share; the waits are counted in the loop.  A chunk that reaches past the last k fetches zeros there (edge), so that the counts stay
  auto issue = [&](int slot, int j, const Chunk& c, auto edge) {
    const bool isa = j * NW < NA;
    const uint32_t dst = __builtin_amdgcn_readfirstlane(lds0 + (uint32_t)(slot * SLOT + (wave + NW * j) * 512) * 2u);
    if constexpr (!edge.value) {
      lds_dma16(dst, isa ? c.a : c.b, off[j]);
    } else {
      int k, x;
      place(isa ? TA : TB, isa ? BM : BN, isa ? wave + NW * j : wave + NW * j - NA, k, x);
      lds_dma16(dst, c.k + k >= segend ? reinterpret_cast<const char*>(tg_zero) : (isa ? c.a : c.b) + off[j]);
    }
  };
  auto next_chunk = [&]() -> Chunk {
    const Chunk c{pa, pb, segk};
    segk += 32; pa += adva; pb += advb;
    if constexpr (FOLD) {
      if (segk >= segend && sum + 1 < g.nsum) {
        ++sum;
        segk = 0;
        pa = reinterpret_cast<const char*>(g.A[sum] + (TA ? (long)m0 : (long)m0 * g.lda[0]));
        pb = reinterpret_cast<const char*>(g.B[sum] + (TB ? (long)n0 : (long)n0 * g.ldb[0]));
      }
    }
    return c;
  };
  const int trf = (r16 >> 2) | (q & 1) << 2;                              // k & 7 of the lane's row in a transposed read: 4 q + r16 / 4
  auto operand = [&](const bf16_t* img, int x, int bx, bool tr) -> tbf16x8 {
    tbf16x4 lo, hi;
    if (tr) {                                                             // lane 4 a + p of a group: k row a, columns 4 p ..
      int f = bx == 64 ? trf >> 1 : trf;                                  // (k + 16: the same piece)
      asm volatile("" : "+v"(f));                                         // an address at a time: all of them ahead of the loop are 12 registers
      const bf16_t* p = img + (4 * q + (r16 >> 2)) * bx + (((x >> 4) ^ f) << 4) + 4 * (r16 & 3);
      lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tbf16x4*)p);
      hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) tbf16x4*)(p + 16 * bx));
    } else {
      const bf16_t* p = img + (x + r16) * 32 + (q & 1) * 4;
      const int f = (r16 >> 2) & 3;
      lo = *reinterpret_cast<const tbf16x4*>(p + (((q >> 1) ^ f) << 3));
      hi = *reinterpret_cast<const tbf16x4*>(p + ((((q >> 1) + 2) ^ f) << 3));
    }
    return __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
  };
  auto row_a = [&](int slot, int i) { return operand(lds + slot * SLOT, (wm * MI + i) * 16, BM, TA); };
  auto row_b = [&](int slot, int i) { return operand(lds + slot * SLOT + BM * 32, (wn * NI + i) * 16, BN, TB); };
  tf32x4 acc[MI][NI];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j) acc[i][j] = tf32x4(0.0f);
  tbf16x8 fa[MI], fb[2][NI];
  if constexpr (PAIR) {
#pragma unroll
    for (int c = 0; c < 4; c += 2) {
      const Chunk lo = next_chunk(), hi = next_chunk();
#pragma unroll
      for (int j = 0; j < NJ; ++j) { issue(c, j, lo, std::true_type()); issue(c + 1, j, hi, std::true_type()); }
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * NJ) : "memory");
  } else {
#pragma unroll
    for (int c = 0; c < NS; ++c) {
      const Chunk lo = next_chunk();
#pragma unroll
      for (int j = 0; j < NJ; ++j) issue(c, j, lo, std::true_type());
    }
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * NJ) : "memory");
  }
  lds_barrier();
#pragma unroll
  for (int j = 0; j < NI; ++j) fb[0][j] = row_b(0, j);
#pragma unroll
  for (int i = 0; i < MI; ++i) fa[i] = row_a(0, i);
  int slot = 0;                                                           // of chunk c
  auto step = [&](auto cur_, auto edge) {
    constexpr int cur = cur_.value;
    const int old = slot, older = slot == 0 ? SLOTS - 1 : slot - 1, nxt = slot + 1 == SLOTS ? 0 : slot + 1;
    slot = nxt;
    constexpr bool fetch = !PAIR || cur == 0;
    Chunk lo{}, hi{};
    if constexpr (fetch) lo = next_chunk();
    if constexpr (PAIR && fetch) hi = next_chunk();
    // a row of products, then a share of the reads of chunk c + 1 and of the fetches (of chunk c + NS; PAIR: for an even c, of chunks c + 4 and c + 5): they ride
    // under the products
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[cur][j], fa[i], acc[i][j], 0, 0, 0);
      if (i == 0) {
        // chunk c + 1 has landed once those behind it (PAIR: the pair behind its own) are all that is outstanding; this wave's reads of chunk c are done, so
        // behind the barrier its slot can be filled again.  Behind the first products: they cover the last reads and the waves' skew
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(PAIR ? 2 * NJ : (NS - 2) * NJ) : "memory");
        lds_barrier();
      }
      fa[i] = row_a(nxt, i);
#pragma unroll
      for (int j = 0; j < NI; ++j)
        if (j * MI / NI == i) fb[cur ^ 1][j] = row_b(nxt, j);
      if constexpr (fetch) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          if (j * MI / NJ == i) {
            issue(PAIR ? older : old, j, lo, edge);
            if constexpr (PAIR) issue(old, j, hi, edge);
          }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  tf32x4 tot[FOLD ? MI : 1][FOLD ? NI : 1];
  int next = FOLD && g.fold > 0 ? g.fold : chunks1;
  bool first = true;
  auto fold = [&](int done) {                                             // a cut of a reduction, or a whole one, joins the sum
    if constexpr (FOLD) {
      if (done != next) return;
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NI; ++j) {
          tot[i][j] = first ? acc[i][j] : tot[i][j] + acc[i][j];
          acc[i][j] = tf32x4(0.0f);
        }
      first = false;
      next += done < chunks1 ? g.fold : chunks1;
    }
  };
  int c = 0;
  auto steps = [&](int end, auto edge) {                                  // (an odd count: the last products are with zeros)
    for (; c < end; c += 2) {
      step(std::integral_constant<int, 0>(), edge);
      fold(c + 1);
      step(std::integral_constant<int, 1>(), edge);
      fold(c + 2);
    }
  };
  // steps that fetch whole chunks, without a branch between the products (one a fetch cost 300 cycles of 1500 a step), then the others
  steps((whole - 4) & ~1, std::false_type());                             // (steps c and c + 1 fetch chunks c + 4 and c + 5)
  steps(chunks, std::true_type());
  if constexpr (FOLD) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j) acc[i][j] = tot[i][j];
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");             // nothing may land in LDS that the next block owns
  // lane: m = r16, n = 4 q + register.  A tile that lies inside C has an epilogue without conditions: a load or a store under one is a block of its own, where a wait for a
  // load is one for every store before it (256 x 256: sums onto C 20 us a tile, 12 now; with a residual 13 and 7.2)
  const int out = g.out, m1 = m0 + wm * MI * 16 + r16, nw = n0 + wn * NI * 16;
  auto epilogue = [&](auto inside_) {
    constexpr bool inside = inside_.value;
    if (out == TG_F32 || out == TG_F32_ADD) {
      const long ld = g.ldc[prob];
      float* c = reinterpret_cast<float*>(g.C[prob]) + (g.parts > 1 ? part * g.cpart[prob] : zc) + (long)m1 * ld + nw + q * 4;
      auto in = [&](int i, int j) { return inside || (m1 + i * 16 < g.M && nw + j * 16 + q * 4 < N); };
      constexpr int AHEAD = MI < 4 ? MI : 4;                              // rows of the old sums in flight
      tf32x4 old[AHEAD][NI];
      auto load = [&](int i) {
#pragma unroll
        for (int j = 0; j < NI; ++j) old[i % AHEAD][j] = in(i, j) ? *reinterpret_cast<const tf32x4*>(c + i * 16 * ld + j * 16) : tf32x4(0.0f);
      };
      if (out == TG_F32_ADD) {
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) load(i);
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
          for (int j = 0; j < NI; ++j) {
            acc[i][j] = old[i % AHEAD][j] + acc[i][j];
            if (in(i, j)) *reinterpret_cast<tf32x4*>(c + i * 16 * ld + j * 16) = acc[i][j];
          }
          if (i + AHEAD < MI) load(i + AHEAD);
          __builtin_amdgcn_sched_barrier(0);                              // (a row's addresses at a time: all of them are 64 registers)
        }
      } else {
#pragma unroll
        for (int i = 0; i < MI; ++i) {
#pragma unroll
          for (int j = 0; j < NI; ++j)
            if (in(i, j)) *reinterpret_cast<tf32x4*>(c + i * 16 * ld + j * 16) = acc[i][j];
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      return;
    }
    // bf16: two column tiles at a time; a swap of lane groups leaves every lane eight columns of one of them, 16 bytes to store and 64 side by side (256 x 256:
    // 4.1 us for stores of 8 bytes, 2.4)
    static_assert(NI % 2 == 0, "pairs of column tiles");
    const int ns = nw + (q & 1) * 16 + (q >> 1) * 8;
    const long at = zc + (long)m1 * g.ldc[prob] + ns;
    auto in = [&](int i, int j) { return inside || (m1 + i * 16 < g.M && ns + j * 16 < N); };
    auto pair = [&](const uint2& lo, const uint2& hi) -> uint4 {
      const auto x = __builtin_amdgcn_permlane16_swap(lo.x, hi.x, false, false), y = __builtin_amdgcn_permlane16_swap(lo.y, hi.y, false, false);
      return make_uint4(x[0], y[0], x[1], y[1]);
    };
    if (out == TG_BF16_RES) {
      // (the pair of a pair is the pair's halves again)
      constexpr int STEP = MI < 4 ? MI : 4;
#pragma unroll
      for (int i0 = 0; i0 < MI; i0 += STEP) {
        uint4 r[STEP][NI / 2];
#pragma unroll
        for (int i = 0; i < STEP; ++i)
#pragma unroll
          for (int j = 0; j < NI; j += 2) r[i][j / 2] = in(i0 + i, j) ? *reinterpret_cast<const uint4*>(g.R + at + (i0 + i) * 16 * g.ldc[prob] + j * 16) : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
        for (int i = 0; i < STEP; ++i)
#pragma unroll
          for (int j = 0; j < NI; j += 2) {
            const uint4 h = pair(make_uint2(r[i][j / 2].x, r[i][j / 2].y), make_uint2(r[i][j / 2].z, r[i][j / 2].w));
            const uint2 hh[2] = {make_uint2(h.x, h.y), make_uint2(h.z, h.w)};
#pragma unroll
            for (int k = 0; k < 2; ++k) {
              tf32x4& v = acc[i0 + i][j + k];
              v[0] = bflo(hh[k].x) + rbf(v[0]); v[1] = bfhi(hh[k].x) + rbf(v[1]); v[2] = bflo(hh[k].y) + rbf(v[2]); v[3] = bfhi(hh[k].y) + rbf(v[3]);
            }
          }
      }
    }
#pragma unroll
    for (int i = 0; i < MI; ++i) {
#pragma unroll
      for (int j = 0; j < NI; j += 2) {
        const tf32x4 &v = acc[i][j], &w = acc[i][j + 1];
        const uint4 o = pair(make_uint2(pack2(f2bf(v[0]), f2bf(v[1])), pack2(f2bf(v[2]), f2bf(v[3]))), make_uint2(pack2(f2bf(w[0]), f2bf(w[1])), pack2(f2bf(w[2]), f2bf(w[3]))));
        if (in(i, j)) *reinterpret_cast<uint4*>(reinterpret_cast<bf16_t*>(g.C[prob]) + at + i * 16 * g.ldc[prob] + j * 16) = o;
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  };
  if (m0 + BM <= g.M && n0 + BN <= N) epilogue(std::true_type());
  else epilogue(std::false_type());
}
