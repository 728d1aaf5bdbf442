// ixt_gemm.h -- the canonical DOT for many rows (>= 128) as an LDS-ring GEMM with fused epilogues (included by ixt_kernels.h).
//
// Same arithmetic as k_dotb / k_gemm (chain c: 16 v_mfma_f32_16x16x32_bf16 over k in [512c, 512c+512) into one accumulator;
// total t = t + chain(c), c ascending), different data movement:
//   * both operands are stored in HBM in fragment order (1 KiB = one wave-instruction), so a K-chunk of a block tile is a list of
//     fragments that LDS-DMA (`global_load_lds_dwordx4`: 64 lanes x 16 B, no VGPRs) drops into an LDS ring slot exactly as the MFMAs
//     read them (lane-linear, conflict-free ds_read_b128);
//   * NS ring slots behind a counted `s_waitcnt vmcnt(N)` and ONE raw s_barrier per chunk: the latency of a chunk is hidden behind the
//     chunks ahead of it, and the reads of the next 32 k run under the products of these;
//   * a block owns whole (tile, all chains) work items: the chain totals stay in registers and the epilogue consumes them on chip --
//     no f32 slice leaves the chip except in the op-level / split forms.
// Block = WR x WC waves; wave tile = RB 16-row blocks x CT 16-column tiles; block tile = 16 WR RB rows x 16 WC CT columns.
// What bounds it: a 128 x 128 tile fetches as many bytes a chunk as the CU's 64 B a cycle bring in the time of its products (512 cycles of each per 64 k;
// measured 31 TB/s over the chip from L2), and a fetch that finds the queue full holds its wave and the MFMAs behind it.  256 x 128 tiles need 3/4 of
// that and win wherever the launch has enough of them: 14336 columns, K 2048, 1525 rows: 122 us (735 TFLOP/s) with 128 x 128 tiles whose chunk was
// read and then multiplied, 112 with the reads under the products, 107 and now 100 with the steps that refill a loop of their own, without a branch, and the barrier behind a
// step's first products.  256 x 128 tiles take 1250 to 1310 cycles per 64 k of which the products are 1068, at 1.6 to 2.3 GHz: the card's power sets the clock.  Tried without gain: the
// fetches of a SIMD's two waves in different halves of a chunk, hot weights, chunk-contiguous operands.
// What a launch spends beside its chunks (256 x 128, 128 x 128): 2 to 3.5 us until the first one is there, and the epilogue, before and now: residual 6.5 and 3.4 -> 2.4 and 1.1 us (loads, then
// stores of 16 bytes), gated unit 4.5 and 2.3 -> 2.7 and 1.5 (ixt_gate), Gemma's 12 -> 2.7, q, k, v 10.7 and 6.0 -> 6.7 and 3.1.
//
// Epilogues (EPI):
//   GEPI_F32      f32 [slice][R][N] (op-level entry point, split-K form)
//   GEPI_UNEMBED  greedy sampling (decoders.py:566-587, inference_utils.py:74-75): bf16-rounded logits on request, one
//                 (max, first index) pair per row and wave column for k_argmax_final
//   GEPI_RESID    h_out = bf16(h_in + bf16(t))                                   (llama2.py:127, :157)
//   GEPI_SWIGLU   act = bf16(bf16(silu(bf16(t_0))) * bf16(t_1)), or the gelu gate  (linears.py:449-464); the fused wi kernel stores
//                 wi_0 tile j and wi_1 tile j as column tiles 2j, 2j+1, so both gates of a feature are in one wave
//   GEPI_ACT      act = bf16(unit(t)), a unit without a gate (ixt_act)
//   GEPI_TANHNORM residual and norms of a decoder with tanh norms (TanhNormEpi)
//   GEPI_QKV      bf16(t), RoPE (embeddings.py:277-315), q -> qbuf, k / v -> the row's page (paged_attention.py:446-471).  Q and K
//                 head columns are stored pair-interleaved (qk_col): a 16-column tile holds features 8j..8j+7 and half+8j..half+8j+7,
//                 so the two RoPE partners of a feature sit in lanes l and l ^ 32 of one accumulator register.
//   GEPI_QKV32    the same with rope_type "llama3.1" (a kernel of its own: its code in the other's way costs every wave instruction fetches)
#pragma once
#include <type_traits>

enum { GEPI_F32 = 0, GEPI_UNEMBED = 1, GEPI_RESID = 2, GEPI_SWIGLU = 3, GEPI_QKV = 4, GEPI_TANHNORM = 5, GEPI_ACT = 6, GEPI_QKV32 = 7 };

// GEPI_TANHNORM: an f32 residual stream between tanh norms, x <- x + post(t), act = bf16(pre(x)), norm(y) = tanh(alpha y) w + b feature by feature (w
// null: no norm).  Nothing in it looks at a row's other features, so it needs no launch of its own.
struct TanhNormEpi {
  const float *post_w, *post_b, *post_alpha, *pre_w, *pre_b, *pre_alpha;      // zeros behind feature E - 1
  float *x, *h32;                                       // [R][E]; h32 (or nullptr): pre(x) in f32
  int E, Ep;                                            // features, and the row length of `act`
};
// four columns of one row; col % 4 == 0, col + 3 < Ep
__device__ __forceinline__ void tanhnorm_epi(const TanhNormEpi& n, bf16_t* act, int row, int col, const f32x4& t) {
  float y[4] = {t[0], t[1], t[2], t[3]}, x[4];
  const bool vec = (n.E & 3) == 0 && col < n.E;
  float* xp = n.x + (size_t)row * n.E + col;
  if (vec) { const float4 v = *reinterpret_cast<const float4*>(xp); x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w; }
  else {
#pragma unroll
    for (int j = 0; j < 4; ++j) x[j] = col + j < n.E ? xp[j] : 0.0f;
  }
  if (n.post_w != nullptr) {
    const float4 w = *reinterpret_cast<const float4*>(n.post_w + col), b = *reinterpret_cast<const float4*>(n.post_b + col);
    const float al = *n.post_alpha;
    y[0] = fmaf(tanh_f32(al * y[0]), w.x, b.x); y[1] = fmaf(tanh_f32(al * y[1]), w.y, b.y);
    y[2] = fmaf(tanh_f32(al * y[2]), w.z, b.z); y[3] = fmaf(tanh_f32(al * y[3]), w.w, b.w);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) x[j] += y[j];
  if (vec) *reinterpret_cast<float4*>(xp) = make_float4(x[0], x[1], x[2], x[3]);
  else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (col + j < n.E) xp[j] = x[j];
  }
  if (n.pre_w != nullptr) {
    const float4 w = *reinterpret_cast<const float4*>(n.pre_w + col), b = *reinterpret_cast<const float4*>(n.pre_b + col);
    const float al = *n.pre_alpha;
    x[0] = fmaf(tanh_f32(al * x[0]), w.x, b.x); x[1] = fmaf(tanh_f32(al * x[1]), w.y, b.y);
    x[2] = fmaf(tanh_f32(al * x[2]), w.z, b.z); x[3] = fmaf(tanh_f32(al * x[3]), w.w, b.w);
  }
  if (n.h32 != nullptr) {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (col + j < n.E) n.h32[(size_t)row * n.E + col + j] = x[j];
  }
  uint2 o;
  o.x = pack2(f2bf(x[0]), f2bf(x[1])); o.y = pack2(f2bf(x[2]), f2bf(x[3]));
  *reinterpret_cast<uint2*>(act + xidx(row, col, n.Ep)) = o;
}

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
// A lane of an accumulator tile holds four columns of one row (8 bytes of bf16): lane group q columns 4 q ..  The tiles of two row blocks, a swap of lane groups apart, are
// 16 bytes a lane: eight columns, 8 (q / 2) .., of the first block on even groups, of the second on odd ones.  rows_split undoes it.
__device__ __forceinline__ u32x4 rows_pair(const uint2& lo, const uint2& hi) {
  const auto x = __builtin_amdgcn_permlane16_swap(lo.x, hi.x, false, false), y = __builtin_amdgcn_permlane16_swap(lo.y, hi.y, false, false);
  return u32x4{x[0], y[0], x[1], y[1]};
}
__device__ __forceinline__ void rows_split(const u32x4& m, uint2& lo, uint2& hi) {
  const auto x = __builtin_amdgcn_permlane16_swap(m.x, m.z, false, false), y = __builtin_amdgcn_permlane16_swap(m.y, m.w, false, false);
  lo = make_uint2(x[0], y[0]); hi = make_uint2(x[1], y[1]);
}
// A value that is there from here on.  An epilogue loads, then fences, computes, fences, and then stores: a store under a condition is a block of its own, and a wait
// in it for a load (or a load behind it) is one for every store before it, too.  128 x 128, residual: 3.4 us for eight stores that waited for each other, 1.1 with all at once.
template <typename T> __device__ __forceinline__ void epi_fence(T& v) { asm volatile("" : "+v"(v)); }

struct GemmEpi {
  float* out;                                           // F32: [slices][R][N]; UNEMBED: rounded logits [R][N] or nullptr
  float* amax_val; int32_t* amax_idx; ColRanges cr;     // UNEMBED: [R][WC ncolg]
  const bf16_t* h_in; bf16_t* h_out;                    // RESID: [R][N] row-major
  bf16_t* act;                                          // SWIGLU: [R][N/2] in xidx layout; ACT: [R][N]
  const int32_t* row_slot; const int32_t* row_pos; const int32_t* row_active; const int32_t* page_map;   // QKV
  const bf16_t* rope_sin; const bf16_t* rope_cos;
  bf16_t* qbuf; bf16_t* kpages; bf16_t* vpages;
  AttnGeom g;
  float q_scalar;                                       // QKV: queries times this bf16 value behind RoPE (0: none)
  const float* xscale; const float* wscale;             // F8: activation scales [rows][chains], column scales [N] (ixt_fp8.h)
  size_t sstride;                                       // F8 + routed experts: floats between two experts' column scales
  TanhNormEpi tn;                                       // TANHNORM (with act)
  int glu; float glu_limit; const float* act_par;       // ACT: the unit's kind and its numbers; SWIGLU: glu > 0 takes that gated unit of the f32 totals instead (ixt_glu), glu < 0 ixt_geglu
  const bf16_t* gate;                                   // SWIGLU, glu <= 0: the gate's table (ixt_gate), IXT_GATE_BYTES
  int32_t* flags;                                       // SPLIT 2: a word a wave of a tile and part, zero between launches
  IxtWait wait;
  const int32_t* rb_exp; size_t wstride;                // routed experts: expert of every 16-row block (-1: none), 16-byte units between experts' kernels
};

template <int N_>
__device__ __forceinline__ void ring_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N_) : "memory");
}
// at most min(M, younger) chunks of NJ fetches outstanding, and no LDS read
template <int NJ, int M>
__device__ __forceinline__ void ring_wait_chunks(int younger) {
  if constexpr (M > 0) {
    if (younger < M) return ring_wait_chunks<NJ, M - 1>(younger);
  }
  ring_wait<M * NJ>();
}

// SPLIT 2 (GEPI_F32): a tile's chains in gridDim.y parts, one block each.  A sum's order stays: part 0 adds its chains up as it goes, a later part keeps each of its chains (at most RING_KEEP) in
// registers, takes the sum so far from the part before it, wave by wave, adds its own in order and hands it on; the last one stores it.  Progress: a part waits for a block of lower
// index on the same XCD (gridDim.x is a multiple of 8), which has started before it; the waits are bounded all the same.  For few tiles of a long K: 256 x 2304 outputs, K 9216, 41 us in
// one part (144 tiles of 64 x 64 for 256 CUs), 35 in three equal ones (72 of 128 x 64), 31 with a chain more for each later part.
// RING_KEEP holds up to 18 chains, the longest that was measured (163 of 256 registers); a sum of more goes to one block a tile.
#define RING_KEEP 7
#define RING_LEFT 2              // a flag whose taker gave up: its setter clears it, so that the next launch finds zeros whatever happened
//   grid = (8 ceil(ncolg / 8) zb, SPLIT 1 ? chains : SPLIT 2 ? parts : 1), block 64 WR WC, dynamic LDS = NS (WC CT + WR RB) KS KiB and, for SWIGLU, the gate's table.
//   Row groups of one column group are block ids b, b + 8, ..: same XCD, the weights meet in its L2.
//   F8 (ixt_fp8.h): both operands are e4m3 fragments of 64 k (still 1 KiB: the ring moves them exactly as bf16 fragments of 32 k); a fragment
//   feeds two v_mfma_f32_16x16x32_fp8_fp8; at the end of every 512-k chain the accumulator is scaled by (a_rc s_n) before it joins the total.
template <int WR, int WC, int RB, int CT, int KS, int NS, int EPI, int SPLIT, bool F8 = false, bool ONCE = false>
__global__ __launch_bounds__(WR * WC * 64, 2) void k_gemm_ring(const u32x4* __restrict__ xt, const u32x4* __restrict__ wt, int K, int N, int R,
                                                               int ncolg, int zb, int wring, GemmEpi e) {
  constexpr int NW = WR * WC;          // waves
  constexpr int TC = WC * CT;          // column tiles of a block
  constexpr int TR = WR * RB;          // row blocks of a block
  constexpr int NWF = TC * KS;         // weight fragments of a chunk
  constexpr int NXF = TR * KS;         // activation fragments
  constexpr int NF = NWF + NXF;
  constexpr int NJ = NF / NW;          // fragments a wave fetches per chunk
  static_assert(NF % NW == 0 && 16 % KS == 0 && (NS - 1) * NJ < 64 && NS > 1 && (KS == 1 || KS % 2 == 0), "ring geometry");
  static_assert(EPI != GEPI_SWIGLU || CT % 2 == 0, "gate pairs need two tiles per wave");
  extern __shared__ __attribute__((aligned(16))) u32x4 st[];   // [NS][NF fragments][64 lanes]
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int bx = blockIdx.x;
  const int colg = (bx / (8 * zb)) * 8 + (bx & 7), rowg = (bx >> 3) % zb;
  if (colg >= ncolg) return;                                    // whole block: no barrier is skipped
  if (e.rb_exp != nullptr) {                                    // routed experts (k_moe_plan, align 128): this row group's expert, or nothing to do
    const int ex = (rowg * (WR * RB) < ((R + 15) >> 4)) ? e.rb_exp[rowg * (WR * RB)] : -1;
    if (ex < 0) return;
    wt += (size_t)ex * e.wstride;
    if constexpr (F8) e.wscale += (size_t)ex * e.sstride;       // the expert's column scales
  }
  const int nsteps = F8 ? K >> 6 : K >> 5, ntile = N >> 4, nrbk = (R + 15) >> 4;   // fragments along k
  const int nchunks = nsteps / KS;
  const int wr = wave / WC, wc = wave % WC;
  const int r_in = lane & 15, cq = lane >> 4;
  // weights: fragment order [tile][k-step] (wring == 0: the layout of the small-batch kernels) or the ring layout (r8frag).  A wave's pieces of a chunk:
  // one offset a piece from the first fragment of the block's tiles, one scalar address that moves from chunk to chunk
  const size_t wadv = (wring ? (size_t)KS * 8 : (size_t)KS) * 1024;    // bytes between two chunks of one tile
  uint32_t off[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const int f = wave + NW * j;
    if (f < NWF) {
      const int tile = wring ? colg * TC + f / KS : min(colg * TC + f / KS, ntile - 1);    // past the end: a valid (wring: padding) tile, results dropped
      off[j] = (uint32_t)(wring ? r8frag(tile, f % KS, nsteps) - r8frag(colg * TC, 0, nsteps) : (size_t)(tile - colg * TC) * nsteps + (f % KS)) * 1024u;
    } else {
      const int rb = min(rowg * TR + (f - NWF) / KS, nrbk - 1);
      off[j] = (uint32_t)((rb - rowg * TR) * nsteps + (f - NWF) % KS) * 1024u;
    }
    off[j] += lane * 16;
  }
  constexpr int CPC = (F8 ? 8 : 16) / KS;                       // chunks per 512-k chain
  const int nch = (nchunks + CPC - 1) / CPC, part = SPLIT == 2 ? (int)blockIdx.y : 0, parts = SPLIT == 2 ? (int)gridDim.y : 1;
  // (a later part has a chain more: it waits for the one before)
  const int chb = SPLIT == 2 ? (part == 0 ? 0 : nch * part / parts - 1) * CPC : SPLIT ? (int)blockIdx.y * CPC : 0;
  const int che = SPLIT == 2 ? min(nchunks, (part + 1 == parts ? nch : nch * (part + 1) / parts - 1) * CPC) : SPLIT ? min(nchunks, chb + CPC) : nchunks;
  const char* pw = reinterpret_cast<const char*>(wt + (wring ? r8frag(colg * TC, 0, nsteps) : (size_t)colg * TC * nsteps) * 64) + chb * wadv;
  const char* px = reinterpret_cast<const char*>(xt + (size_t)rowg * TR * nsteps * 64) + (size_t)chb * KS * 1024;
  const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)((__attribute__((address_space(3))) u32x4*)st));
  // piece j of the next chunk to fetch, into a slot; the waits are counted in the loop.  ONCE (one row group): no other block reads these weights, so they are streamed past the caches (264192 columns, K 2048: 48 rows 219 -> 203 us, 256 rows 386 -> 359; several row groups of small tiles lose
  // by it, and a branch here instead of a second kernel costs them up to 10 %).
  auto issue = [&](int slot, int j) {
    const uint32_t dst = lds0 + (uint32_t)(slot * NF + wave + NW * j) * 1024u;
    if (NW * j >= NWF || (NW * j + NW > NWF && wave + NW * j >= NWF))
      lds_dma16(dst, px, off[j]);
    else lds_dma16<ONCE>(dst, pw, off[j]);
  };
  auto advance = [&]() { pw += wadv; px += (size_t)KS * 1024; };
  bf16_t* const gate = reinterpret_cast<bf16_t*>(st + NS * NF * 64);
  if constexpr (EPI == GEPI_SWIGLU) {                           // (older than every chunk: the first wait covers it)
    if (e.glu <= 0) {
      for (int p = wave; p < IXT_GATE_BYTES / 1024; p += NW) lds_dma16(lds0 + (uint32_t)(NS * NF + p) * 1024u, e.gate, (uint32_t)(p * 1024 + lane * 16));
    }
  }
#pragma unroll
  for (int c = 0; c < NS; ++c)
    if (chb + c < che) {
#pragma unroll
      for (int j = 0; j < NJ; ++j) issue(c, j);
      advance();
    }
  // QKV: the positions of the rows, and of a store's rows (PR row blocks, one for even and one for odd lane groups).  Behind the first fetches, in whose time they come; the first
  // counted wait waits for as many pieces more
  constexpr bool ROWS = EPI == GEPI_QKV || EPI == GEPI_QKV32;
  constexpr int PR = RB % 2 == 0 && EPI == GEPI_QKV ? 2 : 1;
  const int odd = PR == 2 ? cq & 1 : 0;
  int pos[ROWS ? RB : 1], spos[ROWS ? RB / PR : 1], page[ROWS ? RB / PR : 1], act[ROWS ? RB / PR : 1];
  if constexpr (ROWS) {
#pragma unroll
    for (int b = 0; b < RB; ++b) pos[b] = e.row_pos[min((rowg * TR + wr * RB + b) * 16 + r_in, R - 1)];
#pragma unroll
    for (int b = 0; b < RB; b += PR) {
      const int at = min((rowg * TR + wr * RB + b + odd) * 16 + r_in, R - 1);
      spos[b / PR] = e.row_pos[at]; page[b / PR] = e.row_slot[at]; act[b / PR] = e.row_active[at];      // (no use of them here: it would be a wait)
    }
  }
  f32x4 acc[CT][RB], tot[CT][RB];
#pragma unroll
  for (int i = 0; i < CT; ++i)
#pragma unroll
    for (int b = 0; b < RB; ++b) { acc[i][b] = f32x4(0.0f); tot[i][b] = f32x4(0.0f); }
  bf16x8 wf[CT], xf[2][RB];
  auto wfrag = [&](int slot, int ks, int i) { return __builtin_bit_cast(bf16x8, st[(slot * NF + (wc * CT + i) * KS + ks) * 64 + lane]); };
  auto xfrag = [&](int slot, int ks, int b) { return __builtin_bit_cast(bf16x8, st[(slot * NF + NWF + (wr * RB + b) * KS + ks) * 64 + lane]); };
  ring_wait_chunks<NJ, NS - 1>(che - chb - 1);                  // chunk chb
  lds_barrier();
#pragma unroll
  for (int b = 0; b < RB; ++b) xf[0][b] = xfrag(0, 0, b);
#pragma unroll
  for (int i = 0; i < CT; ++i) wf[i] = wfrag(0, 0, i);
  int slot = 0;                                                 // ring slot of chunk ch
  bool refill = false;
  int fill = 0;
  // One k-step: products of the fragments in registers, with the reads of the next step's fragments and the refill of the slot that was read out last dealt
  // between them, so that the matrix cores, the LDS and the fetches run side by side (reading a chunk and then multiplying it took turns: 1 500 cycles a
  // 64-k chunk of a 128 x 128 tile, of which the products are 512).  Behind the first products of a chunk's last step its fragments are all in registers and the
  // next chunk has to be there: one counted wait and one barrier a chunk, behind which its slot is free for chunk ch + NS.  STEADY: there is such a chunk, and
  // there was one in the chunk before; the steps of these are a loop without a branch.
  auto step = [&](int ch, auto ks_, int cur, auto steady) {
    constexpr int ks = ks_.value;
    constexpr bool last = ks == KS - 1;
    constexpr int nks = last ? 0 : ks + 1, from = nks;                // `from`: position of this step among the KS steps of a refill
#pragma unroll
    for (int i = 0; i < CT; ++i) {
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        if constexpr (F8) {
          typedef long l2 __attribute__((ext_vector_type(2)));
          const l2 wl = __builtin_bit_cast(l2, wf[i]), xl = __builtin_bit_cast(l2, xf[cur][b]);
          acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(wl[0], xl[0], acc[i][b], 0, 0, 0);
          acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_fp8_fp8(wl[1], xl[1], acc[i][b], 0, 0, 0);
        } else {
          acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[i], xf[cur][b], acc[i][b], 0, 0, 0);
        }
      }
      if (last && i == 0) {
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (steady.value) ring_wait<(NS - 2) * NJ>();
        else ring_wait_chunks<NJ, NS - 2>(che - ch - 2);
        lds_barrier();
        if constexpr (!steady.value) refill = ch + NS < che;
        fill = slot;
        slot = slot + 1 == NS ? 0 : slot + 1;
      }
      wf[i] = wfrag(slot, nks, i);
#pragma unroll
      for (int b = 0; b < RB; ++b)
        if (b * CT / RB == i) xf[cur ^ 1][b] = xfrag(slot, nks, b);
      const int gi = from * CT + i;
      if (steady.value || refill) {
#pragma unroll
        for (int j = 0; j < NJ; ++j)
          if (j * (KS * CT) / NJ == gi) issue(fill, j);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (from == KS - 1 && (steady.value || refill)) advance();
  };
  // a 512-k chain is complete
  auto chain_end = [&](int ch) {
    if constexpr (F8) {                                         // scale the chain by (activation block scale) x (column scale)
      const int chain = ch / CPC, nchains = (nchunks + CPC - 1) / CPC;
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int row = min((rowg * TR + wr * RB + b) * 16 + r_in, R - 1);
        const float a = e.xscale[(size_t)row * nchains + chain];
#pragma unroll
        for (int i = 0; i < CT; ++i) {
          const int tile = min(colg * TC + wc * CT + i, ntile - 1);
          const float4 sn = *reinterpret_cast<const float4*>(e.wscale + tile * 16 + cq * 4);
          acc[i][b][0] *= a * sn.x; acc[i][b][1] *= a * sn.y; acc[i][b][2] *= a * sn.z; acc[i][b][3] *= a * sn.w;
        }
      }
    }
#pragma unroll
    for (int i = 0; i < CT; ++i)
#pragma unroll
      for (int b = 0; b < RB; ++b) { tot[i][b] = tot[i][b] + acc[i][b]; acc[i][b] = f32x4(0.0f); }
  };
  auto chunk = [&](int ch, auto steady) {
    step(ch, std::integral_constant<int, 0>(), 0, steady);
    if constexpr (KS > 1) step(ch, std::integral_constant<int, 1 % KS>(), 1, steady);
    if constexpr (KS > 2) { step(ch, std::integral_constant<int, 2 % KS>(), 0, steady); step(ch, std::integral_constant<int, 3 % KS>(), 1, steady); }
  };
  static_assert(KS == 1 || KS == 2 || KS == 4, "steps of a chunk");
  if constexpr (KS == 1) {                                      // (an even number of chunks: K is a multiple of 128)
    auto two = [&](int ch, auto steady) {
      step(ch, std::integral_constant<int, 0>(), 0, steady);
      step(ch + 1, std::integral_constant<int, 0>(), 1, steady);
      if (((ch + 2) % CPC) == 0 || ch + 2 == che) chain_end(ch);
    };
    int ch = chb;
    for (; ch + 1 + NS < che; ch += 2) two(ch, std::true_type());
    for (; ch < che; ch += 2) two(ch, std::false_type());
  } else if (SPLIT != 2 || part == 0) {
    auto one = [&](int ch, auto steady) {
      chunk(ch, steady);
      if (((ch + 1) % CPC) == 0 || ch + 1 == che) chain_end(ch);
    };
    int ch = chb;
    one(ch++, std::false_type());
    if (refill) {                                               // (chunk ch - 1 + NS has begun to come)
      for (; ch + NS < che; ++ch) one(ch, std::true_type());
    }
    for (; ch < che; ++ch) one(ch, std::false_type());
  }
  if constexpr (SPLIT == 2) {
    static_assert(EPI == GEPI_F32 && KS > 1 && !F8, "parts of f32 sums");
    f32x4 keep[RING_KEEP][CT][RB];
    if (part > 0) {
#pragma unroll
      for (int q = 0; q < RING_KEEP; ++q) {
        for (int ch = chb + q * CPC; ch < min(che, chb + (q + 1) * CPC); ++ch) chunk(ch, std::false_type());
#pragma unroll
        for (int i = 0; i < CT; ++i)
#pragma unroll
          for (int b = 0; b < RB; ++b) { keep[q][i][b] = acc[i][b]; acc[i][b] = f32x4(0.0f); }
      }
    }
    auto place = [&](int i, int b, float*& p) {
      const int tile = colg * TC + wc * CT + i, row = (rowg * TR + wr * RB + b) * 16 + r_in;
      p = e.out + (size_t)row * N + tile * 16 + cq * 4;
      return tile < ntile && row < R;
    };
    int32_t* flag = e.flags + ((size_t)blockIdx.x * NW + wave) * parts;
    float* p;
    bool ready = true;
    if (part > 0) {
      for (int it = 0; __hip_atomic_load(flag + part - 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0;) {
        if (++it > e.wait.polls) {
          int seen = 0;
          if (lane == 0) __hip_atomic_compare_exchange_strong(flag + part - 1, &seen, RING_LEFT, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          ready = __builtin_amdgcn_readfirstlane(seen) != 0;
          if (!ready) ixt_gave_up(e.wait);
          break;
        }
        __builtin_amdgcn_s_sleep(1);
      }
      asm volatile("" ::: "memory");
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int b = 0; b < RB; ++b) {
          if (!place(i, b, p)) continue;
          unsigned long long* q = reinterpret_cast<unsigned long long*>(p);      // (past the L2: half of a line is another wave's, and may be older)
          const unsigned long long lo = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), hi = __hip_atomic_load(q + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          tot[i][b] = f32x4{__uint_as_float((uint32_t)lo), __uint_as_float((uint32_t)(lo >> 32)), __uint_as_float((uint32_t)hi), __uint_as_float((uint32_t)(hi >> 32))};
        }
#pragma unroll
      for (int q = 0; q < RING_KEEP; ++q)
        if (chb + q * CPC < che) {
#pragma unroll
          for (int i = 0; i < CT; ++i)
#pragma unroll
            for (int b = 0; b < RB; ++b) tot[i][b] = tot[i][b] + keep[q][i][b];
        }
      if (lane == 0 && ready) __hip_atomic_store(flag + part - 1, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    if (part < parts - 1) {
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int b = 0; b < RB; ++b)
          if (place(i, b, p)) stg16_agent(p, tot[i][b]);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (lane == 0 && __hip_atomic_exchange(flag + part, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == RING_LEFT)
        __hip_atomic_store(flag + part, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);      // nobody takes it any more
      return;
    }
  }

  // ---------------------------------------------------------------- epilogues
  if constexpr (EPI == GEPI_F32) {
    float* out = e.out + (SPLIT == 1 ? (size_t)blockIdx.y * R * N : 0);
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      const int tile = colg * TC + wc * CT + i;
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int row = (rowg * TR + wr * RB + b) * 16 + r_in;
        if (tile < ntile && row < R)
          *reinterpret_cast<float4*>(out + (size_t)row * N + tile * 16 + cq * 4) = make_float4(tot[i][b][0], tot[i][b][1], tot[i][b][2], tot[i][b][3]);
      }
    }
  } else if constexpr (EPI == GEPI_UNEMBED) {
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const int row = (rowg * TR + wr * RB + b) * 16 + r_in;
      float bv = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int i = 0; i < CT; ++i) {
        const int tile = colg * TC + wc * CT + i;
        if (tile < ntile) {
          float v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) v[j] = rbf(tot[i][b][j]);
          if (e.out != nullptr && row < R) *reinterpret_cast<float4*>(e.out + (size_t)row * N + tile * 16 + cq * 4) = make_float4(v[0], v[1], v[2], v[3]);
#pragma unroll
          for (int j = 0; j < 4; ++j)
            if (v[j] > bv && col_allowed(e.cr, tile * 16 + cq * 4 + j)) { bv = v[j]; bi = tile * 16 + cq * 4 + j; }   // ascending columns
        }
      }
#pragma unroll
      for (int off = 16; off < 64; off <<= 1) {
        const float ov = __shfl_xor(bv, off, 64);
        const int oi = __shfl_xor(bi, off, 64);
        if (ov > bv || (ov == bv && oi < bi)) { bv = ov; bi = oi; }
      }
      if (cq == 0 && row < R) {
        e.amax_val[(size_t)row * (WC * ncolg) + colg * WC + wc] = bv;
        e.amax_idx[(size_t)row * (WC * ncolg) + colg * WC + wc] = bi;
      }
    }
  } else if constexpr (EPI == GEPI_RESID) {
    if constexpr (RB % 2 == 0) {
      u32x4 m[CT][RB / 2];
      auto at = [&](int i, int b) {
        const int tile = min(colg * TC + wc * CT + i, ntile - 1), row = min((rowg * TR + wr * RB + b + (cq & 1)) * 16 + r_in, R - 1);
        return (size_t)row * N + tile * 16 + 8 * (cq >> 1);
      };
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int b = 0; b < RB; b += 2) m[i][b / 2] = *reinterpret_cast<const u32x4*>(e.h_in + at(i, b));
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int b = 0; b < RB; b += 2) {
          uint2 h[2];
          rows_split(m[i][b / 2], h[0], h[1]);
#pragma unroll
          for (int k = 0; k < 2; ++k) {
            const f32x4& t = tot[i][b + k];
            h[k].x = pack2(f2bf(bflo(h[k].x) + rbf(t[0])), f2bf(bfhi(h[k].x) + rbf(t[1])));
            h[k].y = pack2(f2bf(bflo(h[k].y) + rbf(t[2])), f2bf(bfhi(h[k].y) + rbf(t[3])));
          }
          m[i][b / 2] = rows_pair(h[0], h[1]);
          epi_fence(m[i][b / 2]);
        }
#pragma unroll
      for (int i = 0; i < CT; ++i)
#pragma unroll
        for (int b = 0; b < RB; b += 2)
          if (colg * TC + wc * CT + i < ntile && (rowg * TR + wr * RB + b + (cq & 1)) * 16 + r_in < R) *reinterpret_cast<u32x4*>(e.h_out + at(i, b)) = m[i][b / 2];
    } else {
#pragma unroll
      for (int i = 0; i < CT; ++i) {
        const int tile = colg * TC + wc * CT + i;
#pragma unroll
        for (int b = 0; b < RB; ++b) {
          const int row = (rowg * TR + wr * RB + b) * 16 + r_in;
          if (tile < ntile && row < R) {
            const size_t o = (size_t)row * N + tile * 16 + cq * 4;
            const uint2 hv = *reinterpret_cast<const uint2*>(e.h_in + o);
            uint2 ov;
            ov.x = pack2(f2bf(bflo(hv.x) + rbf(tot[i][b][0])), f2bf(bfhi(hv.x) + rbf(tot[i][b][1])));
            ov.y = pack2(f2bf(bflo(hv.y) + rbf(tot[i][b][2])), f2bf(bfhi(hv.y) + rbf(tot[i][b][3])));
            *reinterpret_cast<uint2*>(e.h_out + o) = ov;
          }
        }
      }
    }
  } else if constexpr (EPI == GEPI_TANHNORM) {
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      const int tile = colg * TC + wc * CT + i;
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int row = (rowg * TR + wr * RB + b) * 16 + r_in;
        if (tile < ntile && row < R) tanhnorm_epi(e.tn, e.act, row, tile * 16 + cq * 4, tot[i][b]);
      }
    }
  } else if constexpr (EPI == GEPI_ACT) {
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      const int tile = colg * TC + wc * CT + i;
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int row = (rowg * TR + wr * RB + b) * 16 + r_in;
        if (tile < ntile && row < R) {
          uint2 ov;
          ov.x = pack2(f2bf(ixt_act(e.glu, tot[i][b][0], e.act_par)), f2bf(ixt_act(e.glu, tot[i][b][1], e.act_par)));
          ov.y = pack2(f2bf(ixt_act(e.glu, tot[i][b][2], e.act_par)), f2bf(ixt_act(e.glu, tot[i][b][3], e.act_par)));
          *reinterpret_cast<uint2*>(e.act + xidx(row, tile * 16 + cq * 4, N)) = ov;
        }
      }
    }
  } else if constexpr (EPI == GEPI_SWIGLU) {
    static_assert(RB % 2 == 0, "pairs of row blocks");
    const int F = N >> 1;
    u32x4 m[CT / 2][RB / 2];
#pragma unroll
    for (int i = 0; i < CT; i += 2)                         // tile even: wi_0 tile tile/2; tile + 1: wi_1 tile tile/2
#pragma unroll
      for (int b = 0; b < RB; b += 2) {
        uint2 o[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          bf16_t v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            v[j] = e.glu > 0 ? f2bf(ixt_glu(e.glu, tot[i][b + k][j], tot[i + 1][b + k][j], e.glu_limit)) : ixt_gate(gate, tot[i][b + k][j], tot[i + 1][b + k][j]);
          o[k].x = pack2(v[0], v[1]); o[k].y = pack2(v[2], v[3]);
        }
        m[i / 2][b / 2] = rows_pair(o[0], o[1]);
        epi_fence(m[i / 2][b / 2]);
      }
#pragma unroll
    for (int i = 0; i < CT; i += 2)
#pragma unroll
      for (int b = 0; b < RB; b += 2) {
        const int tile = colg * TC + wc * CT + i, row = (rowg * TR + wr * RB + b + (cq & 1)) * 16 + r_in;
        if (tile + 1 < ntile && row < R) *reinterpret_cast<u32x4*>(e.act + xidx(row, (tile >> 1) * 16 + 8 * (cq >> 1), F)) = m[i / 2][b / 2];
      }
  } else if constexpr (EPI == GEPI_QKV || EPI == GEPI_QKV32) {
    const AttnGeom& g = e.g;
    const int half = g.hd >> 1, tph = g.hd >> 4;                // tiles per head
    // section (q, k, v), head in it and tile in that of the wave's column tiles
    int sect[CT], hh[CT], th[CT];
    hh[0] = (colg * TC + wc * CT) / tph;
    th[0] = colg * TC + wc * CT - hh[0] * tph;
#pragma unroll
    for (int i = 1; i < CT; ++i) {
      const bool next = th[i - 1] + 1 == tph;
      hh[i] = hh[i - 1] + next;
      th[i] = next ? 0 : th[i - 1] + 1;
    }
#pragma unroll
    for (int i = 0; i < CT; ++i) {
      sect[i] = hh[i] < g.nq ? 0 : hh[i] < g.nq + g.nkv ? 1 : 2;
      hh[i] -= sect[i] == 0 ? 0 : sect[i] == 1 ? g.nq : g.nq + g.nkv;
    }
    bool kv[RB / PR];
#pragma unroll
    for (int b = 0; b < RB / PR; ++b) {
      kv[b] = (rowg * TR + wr * RB + b * PR + odd) * 16 + r_in < R && act[b] != 0;
      const int chunk = spos[b] / g.P;
      spos[b] -= chunk * g.P;                                   // from here on: the token in its page
      page[b] = e.page_map[kv[b] ? (size_t)page[b] * g.mpg + chunk : 0];
    }
    // pair-interleaved tile: lanes cq 0,1 hold x1 = features 8 th + 4 (cq & 1) + j, lanes cq 2,3 the partners x2 = half + the same
    if constexpr (EPI == GEPI_QKV) {
      uint2 sn[CT][RB], cs[CT][RB];                             // (of value tiles, too: not used)
      const uint32_t sign = cq < 2 ? 0x80008000u : 0u;
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const size_t at = (size_t)pos[b] * half + 4 * (cq & 1);
#pragma unroll
        for (int i = 0; i < CT; ++i) {
          sn[i][b] = *reinterpret_cast<const uint2*>(e.rope_sin + at + 8 * th[i]);
          cs[i][b] = *reinterpret_cast<const uint2*>(e.rope_cos + at + 8 * th[i]);
        }
      }
      typedef typename std::conditional<PR == 2, u32x4, u32x2>::type Piece;
      Piece m[CT][RB / PR];
#pragma unroll
      for (int i = 0; i < CT; ++i) {
        if (sect[i] < 2) {
          // first half: bf16(bf16(x1 c) - bf16(x2 s)); second half: bf16(bf16(x2 c) + bf16(x1 s)); two features at a time
#pragma unroll
          for (int b = 0; b < RB; ++b) {
#pragma unroll
            for (int j = 0; j < 4; j += 2) {
              const uint32_t v = pack2(f2bf(tot[i][b][j]), f2bf(tot[i][b][j + 1])), c = j ? cs[i][b].y : cs[i][b].x, s = (j ? sn[i][b].y : sn[i][b].x) ^ sign;
              const auto x = __builtin_amdgcn_permlane32_swap(v, v, false, false);                                     // x1 and x2, on either partner
              const uint32_t other = cq < 2 ? x[1] : x[0];
              const uint32_t a = pack2(f2bf(bflo(v) * bflo(c)), f2bf(bfhi(v) * bfhi(c))), d = pack2(f2bf(bflo(other) * bflo(s)), f2bf(bfhi(other) * bfhi(s)));
              tot[i][b][j] = bflo(a) + bflo(d);
              tot[i][b][j + 1] = bfhi(a) + bfhi(d);
            }
          }
        }
        if (sect[i] == 0 && e.q_scalar != 0.0f) {
#pragma unroll
          for (int b = 0; b < RB; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j) tot[i][b][j] = rbf(tot[i][b][j]) * e.q_scalar;
        }
#pragma unroll
        for (int b = 0; b < RB; b += PR) {
          uint2 o[PR];
#pragma unroll
          for (int k = 0; k < PR; ++k) {
            const f32x4& t = tot[i][b + k];
            o[k] = make_uint2(pack2(f2bf(t[0]), f2bf(t[1])), pack2(f2bf(t[2]), f2bf(t[3])));
          }
          if constexpr (PR == 2) m[i][b / 2] = rows_pair(o[0], o[1]);
          else { m[i][b].x = o[0].x; m[i][b].y = o[0].y; }
          epi_fence(m[i][b / PR]);
        }
      }
      const int qfeat = (cq >= 2 ? half : 0) + (PR == 2 ? 0 : 4 * (cq & 1)), vfeat = PR == 2 ? 8 * (cq >> 1) : 4 * cq;
#pragma unroll
      for (int b = 0; b < RB / PR; ++b) {
        const int row = (rowg * TR + wr * RB + b * PR + odd) * 16 + r_in;
        bf16_t* const qp = e.qbuf + (size_t)row * g.nq * g.hd + qfeat;
        bf16_t* const kp = e.kpages + kpage_off(g, page[b], 0, qfeat >> 3, spos[b]) + (qfeat & 7);
        bf16_t* const vp = e.vpages + vpage_off(g, page[b], 0, spos[b]) + vfeat;
#pragma unroll
        for (int i = 0; i < CT; ++i)
          if (colg * TC + wc * CT + i < ntile && (sect[i] == 0 ? row < R : kv[b])) {
            bf16_t* const to = sect[i] == 0 ? qp + hh[i] * g.hd + 8 * th[i] : sect[i] == 1 ? kp + (hh[i] * (g.hd >> 3) + th[i]) * g.P * 8 : vp + hh[i] * g.P * g.hd + 16 * th[i];
            *reinterpret_cast<Piece*>(to) = m[i][b];
          }
      }
    } else {   // rope_type "llama3.1": f32 tables, one rounding (ixt_rope_pair); the lane's four de-interleaved features are every second feature of the model's order (ixt_qk_feat)
#pragma unroll
      for (int b = 0; b < RB; ++b) {
        const int row = (rowg * TR + wr * RB + b) * 16 + r_in;
#pragma unroll
        for (int i = 0; i < CT; ++i) {
          const int fi = 8 * th[i] + 4 * (cq & 1);
          float v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[j] = rbf(tot[i][b][j]);
            if (sect[i] < 2) {
              const float other = __shfl_xor(v[j], 32, 64);
              float o1, o2;
              ixt_rope_pair(1, e.rope_sin, e.rope_cos, (size_t)pos[b] * half + fi + j, cq < 2 ? v[j] : other, cq < 2 ? other : v[j], o1, o2);
              v[j] = cq < 2 ? o1 : o2;
            }
            if (sect[i] == 0 && e.q_scalar != 0.0f) v[j] = rbf(v[j] * e.q_scalar);
          }
          if (colg * TC + wc * CT + i >= ntile || !(sect[i] == 0 ? row < R : kv[b])) continue;
          if (sect[i] == 2) {
            uint2 ov;
            ov.x = pack2(f2bf(v[0]), f2bf(v[1])); ov.y = pack2(f2bf(v[2]), f2bf(v[3]));
            *reinterpret_cast<uint2*>(e.vpages + vpage_off(g, page[b], hh[i], spos[b]) + th[i] * 16 + cq * 4) = ov;
          } else {
            const int feat = (cq >= 2 ? half : 0) + fi;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
              const int f = ixt_qk_feat(1, feat + j, half);
              if (sect[i] == 0) e.qbuf[((size_t)row * g.nq + hh[i]) * g.hd + f] = f2bf(v[j]);
              else e.kpages[kpage_off(g, page[b], hh[i], f >> 3, spos[b]) + (f & 7)] = f2bf(v[j]);
            }
          }
        }
      }
    }
  }
}
