// ixt_step.h -- the layers of a pass of few rows (R <= 16, llama2 block) as ONE launch (ixt_step.hip).
//
// The five phases of a layer (QKV, attention, output projection, gated units, down projection) depend on each other, but their weights depend on
// nothing.  As launches of their own (ixt_small.h) every phase pays its start, the latency of its first bytes and its tail while the memory idles: 49 us a
// layer for 20 us of bytes.  Here the grid holds the blocks of all phases of all layers in order; a block requests its whole share of the weights (16 KB a
// wave, sixteen waves a CU: 64 MB on the chip, half a layer of the 1B model) and only then waits for the phase before it, so the stream of weights runs through the
// phases' ends, and blocks that exit make room for the next ones.
//
// Progress: a block waits for blocks of lower index only, and those are dispatched before it (each XCD takes its share of the grid in order), so the
// lowest unfinished block never waits for one that has not started, whatever runs beside it and ends by itself.  Two such grids would not: each could hold the
// XCD that the other's lowest block has to start on.  So the host admits one pass with them at a time (ixt_gate.h).  The waits are bounded all the same (step_wait).
// Workgroups that draw their block's index from a counter, and stay, would end beside each other: built, and slower
// (us a step, 1 / 8 slots: 650 / 809 this, 833 / 1316 with the index drawn a block ahead, 780 / 956 behind the block's own wait; the draw holds up the wave's loads behind it).
//
// Data between blocks: written with agent-scope stores (past the XCD's L2), announced by a counter behind the stores' completion, and read by ordinary loads:
// every layer has its own buffers, no block reads a line before it is complete, and a launch starts with clean caches, so no cache can hold an old copy.
// The keys and values of the pages obey that, too: a line that this pass still writes to is not touched ahead of the wait.
//
// The arithmetic is that of k_sdot and k_attn_small, chain by chain, so the results equal theirs bit for bit.
//
// Measured, us a decode step of the 1B model (16 layers), five launches a layer -> this: 1 slot 974 -> 650 (300 keys), 4 slots 1062 -> 723, 8 slots 1174 -> 817, 16 slots
// 1407 -> 1005 (500 keys); the 134M model 418 -> 298 and 589 -> 405.  One slot's layer takes 27 us: projections 3 to 5 each (rows there 0.6, norm 0.5, products and totals 1.2,
// stores until they are visible 0.9), attention 6, arrival to release 0.6 each, and 20 us of bytes beside them.  What it took to get there from 39: sixteen waves a block
// (the norm of the rows is each CU's own work: 8 slots 36.6 -> 31 ms a pass of 32 steps), the down projection's weights in the L2s ahead of time (2 us), arrivals by block over 32
// counters (1 us a phase), keys requested ahead of the wait and one wave for a page's scores and values (2.5 us).
#pragma once
#include "ixt_kernels.h"

#include <type_traits>

enum { STEP_QKV = 0, STEP_ATT, STEP_O, STEP_UP, STEP_DOWN, STEP_PHASES };
#define STEP_NS 32              // counters of a phase, in lines of their own: arrivals on one word take turns (24 on each cost 1 us)
#define STEP_NW 16              // waves of a block; one block a CU

// A layer's weights and pages, as distances in bytes from the launch's workspace: a pointer that a kernel reads from memory is a generic one, and FLAT loads
// hold up the LDS reads behind them.
struct StepLayer { int64_t wqkv, wo, wi, wout, ln1, ln2, kpages, vpages; };

struct StepArgs {
  const StepLayer* layers;
  bf16_t* ws;                   // per layer: q [16][QN], attention [16][QN], hidden [16][E], units [16][F], hidden [16][E]
  size_t lstride;               // elements of a layer's buffers
  const bf16_t* h0;             // [R][E] rows in front of the first layer
  int32_t* cnt;                 // [L][STEP_PHASES][STEP_NS] x 32 words, zero at the start
  IxtWait wait;
  int R, E, F, QN, NQKV, rpl, fresh;       // fresh: positions in front of a row's own that this pass writes, at most
  int nblk[STEP_PHASES], tpb[STEP_PHASES]; // blocks of a phase, tiles of a block
  int per_layer, attw, att_floats, early;   // blocks of a layer; waves and LDS floats of a (row, kv head); blocks of the gated units that start early
  float eps;
  const int32_t *row_slot, *row_pos, *row_active, *page_map;
  const bf16_t *rope_sin, *rope_cos;
  AttnGeom g;
};

template <typename T> __device__ __forceinline__ T* step_at(const StepArgs& a, int64_t off) { return reinterpret_cast<T*>(reinterpret_cast<char*>(a.ws) + off); }
__device__ __forceinline__ void step_st8(bf16_t* p, uint32_t lo, uint32_t hi) {
  __hip_atomic_store(reinterpret_cast<unsigned long long*>(p), (unsigned long long)lo | ((unsigned long long)hi << 32), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int32_t* step_cnt(const StepArgs& a, int layer, int phase) { return a.cnt + ((size_t)layer * STEP_PHASES + phase) * STEP_NS * 32; }

// arrival of a block, by the last of its `waves` storing waves, behind their stores; `met` in LDS is zero
__device__ __forceinline__ void step_arrive(int32_t* cnt, int blk, int waves, int* met) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if ((threadIdx.x & 63) != 0 || (waves > 1 && __hip_atomic_fetch_add(met, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) != waves - 1)) return;
  __hip_atomic_fetch_add(cnt + (blk & (STEP_NS - 1)) * 32, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// The first wave waits until the counters hold all `n` arrivals, the others at the barrier.  Most blocks stand here long before their phase is due: they look at
// one counter now and then until the phase has begun to end, and at all of them, without a pause, from there on.
__device__ __forceinline__ void step_wait(const int32_t* cnt, int n, const IxtWait& w) {
  if (threadIdx.x < 64) {
    const int lane = threadIdx.x & (STEP_NS - 1), mine = (int)blockIdx.x & (STEP_NS - 1);
    const int due = (n + STEP_NS - 1 - lane) / STEP_NS;
    auto look = [&](int i) { return __hip_atomic_load(cnt + i * 32, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
    auto give_up = [&](int it) {         // some block gave up: nobody waits for it
      if (it > w.polls) { ixt_gave_up(w); return true; }
      return (it & 255) == 0 && __hip_atomic_load(w.gave, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
    };
    int it = 0;
    if (mine < n) {
      while (look(mine) == 0) {
        if (give_up(++it)) break;
        __builtin_amdgcn_s_sleep(4);
      }
    }
    while (!__all(look(lane) >= due)) {
      if (give_up(++it)) break;
    }
  }
  __syncthreads();
  asm volatile("" ::: "memory");
}

// One block of a projection: `tpb` tiles of 16 columns x the chains of K, one (tile, chain) a wave: 16 KB of weights in its registers.  NORM: the rows are normed on
// the way into LDS, as k_sdot does.
template <int PHASE>
__device__ __forceinline__ void step_dot(const StepArgs& a, int layer, int blk, u32x4* sx) {
  constexpr bool NORM = PHASE == STEP_QKV || PHASE == STEP_UP;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const StepLayer& L = a.layers[layer];
  const u32x4* w = step_at<const u32x4>(a, PHASE == STEP_QKV ? L.wqkv : PHASE == STEP_O ? L.wo : PHASE == STEP_UP ? L.wi : L.wout);
  const int K = PHASE == STEP_O ? a.QN : PHASE == STEP_DOWN ? a.F : a.E;
  const int N = PHASE == STEP_QKV ? a.NQKV : PHASE == STEP_UP ? 2 * a.F : a.E;
  const int R = a.R, E = a.E, tpb = a.tpb[PHASE];
  const int nsteps = K >> 5, nc = (nsteps + 15) >> 4, ntile = N >> 4;
  const int row = lane & 15, cq = lane >> 4;
  const bool row_ok = row < R;

  __shared__ int met;
  if (tid == 0) met = 0;
  // ---- this wave's weights, all in flight
  const int t = wave % tpb, c = wave / tpb, tile = blk * tpb + t;
  const bool live = c < nc && tile < ntile;
  const int cs = live ? min(16, nsteps - c * 16) : 1;              // steps of the chain (a short last chain reads its last fragment again, unused)
  const u32x4* wbase = w + (live ? ((size_t)tile * nsteps + c * 16) * 64 : 0) + lane;
  u32x4 wv[16];
  if (live) {
#pragma unroll
    for (int s = 0; s < 16; ++s) wv[s] = __builtin_nontemporal_load(wbase + (size_t)min(s, cs - 1) * 64);
  }
  if constexpr (PHASE == STEP_UP) {
    // The units' blocks fill the chip while they wait, and the memory would idle until they end: they pull the down projection's weights -- of the blocks that will
    // run on their XCD (the grid is dealt to the XCDs in turn) -- into its L2.  Only those that start beside the attention do.
    const int dn0 = (int)blockIdx.x - blk + a.nblk[STEP_UP], first = ((int)blockIdx.x - dn0) & 7;      // this XCD's down blocks: first, first + 8, ...
    const int dsteps = a.F >> 5, per = a.tpb[STEP_DOWN] * dsteps, pieces = ((a.nblk[STEP_DOWN] - first + 7) >> 3) * per;      // fragments of 1 KB
    const u32x4* wd = step_at<const u32x4>(a, L.wout);
    if (blk < a.early) {
      for (int p0 = (blk >> 3) * STEP_NW + wave; p0 < pieces; p0 += 8 * (a.early >> 3) * STEP_NW) {
        u32x4 v[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int p = min(p0 + i * (a.early >> 3) * STEP_NW, pieces - 1), b = p / per, f = (first + 8 * b) * per + (p - b * per);
          v[i] = wd[(size_t)min(f, (E >> 4) * dsteps - 1) * 64 + lane];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) asm volatile("" ::"v"(v[i].x), "v"(v[i].y), "v"(v[i].z), "v"(v[i].w));
      }
    }
  }
  // what the epilogue needs of the rows, too
  const AttnGeom& g = a.g;
  const int half = g.hd >> 1, tph = g.hd >> 4, th = tile % tph;
  int pos = 0, page = 0;
  bool wr_kv = false;
  uint2 sv{0, 0}, cv{0, 0};
  if constexpr (PHASE == STEP_QKV) {
    if (c == 0 && row_ok) {
      pos = a.row_pos[row];
      wr_kv = a.row_active[row] != 0;
      if (wr_kv) page = a.page_map[(size_t)a.row_slot[row] * g.mpg + pos / g.P];
    }
    if (c == 0 && !g.rope32) {
      const size_t at = (size_t)pos * half + 8 * th + 4 * (cq & 1);
      sv = *reinterpret_cast<const uint2*>(a.rope_sin + at);
      cv = *reinterpret_cast<const uint2*>(a.rope_cos + at);
    }
  }

  // a wave norms the same 64 chunks of every row it has
  const int nch = K >> 3, nb = (nch + 63) >> 6;
  const int lb = nb == 1 ? 0 : nb == 2 ? 1 : 2;                    // unit u: 64 chunks of row u >> lb (three of a row are dealt as four)
  const int ch = (wave & ((1 << lb) - 1)) * 64 + lane;
  u32x4 scv{0, 0, 0, 0};
  if constexpr (NORM) scv = *reinterpret_cast<const u32x4*>(step_at<const bf16_t>(a, PHASE == STEP_QKV ? L.ln1 : L.ln2) + min(ch, nch - 1) * 8);

  // ---- the phase before
  bf16_t* ws = a.ws + (size_t)layer * a.lstride;
  bf16_t* q = ws;
  bf16_t* ao = q + (size_t)16 * a.QN;
  bf16_t* hm = ao + (size_t)16 * a.QN;
  bf16_t* act = hm + (size_t)16 * E;
  bf16_t* hout = act + (size_t)16 * a.F;
  const bf16_t* hin = layer == 0 ? a.h0 : a.ws + (size_t)layer * a.lstride - (size_t)16 * E;
  if (PHASE == STEP_QKV) {
    if (layer > 0) step_wait(step_cnt(a, layer - 1, STEP_DOWN), a.nblk[STEP_DOWN], a.wait);
  } else {
    step_wait(step_cnt(a, layer, PHASE - 1), a.nblk[PHASE - 1], a.wait);
  }

  f32x4 acc = f32x4(0.0f);
  f32x4* red;
  uint2 hv{0, 0};
  if constexpr (NORM) {
    // rows -> registers (wave = (row, 64 chunks of 8), lane = chunk: the unit of the canonical sum of squares) -> normed -> LDS, row-compact.  The rows of a chunk
    // are rotated by the chunk's index, or the lanes' writes would meet in few banks.
    const bf16_t* x = PHASE == STEP_QKV ? hin : hm;
    const int rpl = a.rpl, Rp = 1 << rpl;
    red = reinterpret_cast<f32x4*>(sx + ((size_t)nch << rpl));
    float* bsum = reinterpret_cast<float*>(red + STEP_NW * 64);   // [64]: the units' sums
    constexpr int NU = 64 / STEP_NW;
    u32x4 hx[NU];
    const int slots = R << lb;                                    // <= 64
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = wave + STEP_NW * i, rw = u >> lb;
      if (u < slots) hx[i] = *reinterpret_cast<const u32x4*>(x + (size_t)rw * K + min(ch, nch - 1) * 8);
    }
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = wave + STEP_NW * i;
      if (u < slots) {
        const float h[8] = {bflo(hx[i].x), bfhi(hx[i].x), bflo(hx[i].y), bfhi(hx[i].y), bflo(hx[i].z), bfhi(hx[i].z), bflo(hx[i].w), bfhi(hx[i].w)};
        float v = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; ++j) v = __builtin_fmaf(h[j], h[j], v);
        v = ch < nch ? v : 0.0f;
        v = xor_sum(v);
        if (lane == 0) bsum[u] = v;
      }
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < NU; ++i) {
      const int u = wave + STEP_NW * i, rw = u >> lb;
      if (u < slots) {
        float bs[4], total = 0.0f;
#pragma unroll
        for (int b = 0; b < 4; ++b) bs[b] = bsum[(rw << lb) + min(b, nb - 1)];
#pragma unroll
        for (int b = 0; b < 4; ++b) total = b < nb ? total + bs[b] : total;
        const float rs = 1.0f / sqrtf(total / (float)K + a.eps);
        if (ch < nch) {
          const float h[8] = {bflo(hx[i].x), bfhi(hx[i].x), bflo(hx[i].y), bfhi(hx[i].y), bflo(hx[i].z), bfhi(hx[i].z), bflo(hx[i].w), bfhi(hx[i].w)};
          const float sc[8] = {bflo(scv.x), bfhi(scv.x), bflo(scv.y), bfhi(scv.y), bflo(scv.z), bfhi(scv.z), bflo(scv.w), bfhi(scv.w)};
          bf16_t o[8];
#pragma unroll
          for (int j = 0; j < 8; ++j) o[j] = f2bf(rbf(h[j] * rs) * sc[j]);
          u32x4 ov;
          ov.x = pack2(o[0], o[1]); ov.y = pack2(o[2], o[3]); ov.z = pack2(o[4], o[5]); ov.w = pack2(o[6], o[7]);
          sx[((size_t)ch << rpl) + (rw ^ (ch & (Rp - 1)))] = ov;
        }
      }
    }
    __syncthreads();
  } else {
    const bf16_t* x = PHASE == STEP_O ? ao : act;
    const int rpl = a.rpl, Rp = 1 << rpl, np = nch << rpl;
    if (c == 0 && live && row_ok) hv = *reinterpret_cast<const uint2*>((PHASE == STEP_O ? hin : hm) + (size_t)row * E + tile * 16 + cq * 4);   // the residual of what this wave will store
    if (np <= 8 * STEP_NW * 64) {
      // the rows through LDS: one round of loads (a fragment straight from memory has idle lanes for the rows that are not there, and its sixteen steps take two)
      red = reinterpret_cast<f32x4*>(sx + np);
      u32x4 xv[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int p = tid + i * STEP_NW * 64;
        if (p - lane < np) xv[i] = *reinterpret_cast<const u32x4*>(x + (size_t)min((p & (Rp - 1)) ^ ((p >> rpl) & (Rp - 1)), R - 1) * K + min(p >> rpl, nch - 1) * 8);
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int p = tid + i * STEP_NW * 64;
        if (p < np) sx[p] = xv[i];
      }
      __syncthreads();
    } else {
      red = reinterpret_cast<f32x4*>(sx);
    }
    if (live && np > 8 * STEP_NW * 64) {
      const bf16_t* xb = x + (size_t)min(row, R - 1) * K + c * 512 + cq * 8;
#pragma unroll
      for (int s0 = 0; s0 < 16; s0 += 8) {
        u32x4 xv[8];
#pragma unroll
        for (int s = 0; s < 8; ++s) xv[s] = *reinterpret_cast<const u32x4*>(xb + min(s0 + s, cs - 1) * 32);
#pragma unroll
        for (int s = 0; s < 8; ++s)
          if (s0 + s < cs) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[s0 + s]), __builtin_bit_cast(bf16x8, xv[s]), acc, 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if (live && (NORM || (nch << a.rpl) <= 8 * STEP_NW * 64)) {
    const int rpl = a.rpl, Rp = 1 << rpl;
    auto product = [&](int s) {
      const int ck = (c * 16 + s) * 4 + cq;
      const bf16x8 xv = __builtin_bit_cast(bf16x8, sx[((size_t)ck << rpl) + ((row ^ ck) & (Rp - 1))]);
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[s]), xv, acc, 0, 0, 0);
    };
    if (cs == 16) {
#pragma unroll
      for (int s = 0; s < 16; ++s) {
        product(s);
        if ((s & 3) == 3) __builtin_amdgcn_sched_barrier(0);
      }
    } else {
#pragma unroll
      for (int s = 0; s < 16; ++s) if (s < cs) product(s);
    }
  }

  // ---- chain totals meet in LDS; the waves of chain 0 add them in order
  if (live) red[((size_t)c * tpb + t) * 64 + lane] = acc;
  __syncthreads();
  if (c != 0 || !live) return;
  if (PHASE == STEP_UP && (t & 1)) return;        // the wi_1 tile's totals are taken by the wi_0 tile's wave
  f32x4 tot = f32x4(0.0f), tot2 = f32x4(0.0f);
  auto total = [&](auto most) {                   // `most` chains at most, all reads ahead of the adds
    constexpr int MC = decltype(most)::value;
    f32x4 v4[MC], w4[MC];
#pragma unroll
    for (int cc = 0; cc < MC; ++cc) {
      v4[cc] = red[((size_t)min(cc, nc - 1) * tpb + t) * 64 + lane];
      if (PHASE == STEP_UP) w4[cc] = red[((size_t)min(cc, nc - 1) * tpb + t + 1) * 64 + lane];
    }
#pragma unroll
    for (int cc = 0; cc < MC; ++cc) {
      if (cc < nc) { tot = tot + v4[cc]; if (PHASE == STEP_UP) tot2 = tot2 + w4[cc]; }
    }
  };
  if (NORM || nc <= 4) total(std::integral_constant<int, 4>());
  else total(std::integral_constant<int, 16>());

  if constexpr (PHASE == STEP_O || PHASE == STEP_DOWN) {
    if (row_ok) {
      bf16_t* dst = (PHASE == STEP_O ? hm : hout) + (size_t)row * E + tile * 16 + cq * 4;
      step_st8(dst, pack2(f2bf(bflo(hv.x) + rbf(tot[0])), f2bf(bfhi(hv.x) + rbf(tot[1]))), pack2(f2bf(bflo(hv.y) + rbf(tot[2])), f2bf(bfhi(hv.y) + rbf(tot[3]))));
    }
    step_arrive(step_cnt(a, layer, PHASE), blk, min(tpb, ntile - blk * tpb), &met);
  } else if constexpr (PHASE == STEP_UP) {
    if (row_ok) {
      bf16_t o[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) o[j] = ixt_swiglu(rbf(tot[j]), rbf(tot2[j]));
      step_st8(act + (size_t)row * a.F + (tile >> 1) * 16 + cq * 4, pack2(o[0], o[1]), pack2(o[2], o[3]));
    }
    step_arrive(step_cnt(a, layer, PHASE), blk, min(tpb, ntile - blk * tpb) / 2, &met);
  } else {
    bf16_t *kpages = step_at<bf16_t>(a, L.kpages), *vpages = step_at<bf16_t>(a, L.vpages);
    // bf16(t), RoPE by partner exchange across lanes l and l ^ 32, q -> its buffer, K / V -> the row's page (k_sdot's epilogue)
    const int QN = g.nq * g.hd, KN = g.nkv * g.hd;
    const int tok = pos % g.P;
    const int col0 = tile * 16;
    float v[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) v[j] = rbf(tot[j]);
    const bool is_v = col0 >= QN + KN;
    const int hh = col0 / g.hd;
    if (!is_v) {
      const int fi = 8 * th + 4 * (cq & 1);
      if (g.rope32) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float other = __shfl_xor(v[j], 32, 64);
          float o1, o2;
          ixt_rope_pair(1, a.rope_sin, a.rope_cos, (size_t)pos * half + fi + j, cq < 2 ? v[j] : other, cq < 2 ? other : v[j], o1, o2);
          v[j] = cq < 2 ? o1 : o2;
        }
      } else {
        const float sn[4] = {bflo(sv.x), bfhi(sv.x), bflo(sv.y), bfhi(sv.y)}, cs_[4] = {bflo(cv.x), bfhi(cv.x), bflo(cv.y), bfhi(cv.y)};
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float other = __shfl_xor(v[j], 32, 64);
          v[j] = cq < 2 ? rbf(rbf(v[j] * cs_[j]) - rbf(other * sn[j])) : rbf(rbf(v[j] * cs_[j]) + rbf(other * sn[j]));
        }
      }
    }
    if (row_ok) {
      const uint32_t lo = pack2(f2bf(v[0]), f2bf(v[1])), hi = pack2(f2bf(v[2]), f2bf(v[3]));
      const int feat = is_v ? th * 16 + cq * 4 : (cq >= 2 ? half : 0) + 8 * th + 4 * (cq & 1);
      if (g.rope32 && !is_v) {   // llama3.1: the lane's four de-interleaved features are every second feature of the model's order (ixt_qk_feat)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int fn_ = ixt_qk_feat(1, feat + j, half);
          bf16_t* dst = hh < g.nq ? q + ((size_t)row * g.nq + hh) * g.hd + fn_ : kpages + kpage_off(g, page, hh - g.nq, fn_ >> 3, tok) + (fn_ & 7);
          if (hh < g.nq || wr_kv) __hip_atomic_store(dst, f2bf(v[j]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      } else if (hh < g.nq) {
        step_st8(q + ((size_t)row * g.nq + hh) * g.hd + feat, lo, hi);
      } else if (wr_kv) {
        if (!is_v) step_st8(kpages + kpage_off(g, page, hh - g.nq, feat >> 3, tok) + (feat & 7), lo, hi);
        else step_st8(vpages + vpage_off(g, page, hh - g.nq - g.nkv, tok) + feat, lo, hi);
      }
    }
    step_arrive(step_cnt(a, layer, PHASE), blk, min(tpb, ntile - blk * tpb), &met);
  }
}

// Attention, k_attn_small's order of operations on pages of 32 tokens.  A (row, kv head) has `attw` waves, a block one or two of them.  Wave w has the 64 keys (two pages) from
// 64 w on, and those 64 attw, 128 attw ... further: it takes their scores (lane = key) and their values (half a wave a page).  Between the waves go the maxima, the page sums and the
// pages' outputs.  Ahead of the wait: a wave's first keys come into registers as far as this pass does not write them, all others into the XCD's L2.
template <int HD, int GQ>
__device__ __forceinline__ void step_attn(const StepArgs& a, int layer, int blk, float* sm) {
  static_assert(HD == 64 || HD == 128, "16 bytes of a key's half, two or four columns a lane");
  constexpr int KC = HD / 8, VD = HD / 32;         // chunks of a key; columns of a lane
  const AttnGeom& g = a.g;
  const bf16_t *kpages = step_at<const bf16_t>(a, a.layers[layer].kpages), *vpages = step_at<const bf16_t>(a, a.layers[layer].vpages);
  __shared__ int met;
  if (threadIdx.x == 0) met = 0;
  const int lane = threadIdx.x & 63, aw = a.attw, nt = aw * 64;
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) & (aw - 1), sub = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6) / aw;
  const int tid = wave * 64 + lane;              // of the pair's threads
  const int npair = a.R * g.nkv, per_blk = STEP_NW / aw, pair = blk * per_blk + sub;
  const bool there = pair < npair;
  const int r = min(pair, npair - 1) / g.nkv, kvh = min(pair, npair - 1) - r * g.nkv;
  const bf16_t* qsrc = a.ws + (size_t)layer * a.lstride + ((size_t)r * g.nq + kvh * GQ) * HD;
  bf16_t* out = a.ws + (size_t)layer * a.lstride + (size_t)16 * a.QN + ((size_t)r * g.nq + kvh * GQ) * HD;
  const int tp = (g.Tmax + 63) & ~63, mpgp = (g.mpg + 3) & ~3;
  float* qs = sm + (size_t)sub * a.att_floats;   // [GQ][HD]
  float* ebuf = qs + GQ * HD;                    // [GQ][Tmax'] scores, exps, weights
  float* psum = ebuf + (size_t)GQ * tp;          // [GQ][mpg']
  int32_t* pm = reinterpret_cast<int32_t*>(psum + GQ * mpgp);   // [mpg'] the row's page list
  float* wred = reinterpret_cast<float*>(pm + mpgp);            // [GQ][16]
  float* pacc = wred + GQ * STEP_NW;             // [GQ][mpg'][HD] the pages' outputs
  const bool active = there && a.row_active[r] != 0;
  const int pos = active ? a.row_pos[r] : -1, kv_len = pos + 1, pages = (kv_len + 31) >> 5;
  const int old = max(pos - a.fresh, 0) & ~7;    // keys whose cache lines (8 tokens of 16 bytes) this pass does not write
  const int j0 = wave * 64 + lane;
  u32x4 k[KC];
  auto kload = [&](int j) {
    const bf16_t* kp = kpages + kpage_off(g, pm[j >> 5], kvh, 0, j & 31);
#pragma unroll
    for (int d = 0; d < KC; ++d) k[d] = *reinterpret_cast<const u32x4*>(kp + d * 256);
  };
  if (active) {
    const int32_t* prow = a.page_map + (size_t)a.row_slot[r] * g.mpg;
    for (int i = tid; i < pages; i += nt) pm[i] = prow[i];
  }
  __syncthreads();
  if (active) {
    if (j0 < old) kload(j0);
    const int per = HD * 4;                      // 16-byte pieces of a page of one head
    auto touch = [&](const bf16_t* pool, int from, int to) {       // pieces of the row's pages, four in flight
      for (int i0 = from + tid; i0 < to; i0 += 4 * nt) {
        u32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = min(i0 + u * nt, to - 1), p = i / per;
          v[u] = reinterpret_cast<const u32x4*>(pool + vpage_off(g, pm[p], kvh, 0))[i - p * per];
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) asm volatile("" ::"v"(v[u].x), "v"(v[u].y), "v"(v[u].z), "v"(v[u].w));
      }
    };
    touch(vpages, 0, (old >> 3) * (per / 4));
    touch(kpages, 2 * aw * per, (old >> 5) * per);                 // (a page of keys is as large as one of values)
  }
  step_wait(step_cnt(a, layer, STEP_QKV), a.nblk[STEP_QKV], a.wait);
  for (int i = tid; i < GQ * HD; i += nt) qs[i] = bf2f(qsrc[i]);
  if (j0 >= old && j0 < kv_len) kload(j0);
  __syncthreads();
  float mx[GQ];
#pragma unroll
  for (int q = 0; q < GQ; ++q) mx[q] = -INFINITY;
#pragma unroll 1
  for (int j = j0; j - lane < kv_len; j += nt) {       // (uniform)
    float s[GQ];
#pragma unroll
    for (int q = 0; q < GQ; ++q) s[q] = 0.0f;
#pragma unroll
    for (int d = 0; d < KC; ++d) {
      const float kf[8] = {bflo(k[d].x), bfhi(k[d].x), bflo(k[d].y), bfhi(k[d].y), bflo(k[d].z), bfhi(k[d].z), bflo(k[d].w), bfhi(k[d].w)};
#pragma unroll
      for (int q = 0; q < GQ; ++q) {
        const float4 qa = *reinterpret_cast<const float4*>(qs + q * HD + d * 8);
        const float4 qb = *reinterpret_cast<const float4*>(qs + q * HD + d * 8 + 4);
        s[q] = __builtin_fmaf(qa.x, kf[0], s[q]); s[q] = __builtin_fmaf(qa.y, kf[1], s[q]); s[q] = __builtin_fmaf(qa.z, kf[2], s[q]); s[q] = __builtin_fmaf(qa.w, kf[3], s[q]);
        s[q] = __builtin_fmaf(qb.x, kf[4], s[q]); s[q] = __builtin_fmaf(qb.y, kf[5], s[q]); s[q] = __builtin_fmaf(qb.z, kf[6], s[q]); s[q] = __builtin_fmaf(qb.w, kf[7], s[q]);
      }
      if (d & 1) __builtin_amdgcn_sched_barrier(0);   // (the queries' reads of all chunks at once would take the file)
    }
#pragma unroll
    for (int q = 0; q < GQ; ++q) asm volatile("" : "+v"(s[q]));  // done here, not where the score is stored
    if (j + nt < kv_len) kload(j + nt);
#pragma unroll
    for (int q = 0; q < GQ; ++q) {
      mx[q] = j < kv_len ? fmaxf(mx[q], s[q]) : mx[q];
      ebuf[(size_t)q * tp + j] = s[q];
    }
  }
  // the values of this wave's first pages: in flight under the softmax
  const int hw = lane >> 5, dc = lane & 31;
  uint32_t vv[32][VD / 2];
  auto vload = [&](int p) {
    if (p < pages) {
      const bf16_t* vp = vpages + vpage_off(g, pm[p], kvh, 0) + dc * VD;
      const int last = min(32, kv_len - p * 32) - 1;
#pragma unroll
      for (int u = 0; u < 32; ++u) {
        if constexpr (VD == 4) { const uint2 w = *reinterpret_cast<const uint2*>(vp + min(u, last) * HD); vv[u][0] = w.x; vv[u][1] = w.y; }
        else vv[u][0] = *reinterpret_cast<const uint32_t*>(vp + min(u, last) * HD);
      }
    }
  };
  vload(2 * wave + hw);
#pragma unroll
  for (int q = 0; q < GQ; ++q) {
    mx[q] = xor_butterfly(mx[q], [](float x, float y) { return fmaxf(x, y); });
    if (lane == 0) wred[q * STEP_NW + wave] = mx[q];
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < GQ; ++q) {
    float m = wred[q * STEP_NW + (lane & (aw - 1))];
    m = xor_butterfly(m, [](float x, float y) { return fmaxf(x, y); });
    float* e = ebuf + (size_t)q * tp;
#pragma unroll 1
    for (int j = j0; j - lane < kv_len; j += nt) e[j] = ixt_exp(e[j] - m);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");         // a page's exps are added by a lane of the wave that wrote them
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // lane = (page of the tile, query head)
  for (int p = 2 * wave + (lane & 1); p < pages && lane < 2 * GQ; p += 2 * aw) {
    const int q = lane >> 1, n = min(32, kv_len - p * 32);
    const float* ep = ebuf + (size_t)q * tp + p * 32;
    float4 x[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) x[u] = *reinterpret_cast<const float4*>(ep + 4 * u);
    float sum = 0.0f;
    if (n == 32) {
#pragma unroll
      for (int u = 0; u < 8; ++u) { sum = sum + x[u].x; sum = sum + x[u].y; sum = sum + x[u].z; sum = sum + x[u].w; }
    } else
#pragma unroll
    for (int u = 0; u < 8; ++u) {
      sum = 4 * u < n ? sum + x[u].x : sum;
      sum = 4 * u + 1 < n ? sum + x[u].y : sum;
      sum = 4 * u + 2 < n ? sum + x[u].z : sum;
      sum = 4 * u + 3 < n ? sum + x[u].w : sum;
    }
    psum[q * mpgp + p] = sum;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < GQ; ++q) {
    float l = 0.0f;
    int p = 0;
    for (; p + 4 <= pages; p += 4) {
      const float4 x = *reinterpret_cast<const float4*>(psum + q * mpgp + p);
      l = l + x.x; l = l + x.y; l = l + x.z; l = l + x.w;
    }
    for (; p < pages; ++p) l = l + psum[q * mpgp + p];
#pragma unroll 1
    for (int j = j0; j - lane < kv_len; j += nt) ebuf[(size_t)q * tp + j] = rbf(ebuf[(size_t)q * tp + j] / l);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");         // the weights of a page are read by the wave that wrote them
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  for (int p = 2 * wave + hw, first = 1; p - hw < pages; p += 2 * aw, first = 0) {
    if (!first) vload(p);
    if (p < pages) {
      float acc[GQ][VD];
#pragma unroll
      for (int q = 0; q < GQ; ++q)
#pragma unroll
        for (int x = 0; x < VD; ++x) acc[q][x] = 0.0f;
      const int n = min(32, kv_len - p * 32);
      auto sum = [&](auto whole) {
#pragma unroll
        for (int u0 = 0; u0 < 32; u0 += 4) {
          if (whole.value || u0 < n) {
#pragma unroll
            for (int q = 0; q < GQ; ++q) {
              const float4 pv4 = *reinterpret_cast<const float4*>(ebuf + (size_t)q * tp + p * 32 + u0);
              const float pv[4] = {pv4.x, pv4.y, pv4.z, pv4.w};
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                if (whole.value || u0 + u < n) {
#pragma unroll
                  for (int x = 0; x < VD; x += 2) {
                    acc[q][x] = __builtin_fmaf(pv[u], bflo(vv[u0 + u][x / 2]), acc[q][x]);
                    acc[q][x + 1] = __builtin_fmaf(pv[u], bfhi(vv[u0 + u][x / 2]), acc[q][x + 1]);
                  }
                }
              }
            }
          }
          if (u0 & 4) __builtin_amdgcn_sched_barrier(0);
        }
      };
      if (__all(n == 32)) sum(std::true_type());
      else sum(std::false_type());
#pragma unroll
      for (int q = 0; q < GQ; ++q)
#pragma unroll
        for (int x = 0; x < VD; x += 2) *reinterpret_cast<float2*>(pacc + ((size_t)q * mpgp + p) * HD + dc * VD + x) = make_float2(acc[q][x], acc[q][x + 1]);
    }
  }
  __syncthreads();
  if (there && tid < GQ * HD / 4) {              // four pages added in order, then the super-blocks
    const int q = tid / (HD / 4);
    const float* pq = pacc + (size_t)q * mpgp * HD + (tid - q * (HD / 4)) * 4;
    f32x4 tot = f32x4(0.0f);
    for (int p = 0; p < pages; p += IXT_SB) {
      f32x4 ss = f32x4(0.0f);
#pragma unroll
      for (int i = 0; i < IXT_SB; ++i) if (p + i < pages) ss = ss + *reinterpret_cast<const f32x4*>(pq + (size_t)(p + i) * HD);
      tot = tot + ss;
    }
    step_st8(out + tid * 4, pack2(f2bf(tot[0]), f2bf(tot[1])), pack2(f2bf(tot[2]), f2bf(tot[3])));
  }
  if (there && wave == 0) step_arrive(step_cnt(a, layer, STEP_ATT), blk, min(per_blk, npair - blk * per_blk), &met);   // (a pair's stores are this wave's: at most 64 lanes)
}

template <int HD, int GQ>
__global__ __launch_bounds__(STEP_NW * 64, STEP_NW / 4) void k_step(StepArgs a) {
  extern __shared__ __attribute__((aligned(16))) u32x4 step_lds[];
  const int layer = blockIdx.x / a.per_layer;
  int b = blockIdx.x - layer * a.per_layer;
  if (b < a.nblk[STEP_QKV]) { step_dot<STEP_QKV>(a, layer, b, step_lds); return; }
  b -= a.nblk[STEP_QKV];
  if (b < a.nblk[STEP_ATT]) { step_attn<HD, GQ>(a, layer, b, reinterpret_cast<float*>(step_lds)); return; }
  b -= a.nblk[STEP_ATT];
  if (b < a.nblk[STEP_O]) { step_dot<STEP_O>(a, layer, b, step_lds); return; }
  b -= a.nblk[STEP_O];
  if (b < a.nblk[STEP_UP]) { step_dot<STEP_UP>(a, layer, b, step_lds); return; }
  step_dot<STEP_DOWN>(a, layer, b - a.nblk[STEP_UP], step_lds);
}

// rows of the embedding in front of the first layer; the counters of the launch behind it, and the pass's word of waits given up.  (Decode rows: k_decode_front.)
static __global__ __launch_bounds__(256) void k_step_begin(const int32_t* tokens, FrontRows f, int32_t* gave) {
  front_row(f, blockIdx.x, gridDim.x, tokens[blockIdx.x]);
  if (blockIdx.x == 0 && threadIdx.x == 0) *gave = 0;
}
