// ixt_mid.h -- passes of 17 to 64 rows (llama2 block): what lies between two attentions as ONE launch (ixt_step.hip).
//
// Attention of such rows runs at the memory's rate as a launch of its own.  The six phases behind it -- output projection, norm, gated units, down projection,
// norm, the next layer's QKV -- took a launch each, 4.7 to 14.4 us for 20 us of weights a layer.  Here they share a launch in k_step's manner (ixt_step.h says why its waits
// end and how data passes between blocks): a block requests its weights, 32 KB a wave, and then waits for the phase before.
//
// A block has 16 units = (tile of 16 columns, chain of 512 k), two a wave, so that a fragment of the rows is read once for two tiles: with one, the LDS port would bound the products
// (1 KB a product of 16 cycles on each of four SIMDs, at 128 B a cycle).  Rows come in groups of 16 through two LDS buffers by LDS-DMA where the units of a block
// share them (K <= 2048); where a block's units are the chains of one tile, each wave reads its own, straight into registers.
// The norms are phases of their own, a wave a row: every block norming all rows, as k_step does for up to 16, would cost 8 us at 64.
//
// Measured, 1B model, ms a pass, a launch a phase -> this: decode steps (32 a pass, 300 keys) of 17 slots 43.5 -> 36.3, 32 slots 46.3 -> 38.8, 33 slots 45.8 -> 41.4, 64 slots 52.6 ->
// 49.1; a prompt of 17 tokens 1.24 -> 1.05, of 57 1.35 -> 1.25.  A launch of 48 rows takes 43 us: output projection 12 (the weights of all phases are on their way beside it), norms 4 each, units 7,
// down projection 10, QKV 6; 20 us of weights lie beside them.  What took it there from 59: whole lines from the norms, the down projection's weights in the L2s ahead of time and
// its row groups in two blocks (3 us), angles ahead of the wait, QKV over twice the blocks (2 us; the CUs are free for its weights only when the down projection ends).  Tried
// without gain: QKV's weights pulled into the L2s by waves of the down projection that have no unit (+8 us: their block ends later), the pull of the down projection's weights held back until the output projection
// is through (+2), the units' weights held back by 2 us (level).
//
// The arithmetic is the canonical one, chain by chain, so the results equal those of the other paths bit for bit.
#pragma once
#include "ixt_step.h"

enum { MID_O = 0, MID_N2, MID_UP, MID_DOWN, MID_N1, MID_QKV, MID_PHASES };
#define MID_NW 8
#define MID_BUF_STEPS 64        // fragments of k in one LDS buffer

struct MidArgs {
  const StepLayer* layers;
  bf16_t* base;                 // what StepLayer's distances start from
  int layer, next;              // the layer of O .. DOWN, and of N1 / QKV (-1: not in this launch)
  const bf16_t *ao, *hin, *scale;        // attention's output (xidx), rows [64][E]; N1's scale (next layer's, or the head's)
  bf16_t *hmid, *hout, *xn1, *xn2, *act, *qbuf;   // rows, rows, operands in xidx layout
  int32_t* cnt;                 // [MID_PHASES][STEP_NS] lines of this launch
  IxtWait wait;
  int R, E, F, QN, NQKV;
  int early;                    // blocks of the gated units that start beside the output projection
  int nblk[MID_PHASES], tpb[MID_PHASES], prev[MID_PHASES];     // blocks, tiles of a block; the phase to wait for (-1: none)
  float eps;
  const int32_t *row_slot, *row_pos, *row_active, *page_map;
  const bf16_t *rope_sin, *rope_cos;
  AttnGeom g;
};
template <typename T> __device__ __forceinline__ T* mid_at(const MidArgs& a, int64_t off) { return reinterpret_cast<T*>(reinterpret_cast<char*>(a.base) + off); }
__device__ __forceinline__ int32_t* mid_cnt(const MidArgs& a, int phase) { return a.cnt + (size_t)phase * STEP_NS * 32; }
__device__ __forceinline__ void mid_wait(const MidArgs& a, int phase) {
  if (a.prev[phase] >= 0) step_wait(mid_cnt(a, a.prev[phase]), a.nblk[a.prev[phase]], a.wait);
  else __syncthreads();
}

// Weights of phase `to` (kernel at `off`, K x ntile tiles), of those of its `nb` blocks that will run on this XCD (the grid, from block p0 on, is dealt to the XCDs in turn), into its L2:
// share `me` of `shares`.  Fetched to 1 KB of LDS that nobody reads: a load to registers would hold its wave up.
__device__ __forceinline__ void mid_touch(const MidArgs& a, int to, int64_t off, int K, int ntile, int p0, int nb, int me, int shares, u32x4* spare) {
  const int lane = threadIdx.x & 63, first = ((int)blockIdx.x - p0) & 7, per = a.tpb[to] * (K >> 5), pieces = ((nb - first + 7) >> 3) * per, all = ntile * (K >> 5);
  const u32x4* w = mid_at<const u32x4>(a, off);
  const uint32_t dst = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)((__attribute__((address_space(3))) u32x4*)spare));
  for (int q = me; q < pieces; q += shares) {
    const int b = q / per;
    lds_dma16(dst, w + (size_t)min((first + 8 * b) * per + (q - b * per), all - 1) * 64 + lane);
  }
}

// GT row groups in all; the down projection's blocks take half of them each (MID_SPLIT blocks a tile, eight blocks apart: on the same XCD)
#define MID_SPLIT 2
template <int PHASE, int GT>
__device__ __forceinline__ void mid_dot(const MidArgs& a, int blk, u32x4* sx) {
  constexpr int G = PHASE == MID_DOWN ? (GT + MID_SPLIT - 1) / MID_SPLIT : GT;
  const int blk_all = blk, g0 = PHASE == MID_DOWN ? (blk >> 3 & (MID_SPLIT - 1)) * G : 0;       // the first group
  if (PHASE == MID_DOWN) blk = (blk >> 3) / MID_SPLIT * 8 + (blk & 7);
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const StepLayer& L = a.layers[PHASE == MID_QKV ? a.next : a.layer];
  const u32x4* w = mid_at<const u32x4>(a, PHASE == MID_QKV ? L.wqkv : PHASE == MID_O ? L.wo : PHASE == MID_UP ? L.wi : L.wout);
  const u32x4* x = reinterpret_cast<const u32x4*>(PHASE == MID_QKV ? a.xn1 : PHASE == MID_O ? a.ao : PHASE == MID_UP ? a.xn2 : a.act + (size_t)g0 * 16 * a.F);
  const int K = PHASE == MID_O ? a.QN : PHASE == MID_DOWN ? a.F : a.E;
  const int N = PHASE == MID_QKV ? a.NQKV : PHASE == MID_UP ? 2 * a.F : a.E;
  const int R = a.R - g0 * 16, E = a.E, tpb = a.tpb[PHASE];      // rows from this block's first group on
  const int nsteps = K >> 5, nc = (nsteps + 15) >> 4, ntile = N >> 4;
  const int row = lane & 15, cq = lane >> 4;
  const AttnGeom& g = a.g;
  __shared__ int met, s_pos[PHASE == MID_QKV ? 16 * G : 1], s_page[PHASE == MID_QKV ? 16 * G : 1];       // position of a row; its page, -1: its key and value are not kept
  __shared__ u32x4 s_rope[PHASE == MID_QKV ? 2 * 8 * 16 * G : 1];                                        // [sin, cos][tile][row]: eight angles
  __shared__ __attribute__((aligned(16))) u32x4 spare[PHASE == MID_UP ? 64 : 1];
  if (tid == 0) met = 0;

  // ---- this wave's two units: chain c[i] of tile t[i]; all weights in flight
  u32x4 wv[2][16];
  int c[2], cs[2];
  bool live[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int u = wave * 2 + i, t = u % tpb, tile = blk * tpb + t;
    c[i] = u / tpb;
    live[i] = c[i] < nc && tile < ntile;
    cs[i] = live[i] ? min(16, nsteps - c[i] * 16) : 1;       // (a short last chain reads its last fragment again, unused)
    const u32x4* wb = w + (live[i] ? ((size_t)tile * nsteps + c[i] * 16) * 64 : 0) + lane;
    if (live[i]) {
#pragma unroll
      for (int s = 0; s < 16; ++s) wv[i][s] = __builtin_nontemporal_load(wb + (size_t)min(s, cs[i] - 1) * 64);
    }
  }
  if constexpr (PHASE == MID_UP) {
    // the down projection's weights into the L2 of the XCD whose blocks will read them, while this block waits (ixt_step.h)
    if (blk < a.early)
      mid_touch(a, MID_DOWN, L.wout, a.F, E >> 4, (int)blockIdx.x - blk + a.nblk[MID_UP], a.nblk[MID_DOWN] / MID_SPLIT, (blk >> 3) * MID_NW + wave, (a.early >> 3) * MID_NW, spare);
  }
  if constexpr (PHASE == MID_QKV) {
    if (!g.rope32)
      for (int i = tid; i < 2 * tpb * 16 * G; i += MID_NW * 64) {
        const int r = i % (16 * G), t = i / (16 * G) % tpb, th = (blk * tpb + t) % (g.hd >> 4);
        s_rope[(i / (16 * G * tpb) * 8 + t) * 16 * G + r] = *reinterpret_cast<const u32x4*>((i < 16 * G * tpb ? a.rope_sin : a.rope_cos) + (size_t)a.row_pos[min(r, R - 1)] * (g.hd >> 1) + 8 * th);
      }
    if (tid < 16 * G) {
      const int r = min(tid, R - 1), pos = a.row_pos[r];
      s_pos[tid] = pos;
      s_page[tid] = tid < R && a.row_active[r] != 0 ? a.page_map[(size_t)a.row_slot[r] * g.mpg + pos / g.P] : -1;
    }
  }
  mid_wait(a, PHASE);

  // the residuals of what this wave will store
  const int tiles = PHASE == MID_UP ? tpb / 2 : tpb, njobs = tiles * G;
  const bf16_t* hres = (PHASE == MID_O ? a.hin : a.hmid) + (size_t)g0 * 16 * E;
  uint2 hv[4];
  if constexpr (PHASE == MID_O || PHASE == MID_DOWN) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int j = wave + MID_NW * k, r = (j / tiles) * 16 + row, tile = blk * tpb + j % tiles;
      hv[k] = uint2{0, 0};
      if (j < njobs && r < R && tile < ntile) hv[k] = *reinterpret_cast<const uint2*>(hres + (size_t)r * E + tile * 16 + cq * 4);
    }
  }

  f32x4 acc[2][G];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int b = 0; b < G; ++b) acc[i][b] = f32x4(0.0f);
  if (tpb > 1 && nsteps <= MID_BUF_STEPS) {
    // a group's rows through LDS, the next group's under its products
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane((uint32_t)(uintptr_t)((__attribute__((address_space(3))) u32x4*)sx));
    auto stage = [&](int b) {
#pragma unroll
      for (int i = 0; i < MID_BUF_STEPS / MID_NW; ++i) {
        const int f = min(wave + MID_NW * i, nsteps - 1);    // (past the end: the last one again)
        lds_dma16(lds0 + (uint32_t)((b & 1) * nsteps + f) * 1024u, x + (size_t)b * nsteps * 64, (uint32_t)(f * 1024 + lane * 16));
      }
    };
    stage(0);
    u32x4 ahead[G > 2 ? G - 2 : 1];                          // the groups behind them into this XCD's L2, a fragment a wave
#pragma unroll
    for (int b = 2; b < G; ++b) ahead[b - 2] = x[((size_t)b * nsteps + ((blk >> 3) * MID_NW + wave) % nsteps) * 64 + lane];
    if constexpr (G > 1) stage(1);
#pragma unroll
    for (int b = 0; b < G; ++b) {
      if (b + 1 < G) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(MID_BUF_STEPS / MID_NW) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();
      auto products = [&](int s) {
        const bf16x8 xv = __builtin_bit_cast(bf16x8, sx[((b & 1) * nsteps + c[0] * 16 + s) * 64 + lane]);
#pragma unroll
        for (int i = 0; i < 2; ++i) acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[i][s]), xv, acc[i][b], 0, 0, 0);
      };
      if (live[0]) {
        if (cs[0] == 16) {
#pragma unroll
          for (int s = 0; s < 16; ++s) {
            products(s);
            if ((s & 7) == 7) __builtin_amdgcn_sched_barrier(0);
          }
        } else {
#pragma unroll
          for (int s = 0; s < 16; ++s)
            if (s < cs[0]) products(s);
        }
      }
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      lds_barrier();                                         // everyone has read this group
      if (b + 2 < G) stage(b + 2);
    }
#pragma unroll
    for (int b = 2; b < G; ++b) asm volatile("" ::"v"(ahead[b - 2].x), "v"(ahead[b - 2].y), "v"(ahead[b - 2].z), "v"(ahead[b - 2].w));
  } else {
    // eight fragments ahead of the eight in use
    u32x4 xv[2][8];
    auto fetch = [&](int n) {                                // n = (unit, group, half)
      const int i = n / (2 * G), b = n / 2 % G, h = n & 1;
      const u32x4* xb = x + ((size_t)b * nsteps + (live[i] ? c[i] * 16 : 0)) * 64 + lane;
#pragma unroll
      for (int s = 0; s < 8; ++s) xv[n & 1][s] = xb[(size_t)min(8 * h + s, cs[i] - 1) * 64];
    };
    fetch(0);
#pragma unroll
    for (int n = 0; n < 4 * G; ++n) {
      if (n + 1 < 4 * G) fetch(n + 1);
      __builtin_amdgcn_sched_barrier(0);
      const int i = n / (2 * G), b = n / 2 % G, h = n & 1;
#pragma unroll
      for (int s = 0; s < 8; ++s)
        if (live[i] && 8 * h + s < cs[i]) acc[i][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[i][8 * h + s]), __builtin_bit_cast(bf16x8, xv[n & 1][s]), acc[i][b], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // ---- chain totals meet in LDS; a wave adds those of a (tile, group), in order
  f32x4* red = reinterpret_cast<f32x4*>(sx);                 // [unit][group][lane]
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int b = 0; b < G; ++b)
      if (live[i]) red[((wave * 2 + i) * G + b) * 64 + lane] = acc[i][b];
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int j = wave + MID_NW * k, b = j / tiles, t = PHASE == MID_UP ? j % tiles * 2 : j % tiles, tile = blk * tpb + t, r = b * 16 + row;
    if (j >= njobs || tile >= ntile) continue;
    f32x4 tot = f32x4(0.0f), tot2 = f32x4(0.0f);
    auto total = [&](auto most) {                            // `most` chains at most, all reads ahead of the adds
      constexpr int MC = decltype(most)::value;
      f32x4 v4[MC], w4[MC];
#pragma unroll
      for (int cc = 0; cc < MC; ++cc) {
        v4[cc] = red[((min(cc, nc - 1) * tpb + t) * G + b) * 64 + lane];
        if (PHASE == MID_UP) w4[cc] = red[((min(cc, nc - 1) * tpb + t + 1) * G + b) * 64 + lane];
      }
#pragma unroll
      for (int cc = 0; cc < MC; ++cc) {
        if (cc < nc) { tot = tot + v4[cc]; if (PHASE == MID_UP) tot2 = tot2 + w4[cc]; }
      }
    };
    if (PHASE == MID_UP || PHASE == MID_QKV || nc <= 4) total(std::integral_constant<int, 4>());
    else total(std::integral_constant<int, 16>());
    if constexpr (PHASE == MID_O || PHASE == MID_DOWN) {
      if (r < R)
        step_st8((PHASE == MID_O ? a.hmid : a.hout) + (size_t)(g0 * 16 + r) * E + tile * 16 + cq * 4, pack2(f2bf(bflo(hv[k].x) + rbf(tot[0])), f2bf(bfhi(hv[k].x) + rbf(tot[1]))),
                 pack2(f2bf(bflo(hv[k].y) + rbf(tot[2])), f2bf(bfhi(hv[k].y) + rbf(tot[3]))));
    } else if constexpr (PHASE == MID_UP) {
      if (r < R) {
        bf16_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = ixt_swiglu(rbf(tot[e]), rbf(tot2[e]));
        step_st8(a.act + xidx(r, (tile >> 1) * 16 + cq * 4, a.F), pack2(o[0], o[1]), pack2(o[2], o[3]));
      }
    } else {
      // bf16(t), RoPE by partner exchange across lanes l and l ^ 32, q -> its buffer, K / V -> the row's page (k_gemm_ring's epilogue)
      const int half = g.hd >> 1, th = tile % (g.hd >> 4), QN = g.nq * g.hd, KN = g.nkv * g.hd, hh = tile * 16 / g.hd;
      const int pos = s_pos[r], page = s_page[r], tok = pos % g.P;
      const bool is_v = tile * 16 >= QN + KN;
      float v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = rbf(tot[e]);
      if (!is_v) {
        const int fi = 8 * th + 4 * (cq & 1);
        if (g.rope32) {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float other = __shfl_xor(v[e], 32, 64);
            float o1, o2;
            ixt_rope_pair(1, a.rope_sin, a.rope_cos, (size_t)pos * half + fi + e, cq < 2 ? v[e] : other, cq < 2 ? other : v[e], o1, o2);
            v[e] = cq < 2 ? o1 : o2;
          }
        } else {
          const u32x4 s8 = s_rope[t * 16 * G + r], c8 = s_rope[(8 + t) * 16 * G + r];
          const uint2 sv = (cq & 1) ? uint2{s8.z, s8.w} : uint2{s8.x, s8.y}, cv = (cq & 1) ? uint2{c8.z, c8.w} : uint2{c8.x, c8.y};
          const float sn[4] = {bflo(sv.x), bfhi(sv.x), bflo(sv.y), bfhi(sv.y)}, cn[4] = {bflo(cv.x), bfhi(cv.x), bflo(cv.y), bfhi(cv.y)};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float other = __shfl_xor(v[e], 32, 64);
            v[e] = cq < 2 ? rbf(rbf(v[e] * cn[e]) - rbf(other * sn[e])) : rbf(rbf(v[e] * cn[e]) + rbf(other * sn[e]));
          }
        }
      }
      if (r < R) {
        bf16_t *kpages = mid_at<bf16_t>(a, L.kpages), *vpages = mid_at<bf16_t>(a, L.vpages);
        const uint2 ov = {pack2(f2bf(v[0]), f2bf(v[1])), pack2(f2bf(v[2]), f2bf(v[3]))};
        const int feat = is_v ? th * 16 + cq * 4 : (cq >= 2 ? half : 0) + 8 * th + 4 * (cq & 1);
        if (g.rope32 && !is_v) {   // llama3.1: the lane's four de-interleaved features are every second feature of the model's order (ixt_qk_feat)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int fn_ = ixt_qk_feat(1, feat + e, half);
            if (hh < g.nq) a.qbuf[((size_t)r * g.nq + hh) * g.hd + fn_] = f2bf(v[e]);
            else if (page >= 0) kpages[kpage_off(g, page, hh - g.nq, fn_ >> 3, tok) + (fn_ & 7)] = f2bf(v[e]);
          }
        } else if (hh < g.nq) {
          *reinterpret_cast<uint2*>(a.qbuf + ((size_t)r * g.nq + hh) * g.hd + feat) = ov;
        } else if (page >= 0) {
          if (!is_v) *reinterpret_cast<uint2*>(kpages + kpage_off(g, page, hh - g.nq, feat >> 3, tok) + (feat & 7)) = ov;
          else *reinterpret_cast<uint2*>(vpages + vpage_off(g, page, hh - g.nq - g.nkv, tok) + feat) = ov;
        }
      }
    }
  }
  if (PHASE == MID_UP) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");      // nothing may land in LDS that the next block owns
  // (behind QKV nobody waits: the launch ends)
  const int storing = min(MID_NW, njobs);                    // (of a last block with fewer tiles some arrive with nothing stored)
  if (PHASE != MID_QKV && wave < storing) step_arrive(mid_cnt(a, PHASE), blk_all, storing, &met);
}

// the norm of eight rows, a wave a row (k_step's order of operations), as the operand of the projections behind it
template <int PHASE>
__device__ __forceinline__ void mid_norm(const MidArgs& a, int blk, u32x4* sx) {
  __shared__ int met;
  if (threadIdx.x == 0) met = 0;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), r = blk * MID_NW + wave, nch = a.E >> 3;
  const bf16_t* scale = PHASE == MID_N1 ? a.scale : mid_at<const bf16_t>(a, a.layers[a.layer].ln2);
  u32x4 sc[4], h[4];
#pragma unroll
  for (int b = 0; b < 4; ++b) sc[b] = *reinterpret_cast<const u32x4*>(scale + min(b * 64 + lane, nch - 1) * 8);
  mid_wait(a, PHASE);
  if (r < a.R) {
    const bf16_t* src = (PHASE == MID_N1 ? a.hout : a.hmid) + (size_t)r * a.E;
#pragma unroll
    for (int b = 0; b < 4; ++b) h[b] = *reinterpret_cast<const u32x4*>(src + min(b * 64 + lane, nch - 1) * 8);
    float total = 0.0f;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float f[8] = {bflo(h[b].x), bfhi(h[b].x), bflo(h[b].y), bfhi(h[b].y), bflo(h[b].z), bfhi(h[b].z), bflo(h[b].w), bfhi(h[b].w)};
      float v = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) v = __builtin_fmaf(f[j], f[j], v);
      v = b * 64 + lane < nch ? v : 0.0f;
      v = xor_sum(v);
      total = b * 64 < nch ? total + v : total;
    }
    const float rs = 1.0f / sqrtf(total / (float)a.E + a.eps);
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const int ch = b * 64 + lane;
      const float f[8] = {bflo(h[b].x), bfhi(h[b].x), bflo(h[b].y), bfhi(h[b].y), bflo(h[b].z), bfhi(h[b].z), bflo(h[b].w), bfhi(h[b].w)};
      const float s[8] = {bflo(sc[b].x), bfhi(sc[b].x), bflo(sc[b].y), bfhi(sc[b].y), bflo(sc[b].z), bfhi(sc[b].z), bflo(sc[b].w), bfhi(sc[b].w)};
      bf16_t o[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = f2bf(rbf(f[j] * rs) * s[j]);
      if (ch < nch) sx[ch * MID_NW + (wave ^ (ch & (MID_NW - 1)))] = u32x4{pack2(o[0], o[1]), pack2(o[2], o[3]), pack2(o[4], o[5]), pack2(o[6], o[7])};
    }
  }
  __syncthreads();
  // the eight rows of a piece of eight features are one line of the operand: written whole (row by row, 16 bytes of a line each, the phase took 9 us, now 4)
  bf16_t* dst = PHASE == MID_N1 ? a.xn1 : a.xn2;
  for (int i = threadIdx.x; i < nch * MID_NW; i += MID_NW * 64) {
    const int ch = i / MID_NW, rr = i % MID_NW;
    if (blk * MID_NW + rr < a.R) stg16_agent(dst + xidx(blk * MID_NW + rr, ch * 8, a.E), sx[ch * MID_NW + (rr ^ (ch & (MID_NW - 1)))]);
  }
  step_arrive(mid_cnt(a, PHASE), blk, MID_NW, &met);
}

// Aligned: 80 to 104 KB of code that every launch reads anew (the weights leave nothing of it in the caches), and where it lies shows.  The same machine code, 45 rows of the 1B model, ms for 32
// steps: at a multiple of 64 KiB 38.5, 256 bytes behind one 38.7, 2 KiB 39.0, 4 KiB to 48 KiB 38.6 to 38.75; wherever the kernels compiled in front of it left it 38.4 to 38.9.
template <int G>
__attribute__((aligned(65536))) __global__ __launch_bounds__(MID_NW * 64, 2) void k_mid(MidArgs a) {
  extern __shared__ __attribute__((aligned(16))) u32x4 mid_lds[];
  int b = blockIdx.x;
  if (b < a.nblk[MID_O]) { mid_dot<MID_O, G>(a, b, mid_lds); return; }
  b -= a.nblk[MID_O];
  if (b < a.nblk[MID_N2]) { mid_norm<MID_N2>(a, b, mid_lds); return; }
  b -= a.nblk[MID_N2];
  if (b < a.nblk[MID_UP]) { mid_dot<MID_UP, G>(a, b, mid_lds); return; }
  b -= a.nblk[MID_UP];
  if (b < a.nblk[MID_DOWN]) { mid_dot<MID_DOWN, G>(a, b, mid_lds); return; }
  b -= a.nblk[MID_DOWN];
  if (b < a.nblk[MID_N1]) { mid_norm<MID_N1>(a, b, mid_lds); return; }
  mid_dot<MID_QKV, G>(a, b - a.nblk[MID_N1], mid_lds);
}
