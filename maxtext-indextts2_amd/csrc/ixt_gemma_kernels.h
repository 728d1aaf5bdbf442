// ixt_gemma_kernels.h -- row kernels of the Gemma-2 block (layers/gemma2.py:69-236, decoders.py:552-565).
// The projections, RoPE, page writes and the attention kernels are the ones of the llama2 block (ixt_kernels.h); what differs is what
// happens between them: the projection output is normalised before the residual add, the gate is GELU(tanh), and the logits are
// divided by sqrt(emb) and soft-capped.  Same canonical orders as ixt_kernels.h (slices from 0; sum of squares: a lane's 8 features by
// fma, xor tree over the wave, blocks of 512 features in order).
#pragma once
#include "ixt_kernels.h"

// =====================================================================================================
// o = bf16(sum of slices)                                 the O- or down-projection of row r
// o = bf16(bf16(o * rsqrt(mean(o^2) + eps)) * post)       when post != nullptr   (gemma2.py:107-116, :135-143)
// h = bf16(h_in + o) -> h_out                             (gemma2.py:118, :146)
// xn = bf16(bf16(h * rsqrt(mean(h^2) + eps)) * next)      when next != nullptr (the following pre-norm), dot kernel's x layout
// A thread keeps its chunks of 8 features (tid + 256 it, E <= 2048 ITS) in registers from the sums to the last norm, and everything it reads is in flight
// before the first of the two sums over the row (one read behind the other: 7.8 us a launch of 256 rows of 2304 -> 6.4; now 5.1).   grid = R, block 256.
// =====================================================================================================
struct GNormArgs {
  const float* part; int slices; size_t slice_stride;
  const bf16_t* h_in; bf16_t* h_out;
  const bf16_t* post; const bf16_t* next;
  bf16_t* xn_out;
  int E; float eps;
};

template <int ITS>
static __global__ __launch_bounds__(256) void k_gnorm(GNormArgs a) {
  __shared__ float blk[2][4 * ITS];                        // block sums of o^2, of h^2
  const int r = row_of_block(blockIdx.x, gridDim.x), tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int E = a.E, nch = E / 8, nblk = (nch + 63) / 64;
  float o[ITS][8];
  u32x4 hin[ITS], post[ITS], next[ITS];
#pragma unroll
  for (int it = 0; it < ITS; ++it) {
    const int ch = it * 256 + tid;
    hin[it] = post[it] = next[it] = u32x4(0u);
#pragma unroll
    for (int j = 0; j < 8; ++j) o[it][j] = 0.0f;
    if (ch < nch) {
      hin[it] = *reinterpret_cast<const u32x4*>(a.h_in + (size_t)r * E + ch * 8);
      if (a.post != nullptr) post[it] = *reinterpret_cast<const u32x4*>(a.post + ch * 8);
      if (a.next != nullptr) next[it] = *reinterpret_cast<const u32x4*>(a.next + ch * 8);
    }
  }
  for (int s = 0; s < a.slices; s += 2) {                  // two slices in flight
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      const int ch = it * 256 + tid;
      if (ch < nch) {
        const float *p = a.part + (size_t)s * a.slice_stride + (size_t)r * E + ch * 8, *q = p + (s + 1 < a.slices ? a.slice_stride : 0);
        const float4 p0 = *reinterpret_cast<const float4*>(p), p1 = *reinterpret_cast<const float4*>(p + 4), q0 = *reinterpret_cast<const float4*>(q), q1 = *reinterpret_cast<const float4*>(q + 4);
        o[it][0] = o[it][0] + p0.x; o[it][1] = o[it][1] + p0.y; o[it][2] = o[it][2] + p0.z; o[it][3] = o[it][3] + p0.w;
        o[it][4] = o[it][4] + p1.x; o[it][5] = o[it][5] + p1.y; o[it][6] = o[it][6] + p1.z; o[it][7] = o[it][7] + p1.w;
        if (s + 1 < a.slices) {
          o[it][0] = o[it][0] + q0.x; o[it][1] = o[it][1] + q0.y; o[it][2] = o[it][2] + q0.z; o[it][3] = o[it][3] + q0.w;
          o[it][4] = o[it][4] + q1.x; o[it][5] = o[it][5] + q1.y; o[it][6] = o[it][6] + q1.z; o[it][7] = o[it][7] + q1.w;
        }
      }
    }
  }
  // the sum of squares of a row: 64 chunks of 8 features at a time (a wave's), in order
  auto square_sum = [&](float* sums) {
#pragma unroll
    for (int it = 0; it < ITS; ++it) {
      float v = 0.0f;
#pragma unroll
      for (int j = 0; j < 8; ++j) v = __builtin_fmaf(o[it][j], o[it][j], v);
      v = xor_sum(v);
      if (lane == 0) sums[it * 4 + wave] = v;
    }
    __syncthreads();
    float total = 0.0f;
    for (int b = 0; b < nblk; ++b) total = total + sums[b];
    return 1.0f / sqrtf(total / (float)E + a.eps);
  };
#pragma unroll
  for (int it = 0; it < ITS; ++it)
#pragma unroll
    for (int j = 0; j < 8; ++j) o[it][j] = rbf(o[it][j]);
  const float rs1 = a.post != nullptr ? square_sum(blk[0]) : 0.0f;
#pragma unroll
  for (int it = 0; it < ITS; ++it) {
    const float hf[8] = {bflo(hin[it].x), bfhi(hin[it].x), bflo(hin[it].y), bfhi(hin[it].y), bflo(hin[it].z), bfhi(hin[it].z), bflo(hin[it].w), bfhi(hin[it].w)};
    const float sc[8] = {bflo(post[it].x), bfhi(post[it].x), bflo(post[it].y), bfhi(post[it].y), bflo(post[it].z), bfhi(post[it].z), bflo(post[it].w), bfhi(post[it].w)};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      float v = o[it][j];
      if (a.post != nullptr) v = rbf(rbf(v * rs1) * sc[j]);
      o[it][j] = rbf(hf[j] + v);
    }
    const int ch = it * 256 + tid;
    if (ch < nch) {
      u32x4 ov;
      ov.x = pack2(f2bf(o[it][0]), f2bf(o[it][1])); ov.y = pack2(f2bf(o[it][2]), f2bf(o[it][3]));
      ov.z = pack2(f2bf(o[it][4]), f2bf(o[it][5])); ov.w = pack2(f2bf(o[it][6]), f2bf(o[it][7]));
      *reinterpret_cast<u32x4*>(a.h_out + (size_t)r * E + ch * 8) = ov;
    }
  }
  if (a.next == nullptr) return;                           // whole grid
  const float rs = square_sum(blk[1]);
#pragma unroll
  for (int it = 0; it < ITS; ++it) {
    const int ch = it * 256 + tid;
    if (ch < nch) {
      const float sc[8] = {bflo(next[it].x), bfhi(next[it].x), bflo(next[it].y), bfhi(next[it].y), bflo(next[it].z), bfhi(next[it].z), bflo(next[it].w), bfhi(next[it].w)};
      bf16_t y[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = f2bf(rbf(o[it][j] * rs) * sc[j]);
      u32x4 ov;
      ov.x = pack2(y[0], y[1]); ov.y = pack2(y[2], y[3]); ov.z = pack2(y[4], y[5]); ov.w = pack2(y[6], y[7]);
      *reinterpret_cast<u32x4*>(a.xn_out + xidx(r, ch * 8, E)) = ov;
    }
  }
}

// =====================================================================================================
// GELU(tanh) gate from partial slices: k_swiglu_part with ixt_geglu (linears.py:449-464 with mlp_activations ["gelu", "linear"]).
// =====================================================================================================
static __global__ __launch_bounds__(256) void k_geglu_part(const float* part, int slices, size_t slice_stride, int F, bf16_t* out /*[R][F] in xidx layout*/) {
  const int f0 = (blockIdx.x * 256 + threadIdx.x) * 8, r = blockIdx.y;
  if (f0 >= F) return;
  const float* p = part + (size_t)r * 2 * F;
  float a[8], b[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) { a[j] = 0.0f; b[j] = 0.0f; }
  for (int s = 0; s < slices; ++s) {
    const float* ps = p + (size_t)s * slice_stride;
    const int ca = (f0 >> 4) * 32 + (f0 & 15);   // wi_0 tile j = column tile 2 j, wi_1 tile j = column tile 2 j + 1 (k_tile_w mode 2)
    const float4 a0 = *reinterpret_cast<const float4*>(ps + ca), a1 = *reinterpret_cast<const float4*>(ps + ca + 4);
    const float4 b0 = *reinterpret_cast<const float4*>(ps + ca + 16), b1 = *reinterpret_cast<const float4*>(ps + ca + 20);
    a[0] = a[0] + a0.x; a[1] = a[1] + a0.y; a[2] = a[2] + a0.z; a[3] = a[3] + a0.w;
    a[4] = a[4] + a1.x; a[5] = a[5] + a1.y; a[6] = a[6] + a1.z; a[7] = a[7] + a1.w;
    b[0] = b[0] + b0.x; b[1] = b[1] + b0.y; b[2] = b[2] + b0.z; b[3] = b[3] + b0.w;
    b[4] = b[4] + b1.x; b[5] = b[5] + b1.y; b[6] = b[6] + b1.z; b[7] = b[7] + b1.w;
  }
  bf16_t o[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) o[j] = ixt_geglu(rbf(a[j]), rbf(b[j]));
  u32x4 ov;
  ov.x = pack2(o[0], o[1]); ov.y = pack2(o[2], o[3]); ov.z = pack2(o[4], o[5]); ov.w = pack2(o[6], o[7]);
  *reinterpret_cast<u32x4*>(out + xidx(r, f0, F)) = ov;
}

static __global__ __launch_bounds__(256) void k_geglu(const bf16_t* a, const bf16_t* b, bf16_t* out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < n) out[i] = ixt_geglu(bf2f(a[i]), bf2f(b[i]));
}

// =====================================================================================================
// Logits of the tied head (decoders.py:552-565), in place on bf16-valued f32 rows, then greedy sampling over the allowed columns
// (first index of the maximum; inference_utils.py:74-75).  normalize: v / sqrt(emb) in f32 (the divisor is an f32 array: the logits
// become f32) and the cap chain in f32; otherwise every primitive of the cap rounds to bf16.  grid = rows, block 256.
// =====================================================================================================
__device__ __forceinline__ float ixt_logit_post(float v, int normalize, float sqrt_emb, float cap) {
  if (normalize) {
    v = v / sqrt_emb;
    if (cap > 0.0f) v = ixt_tanh(v / cap) * cap;
    return v;
  }
  if (cap > 0.0f) v = rbf(rbf(ixt_tanh(rbf(v / cap))) * cap);
  return v;
}

// grid = (ceil(vocab / IXT_LPOST_COLS), rows), block 256: a block post-processes IXT_LPOST_COLS consecutive columns of one row and leaves its
// (maximum, first index) over the allowed columns in amax_val / amax_idx [row][block] for k_argmax_final (one block per row took 0.48 ms at
// 258 176 columns: 9 % of a Gemma-2 2B decode step).
#define IXT_LPOST_COLS 4096
static __global__ __launch_bounds__(256) void k_logits_post(float* logits, int vocab, int normalize, float sqrt_emb, float cap, ColRanges cols, float* amax_val,
                                                     int32_t* amax_idx) {
  __shared__ float bv[256];
  __shared__ int bi[256];
  const int r = blockIdx.y, tid = threadIdx.x;
  float* row = logits + (size_t)r * vocab;
  float best = -INFINITY;
  int bidx = 0x7fffffff;
  const int n_end = min(vocab, (int)(blockIdx.x + 1) * IXT_LPOST_COLS);
  for (int n = blockIdx.x * IXT_LPOST_COLS + tid; n < n_end; n += 256) {
    const float v = ixt_logit_post(row[n], normalize, sqrt_emb, cap);
    row[n] = v;
    bool ok = cols.n == 0;
    for (int i = 0; i < cols.n; ++i) ok = ok || (n >= cols.lo[i] && n < cols.hi[i]);
    if (ok && (bidx == 0x7fffffff || v > best)) { best = v; bidx = n; }   // n ascends within a thread: the first maximum is kept
  }
  bv[tid] = best; bi[tid] = bidx;
  __syncthreads();
  for (int s2 = 128; s2 > 0; s2 >>= 1) {
    if (tid < s2) {
      const float v = bv[tid + s2]; const int i2 = bi[tid + s2];
      if (i2 != 0x7fffffff && (bi[tid] == 0x7fffffff || v > bv[tid] || (v == bv[tid] && i2 < bi[tid]))) { bv[tid] = v; bi[tid] = i2; }
    }
    __syncthreads();
  }
  if (tid == 0) {
    amax_val[(size_t)r * gridDim.x + blockIdx.x] = bi[0] == 0x7fffffff ? -INFINITY : bv[0];
    amax_idx[(size_t)r * gridDim.x + blockIdx.x] = bi[0];
  }
}

// embedding table [V][E] -> [E][V] (the logits kernel of the tied head before it is re-tiled).  grid = (ceil(V/32), ceil(E/32)), block (32, 8).
static __global__ void k_transpose_ve(const bf16_t* __restrict__ src, bf16_t* __restrict__ dst, int V, int E) {
  __shared__ bf16_t tile[32][33];
  const int v0 = blockIdx.x * 32, e0 = blockIdx.y * 32;
  for (int i = threadIdx.y; i < 32; i += 8) {
    const int v = v0 + i, e = e0 + threadIdx.x;
    tile[i][threadIdx.x] = (v < V && e < E) ? src[(size_t)v * E + e] : (bf16_t)0;
  }
  __syncthreads();
  for (int i = threadIdx.y; i < 32; i += 8) {
    const int e = e0 + i, v = v0 + threadIdx.x;
    if (e < E && v < V) dst[(size_t)e * V + v] = tile[threadIdx.x][i];
  }
}
