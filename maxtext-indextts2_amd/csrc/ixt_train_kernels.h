// ixt_train_kernels.h -- gfx950 kernels of the training step (MaxText/train.py:255-472): forward + backward of the
// llama2 block stack, cross entropy with its custom VJP (max_utils.py:563-654), global-norm clip (maxtext_utils.py:825-846) and AdamW
// (optimizers.py:28-38).  Precision: bf16 activations and matmul operands, f32 accumulation (v_mfma_f32_16x16x32_bf16), f32 master
// weights / gradients / optimizer state -- the reference's dtype=bfloat16, weight_dtype=float32 (base.yml:86, :130).
// The tolerance of this path is 1e-4 relative on the loss against the f32 PyTorch restatement the tests hold (tests/test_gpu_train.py); it is NOT the
// bit-exact contract of the decode path, so reductions here use whatever order is fastest unless stated.
#pragma once
#include "ixt_device.h"
#include "ixt_train_gemm.h"

// ---------------------------------------------------------------------------------------------------------------- elementwise / rows
// Rows of bf16 are moved 16 bytes a lane; where a sum has a place in the arithmetic, its terms stay with the threads they always had (thread t: t, t +
// 256, ..), so that the losses and gradients of a step do not depend on how the rows are read.
__device__ __forceinline__ void t_unpack8(const u32x4& w, float (&v)[8]) {
#pragma unroll
  for (int k = 0; k < 4; ++k) { v[2 * k] = bflo(w[k]); v[2 * k + 1] = bfhi(w[k]); }
}
__device__ __forceinline__ u32x4 t_pack8(const float (&v)[8]) {
  u32x4 w;
#pragma unroll
  for (int k = 0; k < 4; ++k) w[k] = pack2(f2bf(v[2 * k]), f2bf(v[2 * k + 1]));
  return w;
}
// zeros: n values at `at`, then `count` times two runs of `run` values at a and b, `stride` apart (n, run, offsets multiples of 4).
// grid = (ceil(n / 1024) + ceil(2 count run / 1024)), block 256.
static __global__ void k_t_zero(float* __restrict__ at, long n, float* __restrict__ a, float* __restrict__ b, long stride, int count, int run) {
  const float4 z = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  const long nb = (n + 1023) / 1024;
  if ((long)blockIdx.x < nb) {
    const long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4;
    if (i < n) *reinterpret_cast<float4*>(at + i) = z;
    return;
  }
  const long i = (((long)blockIdx.x - nb) * 256 + threadIdx.x) * 4, l = i / (2 * run), e = i - l * 2 * run;
  if (l < count) *reinterpret_cast<float4*>((e < run ? a + e : b + e - run) + l * stride) = z;
}
// rows of n (a multiple of 4), ld apart in dst.  grid.y = rows
static __global__ void k_t_cast_bf16(const float* __restrict__ src, bf16_t* __restrict__ dst, long n, long ld) {
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  const float4 v = *reinterpret_cast<const float4*>(src + blockIdx.y * n + i);
  *reinterpret_cast<uint2*>(dst + blockIdx.y * ld + i) = make_uint2(pack2(f2bf(v.x), f2bf(v.y)), pack2(f2bf(v.z), f2bf(v.w)));
}

// the sum over the lanes, with those 32, 16, .. 1 away in turn (from 8 on any lane of the other group will do: the lanes of a group hold the same value)
__device__ __forceinline__ float t_wave_sum(float v) {
  auto ror = [](float x, auto ctrl) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true)); };
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(a[0]) + __uint_as_float(a[1]);
  const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(b[0]) + __uint_as_float(b[1]);
  v += ror(v, std::integral_constant<int, 0x128>());
  v += ror(v, std::integral_constant<int, 0x124>());
  v += ror(v, std::integral_constant<int, 0x122>());
  v += ror(v, std::integral_constant<int, 0x121>());
  return v;
}
__device__ __forceinline__ float t_block_sum(float v, float* red) {   // 256 threads
  v = t_wave_sum(v);
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  return red[0] + red[1] + red[2] + red[3];
}

// RMSNorm forward (normalizations.py:57-70): y = bf16(bf16(x r) scale), r = rsqrt(mean(x^2) + eps) saved per row.  E % 8 == 0, E <= 4096.  grid = T, block 256.
static __global__ __launch_bounds__(256) void k_t_rmsnorm_fwd(const bf16_t* __restrict__ x, const bf16_t* __restrict__ scale, bf16_t* __restrict__ y,
                                                       float* __restrict__ rstd, int E, float eps) {
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) bf16_t xs[4096];
  const long row = blockIdx.x;
  const int tid = threadIdx.x;
  u32x4 w[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int e = (tid + i * 256) * 8;
    if (e < E) { w[i] = *reinterpret_cast<const u32x4*>(x + row * E + e); *reinterpret_cast<u32x4*>(xs + e) = w[i]; }
  }
  __syncthreads();
  float s = 0.0f;
  for (int e = tid; e < E; e += 256) { const float v = bf2f(xs[e]); s += v * v; }
  const float tot = t_block_sum(s, red);
  const float r = 1.0f / sqrtf(tot / (float)E + eps);
  if (tid == 0) rstd[row] = r;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int e = (tid + i * 256) * 8;
    if (e < E) {
      float v[8], c[8];
      t_unpack8(w[i], v);
      t_unpack8(*reinterpret_cast<const u32x4*>(scale + e), c);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = rbf(v[k] * r) * c[k];
      *reinterpret_cast<u32x4*>(y + row * E + e) = t_pack8(v);
    }
  }
}
// backward: dy f32 [T][E] (the sum of the consumers' input gradients); dx (f32) is ADDED to dh (the residual-stream gradient), and the sum goes out as
// bf16, too (dh_bf, the next products' operand; nullptr: nobody wants it).
// dscale: a block walks `rpb` rows and keeps its features' partial sums in registers -- written out for k_t_scale_grads (part), or one f32 atomic per
// feature and BLOCK (short rows: the atomics were 10 of 23 us at 2048 x 768; 13 of 145 at 16384 x 2048) (one per feature and row
// took 466 us per launch at 16384 x 2048: 2048 addresses under 33 M atomics).  A row's operands stay in registers between the two passes over it and
// the next row's are in flight meanwhile.  grid = ceil(T / rpb), block 256, E <= 256 FPT.
#define TN_FPT 16
template <int FPT>
static __global__ __launch_bounds__(256) void k_t_rmsnorm_bwd(const float* __restrict__ dy, const bf16_t* __restrict__ x, const bf16_t* __restrict__ scale,
                                                       const float* __restrict__ rstd, float* __restrict__ dh, bf16_t* __restrict__ dh_bf, float* __restrict__ dscale, float* __restrict__ part,
                                                       int E, long T, int rpb) {
  __shared__ float red[4];
  float ds[FPT], sc[FPT], gy[FPT], xv[FPT], hv[FPT];
#pragma unroll
  for (int i = 0; i < FPT; ++i) {
    const int e = threadIdx.x + i * 256;
    ds[i] = 0.0f;
    sc[i] = e < E ? bf2f(scale[e]) : 0.0f;
  }
  const long row0 = (long)blockIdx.x * rpb, row1 = row0 + rpb < T ? row0 + rpb : T;
  auto fetch = [&](long row) {
#pragma unroll
    for (int i = 0; i < FPT; ++i) {
      const int e = threadIdx.x + i * 256;
      if (e < E) { gy[i] = dy[row * E + e]; xv[i] = bf2f(x[row * E + e]); hv[i] = dh[row * E + e]; }
    }
  };
  fetch(row0);
  for (long row = row0; row < row1; ++row) {
    const float r = rstd[row];
    float s = 0.0f, g0[FPT], xh[FPT], h0[FPT];
#pragma unroll
    for (int i = 0; i < FPT; ++i) { g0[i] = gy[i]; xh[i] = xv[i] * r; h0[i] = hv[i]; }
    if (row + 1 < row1) fetch(row + 1);
#pragma unroll
    for (int i = 0; i < FPT; ++i)
      if (threadIdx.x + i * 256 < E) s += g0[i] * sc[i] * xh[i];
    const float mean = t_block_sum(s, red) / (float)E;
#pragma unroll
    for (int i = 0; i < FPT; ++i) {
      const int e = threadIdx.x + i * 256;
      if (e < E) {
        const float h = h0[i] + r * (g0[i] * sc[i] - xh[i] * mean);
        dh[row * E + e] = h;
        if (dh_bf != nullptr) dh_bf[row * E + e] = f2bf(h);
        ds[i] += g0[i] * xh[i];
      }
    }
  }
#pragma unroll
  for (int i = 0; i < FPT; ++i) {
    const int e = threadIdx.x + i * 256;
    if (e < E) {
      if (part != nullptr) part[(long)blockIdx.x * E + e] = ds[i];
      else atomicAdd(dscale + e, ds[i]);
    }
  }
}
// the scale gradients of all norms from their blocks' parts [norms][n][E]: norm y is first (y < L), second (y < 2 L) or final; offsets into the gradients.
// grid = (ceil(E / 64), 2 L + 1), block 1024 = 64 features x 16 runs of parts
static __global__ __launch_bounds__(1024) void k_t_scale_grads(const float* __restrict__ part, int n, int E, float* __restrict__ g, int L, long o1, long o2, long layer, long o_final) {
  __shared__ float run[16][64];
  const int f = threadIdx.x & 63, r = threadIdx.x >> 6, e = blockIdx.x * 64 + f, y = blockIdx.y;
  const float* p = part + ((long)y * n + (long)n * r / 16) * E + e;
  const int m = (long)n * (r + 1) / 16 - (long)n * r / 16;
  float s = 0.0f;
  if (e < E)
    for (int i = 0; i < m; i += 8) {
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = i + k < m ? p[(long)(i + k) * E] : 0.0f;
#pragma unroll
      for (int k = 0; k < 8; ++k) s += v[k];
    }
  run[r][f] = s;
  __syncthreads();
  if (r == 0 && e < E) {
    for (int k = 1; k < 16; ++k) s += run[k][f];
    g[(y < L ? o1 + y * layer : y < 2 * L ? o2 + (y - L) * layer : o_final) + e] = s;
  }
}
// out[i] = parts[0][i] + parts[1][i] + ... (split-K partial products, in order)
static __global__ void k_t_sum_parts(const float* __restrict__ parts, int nparts, long n, float* __restrict__ out) {   // n a multiple of 64
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= n) return;
  float4 t = *reinterpret_cast<const float4*>(parts + i);
  for (int p = 1; p < nparts; ++p) {
    const float4 v = *reinterpret_cast<const float4*>(parts + (long)p * n + i);
    t.x += v.x; t.y += v.y; t.z += v.z; t.w += v.w;
  }
  *reinterpret_cast<float4*>(out + i) = t;
}

// Where the walks over keys (ixt_train_attn.h) have features i .. i + 3 of a head, i a multiple of 4: of every 32 the runs of four 0, 4, 1, 5, 2, 6, 3, 7, so that a lane's 16 bytes are the
// two runs that a product of k_tgemm puts on it.
__device__ __forceinline__ int ta_place4(int i) { return (i & ~31) + ((i >> 2 & 3) << 3) + (i >> 4 & 1) * 4; }
// RoPE (embeddings.py:277-315) on q bf16 [T][H][D] and k [T][KVH][D] with per-token positions; INV: the transposed rotation (backward).  A thread turns
// four pairs (D % 8 == 0).  RUNS (heads of 64 and 128): features in the order of ta_place4 on the attention's side; a head's threads are lanes of one wave, whose loads stand in front of its
// stores.  grid = ceil(T (H + KVH) (D / 8) / 256), block 256.
template <bool INV, bool RUNS>
__global__ void k_t_rope(bf16_t* __restrict__ q, bf16_t* __restrict__ k, const int32_t* __restrict__ pos, const bf16_t* __restrict__ sn, const bf16_t* __restrict__ cs, int H, int KVH,
                         int D, long T) {
  const int quads = D / 8, half = D / 2;
  const long id = (long)blockIdx.x * 256 + threadIdx.x;
  const long t = id / ((H + KVH) * quads);
  if (t >= T) return;
  const int in = (int)(id - t * ((H + KVH) * quads)), h = in / quads, i = (in - h * quads) * 4;
  bf16_t* const head = h < H ? q + (t * H + h) * D : k + (t * KVH + h - H) * D;
  const bf16_t* const from = head + (RUNS && INV ? ta_place4(i) : i);
  bf16_t* const to = head + (RUNS && !INV ? ta_place4(i) : i);
  const long at = (long)pos[t] * half + i;
  const uint2 a = *reinterpret_cast<const uint2*>(from), b = *reinterpret_cast<const uint2*>(from + half), sw = *reinterpret_cast<const uint2*>(sn + at), cw = *reinterpret_cast<const uint2*>(cs + at);
  const float x1[4] = {bflo(a.x), bfhi(a.x), bflo(a.y), bfhi(a.y)}, x2[4] = {bflo(b.x), bfhi(b.x), bflo(b.y), bfhi(b.y)};
  const float s[4] = {bflo(sw.x), bfhi(sw.x), bflo(sw.y), bfhi(sw.y)}, c[4] = {bflo(cw.x), bfhi(cw.x), bflo(cw.y), bfhi(cw.y)};
  bf16_t u[4], v[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if (!INV) { u[j] = f2bf(rbf(x1[j] * c[j]) - rbf(x2[j] * s[j])); v[j] = f2bf(rbf(x2[j] * c[j]) + rbf(x1[j] * s[j])); }
    else { u[j] = f2bf(x1[j] * c[j] + x2[j] * s[j]); v[j] = f2bf(x2[j] * c[j] - x1[j] * s[j]); }
  }
  if constexpr (RUNS) wave_lds_sync();                     // (orders the compiler; the hardware has the wave's loads in front of its stores anyway)
  *reinterpret_cast<uint2*>(to) = make_uint2(pack2(u[0], u[1]), pack2(u[2], u[3]));
  *reinterpret_cast<uint2*>(to + half) = make_uint2(pack2(v[0], v[1]), pack2(v[2], v[3]));
}

// Attention softmax over scores f32 [BH][S][S] with the train-mode mask (attentions.py:586-618: same segment AND col <= row), P bf16 out.  Columns up to
// the end of the row's 256-column block are written (zeros past the row): the products that follow go no further.  The row stays in registers
// (S <= 256 MAXV; longer rows are read again), bf16 goes out 16 bytes a lane through LDS; thread t owns the columns t, t + 256, ..
// grid = (S, BH), block 256; one row per block.
__device__ __forceinline__ void t_store_tiles(const bf16_t* tile, bf16_t* __restrict__ out, int n, int tid) {   // n a multiple of 8
  for (int j = tid * 8; j < n; j += 2048) *reinterpret_cast<u32x4*>(out + j) = *reinterpret_cast<const u32x4*>(tile + j);
}
static __global__ __launch_bounds__(256) void k_t_softmax_fwd(const float* __restrict__ sc, const int32_t* __restrict__ seg, bf16_t* __restrict__ P, int S, int H) {
  __shared__ float red[4];
  const int row = blockIdx.x;
  const long bh = blockIdx.y, b = bh / H;
  const float* s = sc + (bh * S + row) * S;
  bf16_t* p = P + (bh * S + row) * S;
  const int myseg = seg[b * S + row], end = min(S, (row / 256 + 1) * 256);
  float m = -INFINITY;
  for (int j = threadIdx.x; j <= row; j += 256)
    if (seg[b * S + j] == myseg) m = fmaxf(m, s[j]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  __syncthreads();
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float l = 0.0f;
  for (int j = threadIdx.x; j <= row; j += 256)
    if (seg[b * S + j] == myseg) l += ixt_exp(s[j] - m);
  l = t_block_sum(l, red);
  for (int j = threadIdx.x; j < end; j += 256) {
    const bool on = j <= row && seg[b * S + j] == myseg;
    p[j] = on ? f2bf(ixt_exp(s[j] - m) / l) : (bf16_t)0;
  }
}
// A wave a row, for rows of at most 256 MAXV <= 2048 columns: no wave waits for another (a block a row: 25.7 us for 48 heads of 512 x 512, 510 for 128 of 2048 x 2048, now 14.4 and 390).  The sums are
// those of the block: lane L adds up what threads L, L + 64, .. of it would, and their waves' sums are added in the same order.
template <int MAXV>
static __global__ __launch_bounds__(256) void k_t_softmax_fwd_wave(const float* __restrict__ sc, const int32_t* __restrict__ seg, bf16_t* __restrict__ P, int S, int H) {
  __shared__ __attribute__((aligned(16))) bf16_t tiles[4][256 * MAXV];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), row = blockIdx.x * 4 + wave;
  if (row >= S) return;                                    // whole wave: no barrier in here
  const long bh = blockIdx.y, b = bh / H;
  const float* s = sc + (bh * S + row) * S;
  const int32_t* sg = seg + b * S;
  bf16_t* tile = tiles[wave];
  const int myseg = sg[row], nv = row / 256 + 1;
  float v[MAXV][4], m = -INFINITY;
  int g[MAXV][4];
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) {                                          // every load at once
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int j = min(i * 256 + w * 64 + lane, row);
        v[i][w] = s[j]; g[i][w] = sg[j];
      }
    }
  uint32_t on = 0;
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const bool see = i * 256 + w * 64 + lane <= row && g[i][w] == myseg;
        on |= see ? 1u << (i * 4 + w) : 0u;
        m = fmaxf(m, see ? v[i][w] : -INFINITY);
      }
    }
  m = xor_butterfly(m, [](float x, float y) { return fmaxf(x, y); });
  float l[4] = {0.0f, 0.0f, 0.0f, 0.0f};
  bool small = false;
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const bool see = on >> (i * 4 + w) & 1u;
        v[i][w] = see ? ixt_exp(v[i][w] - m) : 0.0f;
        small = small || (see && v[i][w] < 0x1p-96f);
        l[w] += v[i][w];
      }
    }
  const float sum = t_wave_sum(l[0]) + t_wave_sum(l[1]) + t_wave_sum(l[2]) + t_wave_sum(l[3]), rl = 1.0f / sum;
  auto write = [&](auto quotient) {
#pragma unroll
    for (int i = 0; i < MAXV; ++i)
      if (i < nv) {
#pragma unroll
        for (int w = 0; w < 4; ++w) tile[i * 256 + w * 64 + lane] = f2bf(quotient(v[i][w]));
      }
  };
  // the quotient by the reciprocal and two corrections, the last of which rounds as a division does where no residue is lost below the normal numbers
  if (__any(small)) write([&](float e) { return e / sum; });
  else write([&](float e) {
    float q = e * rl;
    q = __builtin_fmaf(__builtin_fmaf(-q, sum, e), rl, q);
    return __builtin_fmaf(__builtin_fmaf(-q, sum, e), rl, q);
  });
  wave_lds_sync();
  const int n = min(S, nv * 256);
  bf16_t* out = P + (bh * S + row) * S;
  for (int j = lane * 8; j < n; j += 512) *reinterpret_cast<u32x4*>(out + j) = *reinterpret_cast<const u32x4*>(tile + j);
}
template <int MAXV>
static __global__ __launch_bounds__(256) void k_t_softmax_fwd_reg(const float* __restrict__ sc, const int32_t* __restrict__ seg, bf16_t* __restrict__ P, int S, int H) {
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) bf16_t tile[256 * MAXV];
  const int row = blockIdx.x, tid = threadIdx.x;
  const long bh = blockIdx.y, b = bh / H;
  const float* s = sc + (bh * S + row) * S;
  const int myseg = seg[b * S + row], nv = row / 256 + 1;
  float v[MAXV];
  int sg[MAXV];
  unsigned on = 0;
  float m = -INFINITY;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {                         // every load at once: behind the test of its segment each was a latency of its own (2048 x 2048, 128 heads: 716 us -> 510)
    const int j = min(tid + i * 256, row);
    if (i < nv) { v[i] = s[j]; sg[i] = seg[b * S + j]; }
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    if (i < nv && tid + i * 256 <= row && sg[i] == myseg) on |= 1u << i;
    else v[i] = -INFINITY;
  }
#pragma unroll
  for (int i = 0; i < MAXV; ++i) m = fmaxf(m, v[i]);
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float l = 0.0f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    if (i < nv) { v[i] = ((on >> i) & 1u) ? ixt_exp(v[i] - m) : 0.0f; l += v[i]; }
  }
  l = t_block_sum(l, red);
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) tile[tid + i * 256] = f2bf(v[i] / l);
  __syncthreads();
  t_store_tiles(tile, P + (bh * S + row) * S, min(S, nv * 256), tid);
}
// dS = P o (dP - sum_j dP P), bf16 out (a separate buffer), columns as above.  grid = (S, BH), block 256.
static __global__ __launch_bounds__(256) void k_t_softmax_bwd(const float* __restrict__ dP, const bf16_t* __restrict__ P, bf16_t* __restrict__ dS, int S) {
  __shared__ float red[4];
  const int row = blockIdx.x, end = min(S, (row / 256 + 1) * 256);
  const long base = ((long)blockIdx.y * S + row) * S;
  float s = 0.0f;
  for (int j = threadIdx.x; j <= row; j += 256) s += dP[base + j] * bf2f(P[base + j]);
  const float dot = t_block_sum(s, red);
  for (int j = threadIdx.x; j < end; j += 256) {
    const float p = j <= row ? bf2f(P[base + j]) : 0.0f;
    dS[base + j] = j <= row ? f2bf(p * (dP[base + j] - dot)) : (bf16_t)0;
  }
}
// a wave a row, as k_t_softmax_fwd_wave: 48 heads of 512 x 512 20.8 us by blocks, now 13.1; 128 of 2048 x 2048, where a wave would hold 32 columns a lane, 413 by blocks and 444 so
template <int MAXV>
static __global__ __launch_bounds__(256) void k_t_softmax_bwd_wave(const float* __restrict__ dP, const bf16_t* __restrict__ P, bf16_t* __restrict__ dS, int S) {
  __shared__ __attribute__((aligned(16))) bf16_t tiles[4][256 * MAXV];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), row = blockIdx.x * 4 + wave;
  if (row >= S) return;                                    // whole wave: no barrier in here
  bf16_t* tile = tiles[wave];
  const int nv = row / 256 + 1, n = min(S, nv * 256);
  const long base = ((long)blockIdx.y * S + row) * S;
  float g[MAXV][4];
  u32x4 p[MAXV / 2];
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) {
#pragma unroll
      for (int w = 0; w < 4; ++w) g[i][w] = dP[base + min(i * 256 + w * 64 + lane, row)];
    }
#pragma unroll
  for (int i = 0; i < MAXV / 2; ++i)
    if (i * 512 + lane * 8 < n) p[i] = *reinterpret_cast<const u32x4*>(P + base + i * 512 + lane * 8);
#pragma unroll
  for (int i = 0; i < MAXV / 2; ++i)
    if (i * 512 + lane * 8 < n) *reinterpret_cast<u32x4*>(tile + i * 512 + lane * 8) = p[i];
  wave_lds_sync();
  float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int j = i * 256 + w * 64 + lane;
        const bool in = j <= row;
        s[w] += (in ? g[i][w] : 0.0f) * (in ? bf2f(tile[j]) : 0.0f);
      }
    }
  const float dot = t_wave_sum(s[0]) + t_wave_sum(s[1]) + t_wave_sum(s[2]) + t_wave_sum(s[3]);
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int j = i * 256 + w * 64 + lane;
        const bool in = j <= row;
        tile[j] = f2bf((in ? bf2f(tile[j]) : 0.0f) * ((in ? g[i][w] : 0.0f) - dot));
      }
    }
  wave_lds_sync();
  for (int j = lane * 8; j < n; j += 512) *reinterpret_cast<u32x4*>(dS + base + j) = *reinterpret_cast<const u32x4*>(tile + j);
}
template <int MAXV>
static __global__ __launch_bounds__(256) void k_t_softmax_bwd_reg(const float* __restrict__ dP, const bf16_t* __restrict__ P, bf16_t* __restrict__ dS, int S) {
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) bf16_t tile[256 * MAXV];
  const int row = blockIdx.x, tid = threadIdx.x, nv = row / 256 + 1, n = min(S, nv * 256);
  const long base = ((long)blockIdx.y * S + row) * S;
  float g[MAXV], pv[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int j = tid + i * 256;
    g[i] = i < nv && j <= row ? dP[base + j] : 0.0f;
  }
  for (int j = tid * 8; j < n; j += 2048) *reinterpret_cast<u32x4*>(tile + j) = *reinterpret_cast<const u32x4*>(P + base + j);
  __syncthreads();
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int j = tid + i * 256;
    pv[i] = i < nv && j <= row ? bf2f(tile[j]) : 0.0f;
    if (i < nv) s += g[i] * pv[i];
  }
  const float dot = t_block_sum(s, red);
#pragma unroll
  for (int i = 0; i < MAXV; ++i)
    if (i < nv) tile[tid + i * 256] = f2bf(pv[i] * (g[i] - dot));
  __syncthreads();
  t_store_tiles(tile, dS + base, n, tid);
}

// SwiGLU (linears.py:449-464) forward: act = bf16(bf16(a sg) b), sg = bf16(sigmoid(a)); backward through the unrounded formula.
static __global__ void k_t_swiglu_fwd(const bf16_t* __restrict__ a, const bf16_t* __restrict__ b, bf16_t* __restrict__ act, long n) {   // n a multiple of 8
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (i >= n) return;
  const u32x4 aw = *reinterpret_cast<const u32x4*>(a + i), bw = *reinterpret_cast<const u32x4*>(b + i);
  u32x4 o;
#pragma unroll
  for (int k = 0; k < 4; ++k) o[k] = pack2(ixt_swiglu(bflo(aw[k]), bflo(bw[k])), ixt_swiglu(bfhi(aw[k]), bfhi(bw[k])));
  *reinterpret_cast<u32x4*>(act + i) = o;
}
static __global__ void k_t_swiglu_bwd(const bf16_t* __restrict__ dact, const bf16_t* __restrict__ a, const bf16_t* __restrict__ b, bf16_t* __restrict__ da,
                               bf16_t* __restrict__ db, long n) {
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (i >= n) return;
  float av[8], bv[8], g[8], oa[8], ob[8];
  t_unpack8(*reinterpret_cast<const u32x4*>(a + i), av);
  t_unpack8(*reinterpret_cast<const u32x4*>(b + i), bv);
  t_unpack8(*reinterpret_cast<const u32x4*>(dact + i), g);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float sg = 1.0f / (1.0f + ixt_exp(-av[k]));
    oa[k] = g[k] * bv[k] * sg * (1.0f + av[k] * (1.0f - sg));
    ob[k] = g[k] * av[k] * sg;
  }
  *reinterpret_cast<u32x4*>(da + i) = t_pack8(oa);
  *reinterpret_cast<u32x4*>(db + i) = t_pack8(ob);
}

static __global__ void k_t_f32_to_bf16(const float* __restrict__ a, bf16_t* __restrict__ out, long n) {   // n a multiple of 8
  const long i = ((long)blockIdx.x * blockDim.x + threadIdx.x) * 8;
  if (i >= n) return;
  const float4 u = *reinterpret_cast<const float4*>(a + i), v = *reinterpret_cast<const float4*>(a + i + 4);
  const float w[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
  *reinterpret_cast<u32x4*>(out + i) = t_pack8(w);
}

// embedding: forward gather (embeddings.py:154) = k_embed of ixt_kernels.h; backward scatter-add of dh f32 [T][E] into dE f32 [V][E]
static __global__ void k_t_embed_bwd(const float* __restrict__ dh, const int32_t* __restrict__ ids, float* __restrict__ dE, int E, int V) {
  const long t = blockIdx.y;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= E) return;
  int id = ids[t];
  id = id < 0 ? 0 : (id >= V ? V - 1 : id);
  atomicAdd(dE + (long)id * E + e, dh[t * E + e]);
}

// cross entropy with the reference's VJP (max_utils.py:563-654, z_loss = 0) on a chunk of logits [Tc][V] (bf16, decoders.py:570,586):
// loss_row = log(sum exp(l - max)) + max - l[target]; dlogits = (softmax - onehot) * weight, bf16.  The row is read 2048 columns at a time, 16 bytes a
// thread; the sum's terms reach the threads that own them (column mod 256) through LDS.  grid = Tc, block 256.
static __global__ __launch_bounds__(256) void k_t_xent(const bf16_t* __restrict__ logits, const int32_t* __restrict__ targets, const int32_t* __restrict__ tseg,
                                                bf16_t* __restrict__ dlogits, float* __restrict__ row_loss, int V, long ld) {
  __shared__ float red[4];
  __shared__ __attribute__((aligned(16))) bf16_t tile[2][2048];
  const long row = blockIdx.x;
  const int tid = threadIdx.x;
  const bf16_t* l = logits + row * ld;
  float m = -INFINITY;
  for (int j = tid * 8; j < V; j += 2048) {
    float v[8];
    t_unpack8(*reinterpret_cast<const u32x4*>(l + j), v);
#pragma unroll
    for (int k = 0; k < 8; ++k) m = fmaxf(m, v[k]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) m = fmaxf(m, __shfl_xor(m, off, 64));
  __syncthreads();
  if ((tid & 63) == 0) red[tid >> 6] = m;
  __syncthreads();
  m = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
  float s = 0.0f;
  u32x4 w = tid * 8 < V ? *reinterpret_cast<const u32x4*>(l + tid * 8) : u32x4(0u);
  int buf = 0;
  for (int j0 = 0; j0 < V; j0 += 2048, buf ^= 1) {
    *reinterpret_cast<u32x4*>(&tile[buf][tid * 8]) = w;
    __syncthreads();                                     // (the other buffer is written next: one barrier per tile)
    if (j0 + 2048 + tid * 8 < V) w = *reinterpret_cast<const u32x4*>(l + j0 + 2048 + tid * 8);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (j0 + i * 256 + tid < V) s += ixt_exp(bf2f(tile[buf][i * 256 + tid]) - m);
  }
  s = t_block_sum(s, red);
  const float wt = tseg[row] != 0 ? 1.0f : 0.0f;
  const int tg = targets[row];
  if (tid == 0) row_loss[row] = wt * (logf(s) + m - bf2f(l[tg]));
  const float inv = wt / s;
  for (int j = tid * 8; j < V; j += 2048) {
    float v[8];
    t_unpack8(*reinterpret_cast<const u32x4*>(l + j), v);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = ixt_exp(v[k] - m) * inv - (j + k == tg ? wt : 0.0f);
    *reinterpret_cast<u32x4*>(dlogits + row * ld + j) = t_pack8(v);
  }
}

// The same for wide rows, a block of sixteen waves a row and CU: the rows in work (256 of 528 KB) stay in the memory-side cache between the three passes over them
// (2048 rows of 264192 columns: 971 us a chunk with eight blocks of four waves on a CU, all 2048 rows in work at once and 4.3 GB from memory; now 737).
// The terms of the sum are worked out 16 bytes of logits a thread and added up by the four waves of the form above, column by column in its order.  grid = Tc, block 1024.
static __global__ __launch_bounds__(1024) void k_t_xent_wide(const bf16_t* __restrict__ logits, const int32_t* __restrict__ targets, const int32_t* __restrict__ tseg,
                                                      bf16_t* __restrict__ dlogits, float* __restrict__ row_loss, int V, long ld) {
  extern __shared__ __attribute__((aligned(16))) float term[];   // [2][8192]
  __shared__ float red[16];
  const long row = blockIdx.x;
  const int tid = threadIdx.x, wave = tid >> 6;
  const bf16_t* l = logits + row * ld;
  auto load = [&](int j) { return *reinterpret_cast<const u32x4*>(l + min(j, V - 8)); };      // (V a multiple of 8; past the end: the last eight again)
  float m = -INFINITY;
  for (int j = tid * 8; j < V; j += 4 * 8192) {
    u32x4 w[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) w[u] = load(j + u * 8192);
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      float v[8];
      t_unpack8(w[u], v);
#pragma unroll
      for (int k = 0; k < 8; ++k) m = fmaxf(m, v[k]);
    }
  }
  m = xor_butterfly(m, [](float x, float y) { return fmaxf(x, y); });
  if ((tid & 63) == 0) red[wave] = m;
  __syncthreads();
#pragma unroll
  for (int k = 0; k < 16; ++k) m = fmaxf(m, red[k]);
  float s = 0.0f;
  u32x4 w = load(tid * 8);
  int buf = 0;
  for (int j0 = 0; j0 < V; j0 += 8192, buf ^= 8192) {
    float v[8];
    t_unpack8(w, v);
    w = load(j0 + 8192 + tid * 8);
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = ixt_exp(v[k] - m);
    float4* to = reinterpret_cast<float4*>(term + buf + tid * 8);
    to[0] = make_float4(v[0], v[1], v[2], v[3]); to[1] = make_float4(v[4], v[5], v[6], v[7]);
    __syncthreads();                                     // (the other buffer is written next: one barrier per tile)
    if (wave < 4) {
      const int n = min(32, (V - j0 - tid + 255) >> 8);  // rows of 256 columns that hold this thread's
      if (n == 32) {
#pragma unroll
        for (int i = 0; i < 32; ++i) s += term[buf + i * 256 + tid];
      } else {
        for (int i = 0; i < n; ++i) s += term[buf + i * 256 + tid];
      }
    }
  }
  __syncthreads();
  s = t_wave_sum(s);
  if (wave < 4 && (tid & 63) == 0) red[wave] = s;
  __syncthreads();
  s = red[0] + red[1] + red[2] + red[3];
  const float wt = tseg[row] != 0 ? 1.0f : 0.0f;
  const int tg = targets[row];
  if (tid == 0) row_loss[row] = wt * (logf(s) + m - bf2f(l[tg]));
  const float inv = wt / s;
  for (int j = tid * 8; j < V; j += 2 * 8192) {
    const u32x4 x[2] = {load(j), load(j + 8192)};
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const int at = j + u * 8192;
      if (at >= V) continue;
      float v[8];
      t_unpack8(x[u], v);
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] = ixt_exp(v[k] - m) * inv;
      if ((unsigned)(tg - at) < 8u) {
#pragma unroll
        for (int k = 0; k < 8; ++k) v[k] -= at + k == tg ? wt : 0.0f;
      }
      *reinterpret_cast<u32x4*>(dlogits + row * ld + at) = t_pack8(v);
    }
  }
}

// out[i] = 1 where s[i] != 0 (the weight of a target position, train.py:308-309)
static __global__ void k_t_nonzero(const int32_t* __restrict__ s, float* __restrict__ out, long n) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = s[i] != 0 ? 1.0f : 0.0f;
}

// fixed-order sum of n floats by one block (deterministic), optionally of squares; out[0] (+)= sum
static __global__ __launch_bounds__(256) void k_t_reduce(const float* __restrict__ x, long n, int squares, float* __restrict__ out, int accumulate) {
  __shared__ float red[4];
  double s = 0.0;
  for (long i = threadIdx.x; i < n; i += 256) { const float v = x[i]; s += squares ? (double)v * v : (double)v; }
  float f = (float)s;
  f = t_block_sum(f, red);
  if (threadIdx.x == 0) out[0] = (accumulate ? out[0] : 0.0f) + f;
}
// sum of squares of a large buffer: one partial per block, then k_t_reduce over the partials.  grid = nblk, block 256.
static __global__ __launch_bounds__(256) void k_t_sumsq_partial(const float* __restrict__ x, long n, float* __restrict__ part) {
  __shared__ float red[4];
  float s = 0.0f;
  const long step = (long)gridDim.x * 256;
  long i = (long)blockIdx.x * 256 + threadIdx.x;
  for (; i + 7 * step < n; i += 8 * step) {              // eight loads in flight, added one after the other
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; ++k) v[k] = x[i + k * step];
#pragma unroll
    for (int k = 0; k < 8; ++k) s += v[k] * v[k];
  }
  for (; i < n; i += step) { const float v = x[i]; s += v * v; }
  s = t_block_sum(s, red);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}

// optax.clip_by_global_norm + optax.adamw (optimizers.py:28-38): g <- g * gscale (1 / total_weights and the clip factor), mu, nu, bias
// correction with `count` (1 at the first step), decoupled weight decay, p -= lr * update; the bf16 copy of the parameter is refreshed.
struct AdamArgs { float lr, b1, b2, eps, eps_root, wd, bc1, bc2; };
static __global__ void k_t_adamw(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ mu, float* __restrict__ nu, bf16_t* __restrict__ pb,
                          const float* __restrict__ gscale, long n, long ld, AdamArgs a) {
  const long x = (long)blockIdx.x * blockDim.x + threadIdx.x, i = blockIdx.y * n + x;
  if (x >= n) return;
  const float gv = g[i] * gscale[0];
  const float m = a.b1 * mu[i] + (1.0f - a.b1) * gv;
  const float v = a.b2 * nu[i] + (1.0f - a.b2) * gv * gv;
  mu[i] = m; nu[i] = v;
  const float upd = (m / a.bc1) / (sqrtf(v / a.bc2 + a.eps_root) + a.eps) + a.wd * p[i];
  const float np_ = p[i] - a.lr * upd;
  p[i] = np_;
  pb[blockIdx.y * ld + x] = f2bf(np_);
}
// gscale[0] = (1 / denom) * min(1, clip / (norm / denom)) with norm = sqrt(sumsq[0]); norms_out = {raw grad norm, clipped grad norm}
static __global__ void k_t_clip_scale(const float* __restrict__ sumsq, float denom, float clip, float* __restrict__ gscale, float* __restrict__ norms_out) {
  const float raw = sqrtf(sumsq[0]) / denom;
  const float f = (clip > 0.0f && raw >= clip) ? clip / raw : 1.0f;
  gscale[0] = f / denom;
  norms_out[0] = raw;
  norms_out[1] = raw * f;
}
