// ixt_device.h -- scalar numerics shared by every kernel ("IXT-MFMA-v2").
// Compiled with -ffp-contract=off: a*b+c never fuses; every fused multiply-add is an explicit fmaf.
#pragma once
#include "ixt_lds_room.h"

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

typedef uint16_t bf16_t;

// room for `bytes` of dynamic LDS in launches of Kernel on the current device, asked for once a device
template <auto Kernel> static inline hipError_t lds_room(size_t bytes) {
  static IxtLdsRoom room;
  int device = -1;
  const hipError_t e = hipGetDevice(&device);
  if (e != hipSuccess) return e;
  return (hipError_t)room.ask(device, bytes, [&] { return (int)hipFuncSetAttribute(reinterpret_cast<const void*>(Kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes); });
}

#define IXT_MK 32      // k per matrix instruction (v_mfma_f32_16x16x32_bf16)
#define IXT_CHAIN 512  // k per accumulator chain of the canonical dot = the unit of a split-K slice
#define IXT_KALIGN 128 // feature dimensions must be multiples of this
#define IXT_SB 4     // logical pages per attention super-block

__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float(((uint32_t)h) << 16); }

// round-to-nearest-even; NaN stays NaN.  gfx950 has the conversion in hardware (v_cvt_pk_bf16_f32: RNE, subnormals kept under this
// build's -fno-gpu-flush-denormals-to-zero); tests/test_gpu_ops.py::test_bf16_conversion_exhaustive compares it with the integer
// formula (u + 0x7fff + ((u >> 16) & 1)) >> 16 over all 2^32 inputs (NaN payloads aside).
__device__ __forceinline__ bf16_t f2bf(float f) { return __builtin_bit_cast(bf16_t, (__bf16)f); }
__device__ __forceinline__ bf16_t f2bf_int(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((u >> 16) | 0x0040u);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (bf16_t)(u >> 16);
}
__device__ __forceinline__ float rbf(float f) { return bf2f(f2bf(f)); }

// two bf16 packed in one dword: low half = element 0
__device__ __forceinline__ float bflo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bfhi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }
__device__ __forceinline__ uint32_t pack2(bf16_t lo, bf16_t hi) { return (uint32_t)lo | ((uint32_t)hi << 16); }

// exp from IEEE-only operations; argument clamped to [-80, 80] (no subnormals, no overflow).
__device__ __forceinline__ float ixt_exp(float x) {
  x = fminf(fmaxf(x, -80.0f), 80.0f);
  float n = __builtin_rintf(x * 1.44269504088896340736f);
  float r = __builtin_fmaf(n, -0.693145751953125f, x);
  r = __builtin_fmaf(n, -1.42860682030941723212e-6f, r);
  float p = 1.98412698412698412698e-4f;
  p = __builtin_fmaf(p, r, 1.38888888888888888889e-3f);
  p = __builtin_fmaf(p, r, 8.33333333333333333333e-3f);
  p = __builtin_fmaf(p, r, 4.16666666666666666667e-2f);
  p = __builtin_fmaf(p, r, 1.66666666666666666667e-1f);
  p = __builtin_fmaf(p, r, 0.5f);
  p = __builtin_fmaf(p, r, 1.0f);
  p = __builtin_fmaf(p, r, 1.0f);
  int e = (int)n;
  float s = __uint_as_float((uint32_t)(e + 127) << 23);
  return p * s;
}

// natural logarithm from IEEE-only operations (positive normal arguments): x = 2^e f, f in [sqrt(1/2), sqrt(2)); z = (f - 1) / (f + 1);
// log f = 2 z (1 + z^2/3 + ... + z^10/11) by Horner fma; result = fma(e, ln2_hi, fma(e, ln2_lo, log f)).
__device__ __forceinline__ float ixt_log(float x) {
  const uint32_t u = __float_as_uint(x);
  int e = (int)(u >> 23) - 127;
  float f = __uint_as_float((u & 0x007fffffu) | 0x3f800000u);
  if (f > 1.41421356237309504880f) { f = f * 0.5f; e = e + 1; }
  const float z = (f - 1.0f) / (f + 1.0f);
  const float w = z * z;
  float p = 9.09090909090909090909e-2f;
  p = __builtin_fmaf(p, w, 1.11111111111111111111e-1f);
  p = __builtin_fmaf(p, w, 1.42857142857142857143e-1f);
  p = __builtin_fmaf(p, w, 0.2f);
  p = __builtin_fmaf(p, w, 3.33333333333333333333e-1f);
  p = __builtin_fmaf(p, w, 1.0f);
  const float lf = (z + z) * p;
  const float fe = (float)e;
  return __builtin_fmaf(fe, 0.693145751953125f, __builtin_fmaf(fe, 1.42860682030941723212e-6f, lf));
}

__device__ __forceinline__ float ixt_sigmoid(float a) { return rbf(1.0f / (1.0f + ixt_exp(-a))); }
// MlpBlock gate: bf16(bf16(a * bf16(sigmoid(a))) * b)
__device__ __forceinline__ bf16_t ixt_swiglu(float a, float b) {
  float u = rbf(a * ixt_sigmoid(a));
  return f2bf(u * b);
}

// tanh from IEEE-only operations.  |x| < 1/16: odd series x (1 - x^2/3 + 2 x^4/15 - 17 x^6/315) by Horner fma (next term < 2e-13 relative);
// |x| >= 10: 1 (1 - tanh < 2^-25); else (1 - e) / (1 + e), e = ixt_exp(-2 |x|).  Sign copied from x.
__device__ __forceinline__ float ixt_tanh(float x) {
  const float a = fabsf(x);
  float t;
  if (a < 0.0625f) {
    const float w = a * a;
    float p = -5.39682539682539682540e-2f;
    p = __builtin_fmaf(p, w, 1.33333333333333333333e-1f);
    p = __builtin_fmaf(p, w, -3.33333333333333333333e-1f);
    p = __builtin_fmaf(p, w, 1.0f);
    t = a * p;
  } else if (a >= 10.0f) {
    t = 1.0f;
  } else {
    const float e = ixt_exp(-2.0f * a);
    t = (1.0f - e) / (1.0f + e);
  }
  return copysignf(t, x);
}

// Gemma MlpBlock gate (mlp_activations ["gelu", "linear"], linears.py:449-464; jax.nn.gelu approximate=True on bf16 values, every
// primitive rounded to bf16): cdf = 0.5 (1 + tanh(c (a + 0.044715 a^3))), bf16(bf16(a * cdf) * b)
__device__ __forceinline__ float ixt_gelu_cdf(float a) {
  const float x3 = rbf(rbf(a * a) * a);
  const float u = rbf(a + rbf(0.044677734375f * x3));       // bf16(0.044715)
  const float th = rbf(ixt_tanh(rbf(0.796875f * u)));       // bf16(sqrt(2 / pi))
  return rbf(0.5f * rbf(1.0f + th));
}
__device__ __forceinline__ bf16_t ixt_geglu(float a, float b) {
  const float g = rbf(a * ixt_gelu_cdf(a));
  return f2bf(g * b);
}

// A gate whose argument is a bf16 value `a` is bf16(a * w(a)), w(a) a bf16 value that depends on `a` alone: bf16(sigmoid(a)), or Gemma's cdf.  Table of w over
// sign and 2^-10 <= |a| <= 2^7; below, w is its value at 2^-10 of that sign (1/2: what is added to 1/2 or 1 is less than half a step of bf16), above, its
// value at 2^7 (ixt_exp clamps its argument at 80, tanh is 1 from 10 on).
#define IXT_GATE_LO ((127 - 10) << 7)
#define IXT_GATE_N (17 * 128 + 1)                    // of one sign
#define IXT_GATE_BYTES 9216                          // both, in whole KiB
__device__ __forceinline__ int ixt_gate_at(uint32_t a) {
  return min(max((int)(a & 0x7fffu), IXT_GATE_LO), IXT_GATE_LO + IXT_GATE_N - 1) - IXT_GATE_LO + (int)(a >> 15) * IXT_GATE_N;
}
// ixt_swiglu / ixt_geglu of bf16(t0) and bf16(t1), bit for bit
__device__ __forceinline__ bf16_t ixt_gate(const bf16_t* table, float t0, float t1) {
  const bf16_t a = f2bf(t0);
  return f2bf(rbf(bf2f(a) * bf2f(table[ixt_gate_at(a)])) * rbf(t1));
}

// gated units in f32, by kind (IXT_GLU_*).  1: g = min(a, limit), u = clamp(b, -limit, limit), g sigmoid(1.702 g) (u + 1); 2: tanh form of gelu, as
// a sigmoid(2 sqrt(2 / pi) (a + 0.044715 a^3)) b; 3: a sigmoid(a) b (ixt_glu)
__device__ __forceinline__ float ixt_glu_clamped(float a, float b, float limit) {
  const float g = fminf(a, limit), u = fminf(fmaxf(b, -limit), limit);
  return g / (1.0f + expf(-1.702f * g)) * (u + 1.0f);
}
// 2^x and 1 / x of the hardware (1 ulp; results below the normal range go to zero)
__device__ __forceinline__ float hw_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ float hw_rcp(float x) { return __builtin_amdgcn_rcpf(x); }
__device__ __forceinline__ float ixt_glu(int kind, float a, float b, float limit) {
  if (kind == 1) return ixt_glu_clamped(a, b, limit);
  const float z = kind == 2 ? 1.59576912160573071176f * fmaf(0.044715f * a * a, a, a) : a;
  return a * hw_rcp(1.0f + hw_exp2(-1.44269504088896340736f * z)) * b;
}
// units without a gate, by kind (from IXT_ACT_RELU2 = 4 on): max(u, 0)^2; 5: par[0] u^2 + u / 2 for u > 0, par[1] (exp(u) - 1 - u) + u / 2 for the others
__device__ __forceinline__ float ixt_act(int kind, float u, const float* __restrict__ par) {
  const float p = fmaxf(u, 0.0f);
  if (kind == 4) return p * p;
  const float n = fminf(u, 0.0f);
  return fmaf(0.5f, u, fmaf(par[0] * p, p, par[1] * (hw_exp2(1.44269504088896340736f * n) - 1.0f - n)));
}
// tanh in f32, error below 1e-6 of the value: (1 - e) / (1 + e), e = exp(-2 |x|); |x| < 1/16 by the odd series (next term < 2e-13 relative)
__device__ __forceinline__ float tanh_f32(float x) {
  const float a = fabsf(x), w = a * a, e = hw_exp2(-2.88539008177792681472f * a);
  const float p = fmaf(fmaf(fmaf(-5.39682539682539682540e-2f, w, 1.33333333333333333333e-1f), w, -3.33333333333333333333e-1f), w, 1.0f);
  return copysignf(a < 0.0625f ? a * p : (1.0f - e) * hw_rcp(1.0f + e), x);
}

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// LDS-DMA by hand: 16 bytes a lane from memory to LDS, lane l's to byte `dst` + 16 l (dst uniform, it goes through M0).  No register is written, and the kernels
// count the waits themselves: behind the builtin the compiler waits for every fetch in flight ahead of an LDS read that it cannot tell from their targets.
// A write of M0 has to stand one wait state in front of a fetch that uses it (the compiler puts this s_nop there for the builtin, but does not look into
// asm), and M0 is named as overwritten: otherwise a fetch of the compiler's own may go to the slot of this one.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"          // (M0 is a reserved register: the compiler keeps nothing in it across this)
#define IXT_LDS_DMA "s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 "
// from base + off, base uniform; ONCE: past the caches
template <bool ONCE = false> __device__ __forceinline__ void lds_dma16(uint32_t dst, const void* base, uint32_t off) {
  if constexpr (ONCE) asm volatile(IXT_LDS_DMA "%1, %2 nt" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
  else asm volatile(IXT_LDS_DMA "%1, %2" ::"s"(dst), "v"(off), "s"(base) : "memory", "m0");
}
// from a lane's own address
__device__ __forceinline__ void lds_dma16(uint32_t dst, const void* src) { asm volatile(IXT_LDS_DMA "%1, off" ::"s"(dst), "v"(src) : "memory", "m0"); }
#undef IXT_LDS_DMA
#pragma clang diagnostic pop
// barrier of a block behind which LDS is read that such fetches (or other waves) filled.  The builtin orders nothing for the compiler, which does not see
// the fetches write: without the fence a read may move in front of it.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// 16 bytes past the XCD's L2 (sc1: agent scope).  A store of more than 8 bytes is still reading its registers when the next instruction issues: the wait state that the compiler puts
// in front of a vector instruction that writes them has to stand here (without it one row of a wave in thousands of launches was wrong)
template <typename V> __device__ __forceinline__ void stg16_agent(void* p, const V& v) {
  static_assert(sizeof(V) == 16, "four registers");
  asm volatile("global_store_dwordx4 %0, %1, off sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
}

// Waits of a block for another one of its launch are bounded: `polls` looks, then the block says so and goes on.  `gave` is the pass's own word on the device (cleared in front of a pass; who
// sees it set waits no more, and k_decode_finish marks the result), `fault` the context's in host memory, which the next call reports.
struct IxtWait { int32_t *gave, *fault; int polls; };
__device__ __forceinline__ void ixt_gave_up(const IxtWait& w) {
  __hip_atomic_store(w.gave, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(w.fault, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// agent-scope (L1-bypassing) accesses for state one wave re-reads after writing it
__device__ __forceinline__ int ldg_i32(const int32_t* p) { return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }
__device__ __forceinline__ void stg_i32(int32_t* p, int v) { __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); }

// v of the lane 1, 2, 4, 8, 16, 32 away combined with this lane's, in the order of the xor-butterfly of the canonical sums: from 4 on the lanes of a group hold the same
// value already, so that any lane of the other group will do (row_half_mirror, row_mirror, swaps of rows and halves), and no step goes through LDS.
template <typename F> __device__ __forceinline__ float xor_butterfly(float v, F f) {
  auto dpp = [](float x, auto ctrl) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), decltype(ctrl)::value, 0xf, 0xf, true)); };
  v = f(v, dpp(v, std::integral_constant<int, 0xb1>()));           // quad_perm 1 0 3 2
  v = f(v, dpp(v, std::integral_constant<int, 0x4e>()));           // quad_perm 2 3 0 1
  v = f(v, dpp(v, std::integral_constant<int, 0x141>()));          // row_half_mirror
  v = f(v, dpp(v, std::integral_constant<int, 0x140>()));          // row_mirror
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float xor_sum(float v) { return xor_butterfly(v, [](float x, float y) { return x + y; }); }

// between LDS writes of a wave's lanes and reads of other lanes of it: the hardware keeps a wave's LDS accesses in order, this keeps the compiler to it (no instruction)
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The row of block b where a block takes a row of R and writes it to an operand (xidx: 16 bytes of a line of eight rows at a time): the eight rows of a line go to blocks that the
// dispatcher deals to one XCD, so that its L2 holds the line whole when it is written back (with
// sums over the lanes that need no LDS, us before / now: k_rownorm of 1592 rows of 2048 7.8 / 5.9, of 1024 6.5 / 5.2; k_gnorm of 256 rows of 2304 6.3 / 5.1).
__device__ __forceinline__ int row_of_block(int b, int R) {
  return (b | 63) < R ? (b & ~63) + (b & 7) * 8 + (b >> 3 & 7) : b;
}
