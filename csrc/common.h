// Shared device helpers for the gfx950 (CDNA4) kernel library.
//
// Everything here is written for wave64 / MFMA hardware directly: bf16 values
// travel as raw 16-bit patterns (ushort) so loads vectorise to 16 B/lane, and
// reductions are 64-lane butterflies.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernels.h"

#define LK_DEVICE __device__ __forceinline__

typedef unsigned short bf16_t;  // raw bf16 bits
typedef short short8 __attribute__((ext_vector_type(8)));
typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned int uint4_t __attribute__((ext_vector_type(4)));

constexpr int kWave = 64;

LK_DEVICE float bf2f(bf16_t v) { return __uint_as_float(((unsigned)v) << 16); }

// round-to-nearest-even f32 -> bf16: gfx950 has v_cvt_pk_bf16_f32, which the
// __bf16 cast lowers to (NaN stays NaN, unlike the integer rounding trick).
LK_DEVICE bf16_t f2bf(float f) {
  __bf16 b = (__bf16)f;
  return __builtin_bit_cast(bf16_t, b);
}

// two f32 -> one dword of 2 x bf16 (lo in bits 0-15): a vector conversion lowers to ONE
// v_cvt_pk_bf16_f32 (two scalar casts cost two converts + a shift + an or)
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float floatx2_t __attribute__((ext_vector_type(2)));
LK_DEVICE unsigned pack_bf2(float lo, float hi) {
  return __builtin_bit_cast(unsigned, __builtin_convertvector((floatx2_t){lo, hi}, bf16x2_t));
}

// Butterflies over the 64 lanes in the order 32, 16, 8, 4, 2, 1 (every lane ends with the same bits), by lane swaps and row rotations
// of the vector unit: __shfl_xor goes through the LDS unit, whose latency was most of a short row's reduction.
template <int STEP>
LK_DEVICE float wave_partner(float v) {  // the value of lane ^ STEP or of another lane that holds the same partial result
  return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v), 0x120 + STEP, 0xf, 0xf, true));  // row_ror
}
template <typename F>
LK_DEVICE float wave_all(float v, F f) {
  auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(h[0]), __uint_as_float(h[1]));
  auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = f(__uint_as_float(q[0]), __uint_as_float(q[1]));
  v = f(v, wave_partner<8>(v));
  v = f(v, wave_partner<4>(v));
  v = f(v, wave_partner<2>(v));
  return f(v, wave_partner<1>(v));
}
LK_DEVICE float wave_sum(float v) {
  return wave_all(v, [](float a, float b) { return a + b; });
}
LK_DEVICE float wave_max(float v) {
  return wave_all(v, [](float a, float b) { return fmaxf(a, b); });
}

// block-wide sum for blockDim.x = NW*64; `red` must hold NW floats.
template <int NW>
LK_DEVICE float block_sum(float v, float* red) {
  v = wave_sum(v);
  if constexpr (NW == 1) {
    return v;
  } else {
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    __syncthreads();
    if (lane == 0) red[w] = v;
    __syncthreads();
    float t = 0.f;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += red[i];
    return t;
  }
}

// 8 x bf16 <-> 8 x f32 through one 16-byte access
LK_DEVICE void load8(const bf16_t* p, float* f) {
  short8 v = *reinterpret_cast<const short8*>(p);
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = bf2f((bf16_t)v[i]);
}
LK_DEVICE void store8(bf16_t* p, const float* f) {
  short8 v;
#pragma unroll
  for (int i = 0; i < 8; ++i) v[i] = (short)f2bf(f[i]);
  *reinterpret_cast<short8*>(p) = v;
}

// Activations shared by the elementwise kernels and the GEMM epilogues.
// the pair (a, b) turned by an angle: (a c - b s, b c + a s), one product rounded before the fma.  Written out, so that every kernel
// that rotates (alone or in a product's epilogue) rounds alike.
LK_DEVICE float rot_lo(float a, float b, float c, float s) { return __builtin_fmaf(a, c, -(b * s)); }
LK_DEVICE float rot_hi(float a, float b, float c, float s) { return __builtin_fmaf(b, c, a * s); }

LK_DEVICE float lk_silu(float x) { return x / (1.f + __expf(-x)); }
// GELU x Phi(x) through the small tail h = Phi(-|x|): log2 h is nearly a parabola, so h = 2^q(|x|) with q a polynomial of degree 8
// (a minimax fit of log2 Phi(-a) over 0 .. 5 that weighs an error by what it moves in a h; its leading coefficient is negative, so h
// goes on falling to 0 behind the fit and for infinities), and x > 0 takes 1 - h.  Against float64 over |x| <= 12: error at most
// 3.9e-7 (half an ulp of the largest values), 5.0e-8 on average, 2e-4 of the value in the negative tail to -5; an erf of 1.5e-7 by
// an exponential and a reciprocal had 4.7e-7, 8.4e-8 and 5e-2.  12 instructions and one transcendental instead of 16 and two: the
// epilogues with it are bound by them; an encoder batch's 768 -> 3072 projection in the one-wave GEMM went from 350 to 316 us.
LK_DEVICE float lk_gelu_erf(float x) {
  const float a = fabsf(x);
  float q = -1.349546437e-06f;
  q = fmaf(q, a, 2.133819362e-05f);
  q = fmaf(q, a, -9.924922779e-05f);
  q = fmaf(q, a, -3.501909960e-04f);
  q = fmaf(q, a, 7.347176317e-03f);
  q = fmaf(q, a, -5.269736424e-02f);
  q = fmaf(q, a, -4.591392875e-01f);
  q = fmaf(q, a, -1.151113987e+00f);
  q = fmaf(q, a, -9.999998212e-01f);
  const float h = __builtin_amdgcn_exp2f(q);
  return x * (x > 0.f ? 1.f - h : h);
}

// Bijective XCD-aware remap of a flat workgroup id (8 XCDs, round-robin dispatch):
// consecutive logical tiles land on the same XCD so they share its L2.
LK_DEVICE int xcd_remap(int bid, int nwg) {
  const int q = nwg / 8, r = nwg % 8;
  const int xcd = bid % 8, idx = bid / 8;
  return (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + idx;
}

// Launch failures are loud: a rejected launch (bad grid / block / LDS request) returns a
// distinct code that the bindings turn into a Python exception (bindings.cpp CHECK_RC), never
// a "successful" op over an uninitialised output.
// (the codes kLkLaunchError / kLkAttrError are in kernels.h, shared with the bindings)
// first refused kernel attribute of the process (sticky: the kernel it belongs to cannot run)
inline hipError_t& lk_attr_error() {
  static hipError_t e = hipSuccess;
  return e;
}
#define LK_CHECK_LAUNCH()                                                           \
  do {                                                                              \
    const hipError_t lk_e_ = hipGetLastError();                                     \
    if (lk_attr_error() != hipSuccess) return kLkAttrError - (int)lk_attr_error(); \
    if (lk_e_ != hipSuccess) return kLkLaunchError - (int)lk_e_;                    \
  } while (0)
// One-time dynamic-LDS opt-in of a kernel, its result kept: a refusal is reported by the
// launch's LK_CHECK_LAUNCH instead of surfacing as an unexplained launch failure.
#define LK_SET_MAX_LDS(kern, bytes)                                                                     \
  do {                                                                                                  \
    static const hipError_t lk_attr_ = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),        \
                                                           hipFuncAttributeMaxDynamicSharedMemorySize, \
                                                           (int)(bytes));                              \
    if (lk_attr_ != hipSuccess) lk_attr_error() = lk_attr_;                                             \
  } while (0)

// Device-side bounds checks for debug builds (`python csrc/build.py --debug`, objects
// under build/csrc-debug): a failing check traps the wave with the kernel's file/line
// instead of silently reading or writing out of range.  Compiled out otherwise.
#ifdef LK_DEBUG
#include <cassert>
#define LK_DASSERT(cond) assert(cond)
#else
#define LK_DASSERT(cond) ((void)0)
#endif
