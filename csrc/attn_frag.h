// Fragment helpers shared by the attention kernels that read a paged K cache [blocks, G, BS, dim] and a
// key-contiguous V cache [blocks, G, vdim, BS] straight into MFMA operands (attn_sigmoid.hip,
// attn_sink.hip), and by the products that read rows straight from memory (moe.hip, head_linear.hip, row_proj.hip):
// element traits of the two activation types, the S^T += K . Q^T step, a padded 16-byte fragment of a row.
#pragma once
#include "common.h"

namespace {

template <typename T>
struct El;
template <>
struct El<bf16_t> {
  static constexpr int V = 8;  // elements per 16-byte fragment
  static LK_DEVICE float ld(const bf16_t* p) { return bf2f(*p); }
  static LK_DEVICE void st(bf16_t* p, float v) { *p = f2bf(v); }
};
template <>
struct El<float> {
  static constexpr int V = 4;
  static LK_DEVICE float ld(const float* p) { return *p; }
  static LK_DEVICE void st(float* p, float v) { *p = v; }
};

LK_DEVICE uint4_t ld16(const void* p) { return *reinterpret_cast<const uint4_t*>(p); }
// NT: read once (the keys and values of a decode step; 64 sequences of 950 keys, 4 kv heads: sigmoid attention 34.1 -> 32.9 us, windowed
// softmax 21.9 -> 20.9 us)
template <bool NT>
LK_DEVICE uint4_t ld16_kv(const void* p) {
  return NT ? __builtin_nontemporal_load(reinterpret_cast<const uint4_t*>(p)) : ld16(p);
}

// S^T += A(16 keys x one 16-byte fragment of dims) . B(the columns' same dims)
template <typename T>
LK_DEVICE floatx4 mma_qk(uint4_t a, uint4_t b, floatx4 c) {
  if constexpr (sizeof(T) == 2) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(short8, a), __builtin_bit_cast(short8, b), c, 0, 0, 0);
  } else {
    const floatx4 fa = __builtin_bit_cast(floatx4, a), fb = __builtin_bit_cast(floatx4, b);
#pragma unroll
    for (int e = 0; e < 4; ++e) c = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[e], fb[e], c, 0, 0, 0);
    return c;
  }
}

// 16 bytes of row `r` at element k (EV elements; zeros past K): one vector load when the row allows it
template <typename T>
LK_DEVICE uint4_t frag(const T* r, int k, int K, bool vec) {
  constexpr int EV = El<T>::V;
  if (vec && k + EV <= K) return ld16(r + k);
  alignas(16) T tmp[EV];
#pragma unroll
  for (int e = 0; e < EV; ++e) tmp[e] = k + e < K ? r[k + e] : T(0);
  return *reinterpret_cast<const uint4_t*>(tmp);
}

typedef void __attribute__((address_space(3))) * lds_void_ptr;

// maximum over the four lane groups (lanes l, l ^ 16, l ^ 32, l ^ 48), in registers
LK_DEVICE float max_groups(float v) {
  // (the swapped pair is taken apart as integers: a bit cast of a vector's element reads element 0)
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const unsigned a0 = a[0], a1 = a[1];
  v = fmaxf(__uint_as_float(a0), __uint_as_float(a1));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  const unsigned b0 = b[0], b1 = b[1];
  return fmaxf(__uint_as_float(b0), __uint_as_float(b1));
}

// one fragment: lane l's 16 bytes at src go to LDS byte off + 16 l (off wave-uniform).  As assembly: the compiler would wait for the
// transfer before the next LDS read of the OTHER buffer; a kernel's loop waits for it itself, ahead of its barrier.
template <bool NT = false>
LK_DEVICE void dma16(unsigned off, const void* src) {
  if constexpr (NT) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off nt" ::"s"(off), "v"(src) : "memory", "m0");
  else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(off), "v"(src) : "memory", "m0");
}

}  // namespace
