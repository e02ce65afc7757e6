// A residual stream kept in f32 next to bf16 (or f32) sublayer outputs:
//   * token + learned position embedding gather into the f32 stream (and a second copy for models
//     that add the embedding output again later);
//   * fused "stream update + RMSNorm": x += m * (a + b) + e, h = x / sqrt(mean(x^2) + eps) * (off + w)
//     -- the update of a block whose sublayers all read one norm's output and are summed, and the
//     next block's norm, in one pass over the row (a, b, e optional; off = 1 for weights stored
//     around zero); with a row index list it gathers rows instead and leaves the stream alone (the
//     rows that feed the LM head);
//   * soft-capped logits: cap * tanh(z / cap), f32 out.
#include "common.h"
#include "kernels.h"

namespace {

template <typename T>
LK_DEVICE float ldv(const T* p);
template <>
LK_DEVICE float ldv<bf16_t>(const bf16_t* p) { return bf2f(*p); }
template <>
LK_DEVICE float ldv<float>(const float* p) { return *p; }
template <typename T>
LK_DEVICE void stv(T* p, float v);
template <>
LK_DEVICE void stv<bf16_t>(bf16_t* p, float v) { *p = f2bf(v); }
template <>
LK_DEVICE void stv<float>(float* p, float v) { *p = v; }

__device__ int g_stream_embed_errors = 0;

template <typename T>
__global__ __launch_bounds__(256) void embed_pos_kernel(const int* __restrict__ ids, const int* __restrict__ positions,
                                                        const T* __restrict__ tok, int vocab,
                                                        const T* __restrict__ pos, int max_pos, int W,
                                                        float* __restrict__ x, float* __restrict__ copy) {
  const long row = blockIdx.x;
  const int id = ids[row], ps = positions[row];
  const bool ok = id >= 0 && id < vocab && ps >= 0 && ps < max_pos;
  if (!ok && threadIdx.x == 0) atomicAdd(&g_stream_embed_errors, 1);
  for (int c = threadIdx.x; c < W; c += 256) {
    const float v = ok ? ldv<T>(tok + (long)id * W + c) + ldv<T>(pos + (long)ps * W + c) : 0.f;
    x[row * W + c] = v;
    if (copy) copy[row * W + c] = v;
  }
}

template <typename T>
__global__ __launch_bounds__(256) void stream_rmsnorm_kernel(float* __restrict__ x, const T* __restrict__ a, long as,
                                                             const float* __restrict__ ab, const T* __restrict__ b, long bs,
                                                             const float* __restrict__ e, float m,
                                                             const float* __restrict__ w, float woff, float eps,
                                                             const long* __restrict__ idx, T* __restrict__ out, long os,
                                                             int W) {
  __shared__ float red[4];
  const long orow = blockIdx.x, row = idx ? idx[orow] : orow;
  float ss = 0.f;
  for (int c = threadIdx.x; c < W; c += 256) {
    float v = x[row * W + c];
    float d = 0.f;
    if (a) d += ldv<T>(a + row * as + c) + (ab ? ab[c] : 0.f);
    if (b) d += ldv<T>(b + row * bs + c);
    v += m * d;
    if (e) v += e[row * W + c];
    if (!idx && (a || b || e)) x[row * W + c] = v;
    ss += v * v;
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)W + eps);
  for (int c = threadIdx.x; c < W; c += 256) {
    float v;
    if (!idx) {
      v = x[row * W + c];  // this thread's own store above (or the untouched stream)
    } else {
      v = x[row * W + c];
      float d = 0.f;
      if (a) d += ldv<T>(a + row * as + c) + (ab ? ab[c] : 0.f);
      if (b) d += ldv<T>(b + row * bs + c);
      v += m * d;
      if (e) v += e[row * W + c];
    }
    stv<T>(out + orow * os + c, v * inv * (w ? woff + w[c] : 1.f));
  }
}

// The same with the row kept in registers and 16-byte (f32) / 8-byte (bf16) accesses: W % 4 == 0, W <= 4 * 256 * MAXV, 16-byte
// aligned rows.  One read of every input, one write of x and of out.  A row is short, so what it costs is the trips to memory: every
// input and the weight are requested before anything waits (columns past the row are its last again, and not used), in registers for
// rows of up to 1,024, 2,048, 4,096 or 8,192 (with eight
// pieces and a test for each, one after the other, whatever the width: 4,095 x 2,048 with a 20.4 -> 16.0 us, with b too 23.8 -> 18.4;
// x 4,096 33.0 -> 29.7, x 768 11.8 -> 7.1; 949 x 2,048 6.7 -> 5.1; 117 and 134 MB at 4,095 x 2,048).
template <typename T, int MAXV>
__global__ __launch_bounds__(256) void stream_rmsnorm_vec_kernel(float* __restrict__ x, const T* __restrict__ a, long as,
                                                                 const float* __restrict__ ab, const T* __restrict__ b,
                                                                 long bs,
                                                                 const float* __restrict__ e, float m,
                                                                 const float* __restrict__ w, float woff, float eps,
                                                                 const long* __restrict__ idx, T* __restrict__ out,
                                                                 long os, int W) {
  using Raw = std::conditional_t<sizeof(T) == 2, short4_t, floatx4>;
  __shared__ float red[4];
  const long orow = blockIdx.x, row = idx ? idx[orow] : orow;
  const int nv = W >> 2;
  floatx4 v[MAXV], g[MAXV], ev[MAXV], abv[MAXV];
  Raw ra[MAXV], rb[MAXV];
  auto wide = [](Raw r) -> floatx4 {
    if constexpr (sizeof(T) == 2) return floatx4{bf2f((bf16_t)r[0]), bf2f((bf16_t)r[1]), bf2f((bf16_t)r[2]), bf2f((bf16_t)r[3])};
    else return r;
  };
  auto get = [&](auto (&to)[MAXV], auto* from) {
#pragma unroll
    for (int i = 0; i < MAXV; ++i) to[i] = *reinterpret_cast<const std::remove_reference_t<decltype(to[0])>*>(from + 4 * min((int)threadIdx.x + 256 * i, nv - 1));
  };
  get(v, x + row * W);
  if (a) get(ra, a + row * as);
  if (b) get(rb, b + row * bs);
  constexpr bool kAll = MAXV <= 4;   // (more registers than the waves behind each other can spare otherwise)
  if (kAll && e) get(ev, e + row * W);
  if (kAll && a && ab) get(abv, ab);
  if (kAll && w) get(g, w);
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + 256 * i;
    floatx4 d = {0.f, 0.f, 0.f, 0.f};
    const int cc = 4 * min(c, nv - 1);
    if (a) d += wide(ra[i]);
    if (a && ab) d += kAll ? abv[i] : *reinterpret_cast<const floatx4*>(ab + cc);
    if (b) d += wide(rb[i]);
    v[i] += m * d;
    if (e) v[i] += kAll ? ev[i] : *reinterpret_cast<const floatx4*>(e + row * W + cc);
    if (c < nv) {
      if (!idx && (a || b || e)) *reinterpret_cast<floatx4*>(x + row * W + 4 * c) = v[i];
      ss += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
    }
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c < nv) {
      floatx4 gi = {1.f, 1.f, 1.f, 1.f};
      if (w) gi = (kAll ? g[i] : *reinterpret_cast<const floatx4*>(w + 4 * c)) + woff;
      const floatx4 r = v[i] * inv * gi;
      T* o = out + orow * os + 4 * c;
      if constexpr (sizeof(T) == 2) {
        short4_t q = {(short)f2bf(r[0]), (short)f2bf(r[1]), (short)f2bf(r[2]), (short)f2bf(r[3])};
        *reinterpret_cast<short4_t*>(o) = q;
      } else {
        *reinterpret_cast<floatx4*>(o) = r;
      }
    }
  }
}

// The stream's first rows and their norm: x f32 = token row (+ position row) * scale (kept twice with `copy`), out = the norm of it, as
// embed_pos_kernel / the embedding of stream_ln.hip and then the kernel above give them, to the bit.  W % 4 == 0, W <= 1024 MAXV, aligned
// rows.  A row was two launches, the first with a trip to memory for every 256 columns: 64 x 2,048 8.4 (with a copy that nobody read) + 4.3 ->
// 5.2 us, with positions 7.4 + 3.7 -> 7.0; 4,095 x 2,048 23.5 + 9.2 -> 18.2, with positions 20.7 + 9.0 -> 20.5.  positions: an id or position outside its table gives zeros and is counted; without, ids are clamped.
template <typename T, int MAXV>
__global__ __launch_bounds__(256) void embed_norm_kernel(const int* __restrict__ ids, const int* __restrict__ positions, const T* __restrict__ tok, long vocab,
                                                         const T* __restrict__ pos, int max_pos, float scale, float* __restrict__ x,
                                                         float* __restrict__ copy, const float* __restrict__ w, float woff, float eps,
                                                         T* __restrict__ out, int W) {
  using Raw = std::conditional_t<sizeof(T) == 2, short4_t, floatx4>;
  __shared__ float red[4];
  const long row = blockIdx.x;
  const int id = ids[row], ps = positions ? positions[row] : 0, nv = W >> 2;
  const bool ok = !positions || (id >= 0 && id < vocab && ps >= 0 && ps < max_pos);
  if (!ok && threadIdx.x == 0) atomicAdd(&g_stream_embed_errors, 1);
  const T* tr = tok + min(max((long)id, 0L), vocab - 1) * W;
  const T* pr = positions ? pos + (long)min(max(ps, 0), max_pos - 1) * W : nullptr;
  auto wide = [](Raw r) -> floatx4 {
    if constexpr (sizeof(T) == 2) return floatx4{bf2f((bf16_t)r[0]), bf2f((bf16_t)r[1]), bf2f((bf16_t)r[2]), bf2f((bf16_t)r[3])};
    else return r;
  };
  floatx4 v[MAXV], g[MAXV];
  Raw rt[MAXV], rp[MAXV];
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = 4 * min((int)threadIdx.x + 256 * i, nv - 1);
    rt[i] = *reinterpret_cast<const Raw*>(tr + c);
    if (positions) rp[i] = *reinterpret_cast<const Raw*>(pr + c);
    g[i] = *reinterpret_cast<const floatx4*>(w + c);
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + 256 * i;
    v[i] = positions ? wide(rt[i]) + wide(rp[i]) : wide(rt[i]) * scale;
    if (!ok) v[i] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (c < nv) {
      *reinterpret_cast<floatx4*>(x + row * W + 4 * c) = v[i];
      if (copy) *reinterpret_cast<floatx4*>(copy + row * W + 4 * c) = v[i];
      ss += v[i][0] * v[i][0] + v[i][1] * v[i][1] + v[i][2] * v[i][2] + v[i][3] * v[i][3];
    }
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c >= nv) continue;
    const floatx4 r = v[i] * inv * (g[i] + woff);
    if constexpr (sizeof(T) == 2) {
      const short4_t q = {(short)f2bf(r[0]), (short)f2bf(r[1]), (short)f2bf(r[2]), (short)f2bf(r[3])};
      *reinterpret_cast<short4_t*>(out + row * W + 4 * c) = q;
    } else {
      *reinterpret_cast<floatx4*>(out + row * W + 4 * c) = r;
    }
  }
}

// The same where a and b are products that come as f32 parts [n, rows, W] (s1 of them a's): each is summed and rounded as the product
// itself would be.  W % 4 == 0, W <= 1024 MAXV; SP >= n parts are requested together.
template <int MAXV, int SP>
__global__ __launch_bounds__(256) void stream_rmsnorm_sums_kernel(float* __restrict__ x, const float* __restrict__ parts, int s1, int n, long plane,
                                                                  const float* __restrict__ ab, const float* __restrict__ e, float m,
                                                                  const float* __restrict__ w, float woff, float eps,
                                                                  const long* __restrict__ idx, bf16_t* __restrict__ out, long os, int W) {
  // (weights in a larger tensor may lie anywhere)
  const bool vec = ((reinterpret_cast<uintptr_t>(ab) | reinterpret_cast<uintptr_t>(w)) & 15) == 0;
  auto ldf4 = [&](const float* p) { return vec ? *reinterpret_cast<const floatx4*>(p) : floatx4{p[0], p[1], p[2], p[3]}; };
  __shared__ float red[4];
  const long orow = blockIdx.x, row = idx ? idx[orow] : orow;
  const int nv = W >> 2;
  floatx4 v[MAXV];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c < nv) {
      floatx4 p[SP], s[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
#pragma unroll
      for (int k = 0; k < SP; ++k) p[k] = *reinterpret_cast<const floatx4*>(parts + min(k, n - 1) * plane + row * W + 4 * c);
      floatx4 t = *reinterpret_cast<const floatx4*>(x + row * W + 4 * c), d;
      const floatx4 z = {0.f, 0.f, 0.f, 0.f};
      const floatx4 bias = ab ? ldf4(ab + 4 * c) : z;
      const floatx4 again = e ? *reinterpret_cast<const floatx4*>(e + row * W + 4 * c) : z;
#pragma unroll
      for (int k = 0; k < SP; ++k) {
        if (k < s1) s[0] += p[k];
        else if (k < n) s[1] += p[k];
      }
#pragma unroll
      for (int j = 0; j < 4; ++j) d[j] = (bf2f(f2bf(s[0][j])) + bias[j]) + bf2f(f2bf(s[1][j]));
      t += m * d;
      if (e) t += again;
      if (!idx) *reinterpret_cast<floatx4*>(x + row * W + 4 * c) = t;
      v[i] = t;
      ss += t[0] * t[0] + t[1] * t[1] + t[2] * t[2] + t[3] * t[3];
    }
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int i = 0; i < MAXV; ++i) {
    const int c = threadIdx.x + 256 * i;
    if (c < nv) {
      floatx4 g = {1.f, 1.f, 1.f, 1.f};
      if (w) g = ldf4(w + 4 * c) + woff;
      const floatx4 r = v[i] * inv * g;
      *reinterpret_cast<uint2*>(out + orow * os + 4 * c) = make_uint2(pack_bf2(r[0], r[1]), pack_bf2(r[2], r[3]));
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softcap_kernel(const T* __restrict__ in, long is, float cap, float* __restrict__ out,
                                                      long os, int V) {
  const long row = blockIdx.x;
  for (int c = blockIdx.y * 256 + threadIdx.x; c < V; c += 256 * gridDim.y) {
    const float z = ldv<T>(in + row * is + c);
    out[row * os + c] = cap > 0.f ? cap * tanhf(z / cap) : z;
  }
}

// out[r][c] = silu(x[r][c]) * x[r][I + c] for f32 rows [gate | up] (the bf16 case is the GEMM's epilogue)
__global__ __launch_bounds__(256) void silu_mul_f32_kernel(const float* __restrict__ x, long xs, float* __restrict__ out,
                                                           long os, int I) {
  const long row = blockIdx.x;
  for (int c = blockIdx.y * 256 + threadIdx.x; c < I; c += 256 * gridDim.y) {
    const float g = x[row * xs + c];
    out[row * os + c] = g / (1.f + expf(-g)) * x[row * xs + I + c];
  }
}

}  // namespace

int lk_silu_mul_f32(const float* x, long xs, float* out, long os, long rows, int I, hipStream_t st) {
  if (rows <= 0) return 0;
  silu_mul_f32_kernel<<<dim3((unsigned)rows, (unsigned)((I + 2047) / 2048)), 256, 0, st>>>(x, xs, out, os, I);
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_stream_embed_errors() {
  int v = 0;
  if (hipMemcpyFromSymbol(&v, HIP_SYMBOL(g_stream_embed_errors), sizeof(int)) != hipSuccess) return -1;
  return v;
}

int lk_embed_pos(const int* ids, const int* positions, const void* tok, int vocab, const void* pos, int max_pos, long rows,
                 int W, float* x, float* copy, int esz, hipStream_t st) {
  if (rows <= 0) return 0;
  if (esz == 2)
    embed_pos_kernel<bf16_t><<<(unsigned)rows, 256, 0, st>>>(ids, positions, (const bf16_t*)tok, vocab, (const bf16_t*)pos,
                                                             max_pos, W, x, copy);
  else
    embed_pos_kernel<float><<<(unsigned)rows, 256, 0, st>>>(ids, positions, (const float*)tok, vocab, (const float*)pos,
                                                            max_pos, W, x, copy);
  LK_CHECK_LAUNCH();
  return 0;
}

// 0: done, 1: not for these sizes or addresses (two launches then)
int lk_embed_norm(const int* ids, const int* positions, const void* tok, long vocab, const void* pos, int max_pos, float scale, long rows, int W,
                  float* x, float* copy, const float* w, float woff, float eps, void* out, int esz, hipStream_t st) {
  const auto al = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (W <= 0 || W % 4 || W > 4096 || vocab <= 0 || (positions && max_pos <= 0) || !al(tok) || !al(pos) || !al(w) || !al(x) || !al(copy) || !al(out)) return 1;
  if (rows <= 0) return 0;
#define LK_EN(T, V) embed_norm_kernel<T, V><<<(unsigned)rows, 256, 0, st>>>(ids, positions, (const T*)tok, vocab, (const T*)pos, max_pos, scale, x, copy, w, woff, eps, (T*)out, W)
#define LK_ENS(T)                 \
  do {                            \
    if (W <= 1024) LK_EN(T, 1);   \
    else if (W <= 2048) LK_EN(T, 2); \
    else LK_EN(T, 4);             \
  } while (0)
  if (esz == 2) LK_ENS(bf16_t);
  else LK_ENS(float);
#undef LK_ENS
#undef LK_EN
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_stream_rmsnorm(float* x, const void* a, long as, const float* a_bias, const void* b, long bs, const float* e, float m, const float* w,
                      float woff, float eps, const long* idx, long out_rows, void* out, long os, int W, int esz,
                      hipStream_t st) {
  if (out_rows <= 0 || W <= 0) return 0;   // (rows of no columns: nothing to read in the place of columns past the last)
  const auto al = [](const void* p, long stride_bytes, int vec_bytes) {
    return p == nullptr || (reinterpret_cast<uintptr_t>(p) % vec_bytes == 0 && stride_bytes % vec_bytes == 0);
  };
  constexpr int kMaxV = 8;
  const int tv = esz == 2 ? 8 : 16;  // bytes of a 4-element access to the activations
  if (W % 4 == 0 && W <= 4 * 256 * kMaxV && al(x, (long)W * 4, 16) && al(e, (long)W * 4, 16) && al(w, 0, 16) && al(a_bias, 0, 16) &&
      al(a, as * (long)esz, tv) && al(b, bs * (long)esz, tv) && al(out, os * (long)esz, tv)) {
#define LK_VEC(T, V)                                                                                                                  \
  stream_rmsnorm_vec_kernel<T, V><<<(unsigned)out_rows, 256, 0, st>>>(x, (const T*)a, as, a_bias, (const T*)b, bs, e, m, w, woff, eps, \
                                                                      idx, (T*)out, os, W)
#define LK_VECS(T)                      \
  do {                                  \
    if (W <= 1024) LK_VEC(T, 1);        \
    else if (W <= 2048) LK_VEC(T, 2);   \
    else if (W <= 4096) LK_VEC(T, 4);   \
    else LK_VEC(T, kMaxV);              \
  } while (0)
    if (esz == 2) LK_VECS(bf16_t);
    else LK_VECS(float);
#undef LK_VECS
#undef LK_VEC
    LK_CHECK_LAUNCH();
    return 0;
  }
  if (esz == 2)
    stream_rmsnorm_kernel<bf16_t><<<(unsigned)out_rows, 256, 0, st>>>(x, (const bf16_t*)a, as, a_bias, (const bf16_t*)b, bs, e, m, w,
                                                                      woff, eps, idx, (bf16_t*)out, os, W);
  else
    stream_rmsnorm_kernel<float><<<(unsigned)out_rows, 256, 0, st>>>(x, (const float*)a, as, a_bias, (const float*)b, bs, e, m, w,
                                                                     woff, eps, idx, (float*)out, os, W);
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_stream_rmsnorm_sums(float* x, const float* parts, int s1, int n, long rows, const float* a_bias, const float* e, float m, const float* w,
                           float woff, float eps, const long* idx, long out_rows, void* out, long os, int W, hipStream_t st) {
  if (out_rows <= 0) return 0;
  const auto a16 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
  if (W < 4 || W % 4 || W > 8192 || n < 2 || n > kMaxSums || s1 < 1 || s1 >= n || !a16(x) || !a16(parts) || !a16(e) ||
      os % 4 || reinterpret_cast<uintptr_t>(out) % 8)
    return -1;
#define LK_SUMS(MAXV, SP)                                                                                                                \
  stream_rmsnorm_sums_kernel<MAXV, SP><<<(unsigned)out_rows, 256, 0, st>>>(x, parts, s1, n, rows * W, a_bias, e, m, w, woff, eps, idx, \
                                                                           (bf16_t*)out, os, W)
  if (W <= 2048 && n <= 8) LK_SUMS(2, 8);
  else if (W <= 2048) LK_SUMS(2, 16);
  else if (n <= 8) LK_SUMS(8, 8);
  else LK_SUMS(8, 16);
#undef LK_SUMS
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_softcap(const void* in, long is, float cap, float* out, long os, long rows, int V, int esz, hipStream_t st) {
  if (rows <= 0) return 0;
  dim3 grid((unsigned)rows, (unsigned)((V + 2047) / 2048));
  if (esz == 2) softcap_kernel<bf16_t><<<grid, 256, 0, st>>>((const bf16_t*)in, is, cap, out, os, V);
  else softcap_kernel<float><<<grid, 256, 0, st>>>((const float*)in, is, cap, out, os, V);
  LK_CHECK_LAUNCH();
  return 0;
}
