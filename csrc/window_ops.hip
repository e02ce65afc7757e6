// Kernels around windowed attention with pooled blocks and latent attention (bf16 or f32 activations;
// everything between the loads and the stores is f32):
//
//   lk_stream_gated_norm  x += rms(v) w_post,  v = mean_parts(y) * sigmoid(g + b);  out = rms(x) w_next
//   lk_rms_cols           out = rms(u[:, col0 : col0 + n]) w
//   lk_rot_kv_write       rotation of adjacent pairs by position * freq[i] (cos and sin times mag) on queries (in
//                         place) and keys; a key head = [per-head part | part shared by the heads | zeros];
//                         keys and values into the paged cache K [NB, G, BS, KD], V [NB, G, VD, BS]; the cached value may
//                         be a blend (1 - b) v + b v2 with a second set of value rows
//   lk_pool_kv_write      mean key / value of every block of P positions whose last position is new in this step,
//                         read from the cache (so it is the mean of what the cache holds) and filed at the block's
//                         index b, taken as a logical position of the sequence's block table, in a second pair
//
// rms(v) = v / sqrt(mean(v^2) + eps).
#include "common.h"
#include "kernels.h"
#include "kv_rows.h"

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

template <typename T, int V>
LK_DEVICE void ldn(const T* p, float (&f)[V]) {
  if constexpr (V == 4 && sizeof(T) == 4) {
    const floatx4 t = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = t[e];
  } else if constexpr (V == 4) {
    const short4_t t = *reinterpret_cast<const short4_t*>(p);
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = bf2f((bf16_t)t[e]);
  } else {
    f[0] = ldv<T>(p);
  }
}

template <typename T, int V>
LK_DEVICE void stn(T* p, const float (&f)[V]) {
  if constexpr (V == 4 && sizeof(T) == 4) {
    *reinterpret_cast<floatx4*>(p) = floatx4{f[0], f[1], f[2], f[3]};
  } else if constexpr (V == 4) {
    *reinterpret_cast<short4_t*>(p) = short4_t{(short)f2bf(f[0]), (short)f2bf(f[1]), (short)f2bf(f[2]), (short)f2bf(f[3])};
  } else {
    stv<T>(p, f[0]);
  }
}

// One workgroup per token; thread i owns the column groups i, i + 256, ... of V adjacent columns (MAXI groups at
// most) in registers through the three passes: gated value and its mean square, stream update and its mean
// square, normed copy.  V = 4: 16-byte f32 / 8-byte bf16 accesses (W % 4 == 0, aligned rows); V = 1 otherwise.
template <typename T, int MAXI, int V>
__global__ __launch_bounds__(256) void stream_gated_norm_kernel(float* __restrict__ x, const T* __restrict__ y, long ys, int parts,
                                                                const T* __restrict__ g, long gs, const float* __restrict__ gb,
                                                                const float* __restrict__ wpost, const float* __restrict__ wnext,
                                                                float eps, T* __restrict__ out, long os, int W) {
  __shared__ float red[4];
  const long row = blockIdx.x;
  const int ng = W / V;
  const float invp = 1.f / (float)parts;
  float v[MAXI][V];
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
    const int c = (threadIdx.x + 256 * i) * V;
    if (threadIdx.x + 256 * i < ng) {
      float a[V], t[V], gv[V], bv[V];
      ldn<T, V>(y + row * parts * ys + c, a);
      for (int p = 1; p < parts; ++p) {
        ldn<T, V>(y + (row * parts + p) * ys + c, t);
#pragma unroll
        for (int e = 0; e < V; ++e) a[e] += t[e];
      }
      ldn<T, V>(g + row * gs + c, gv);
      ldn<float, V>(gb + c, bv);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        const float val = parts > 1 ? a[e] * invp : a[e];
        v[i][e] = val / (1.f + expf(-(gv[e] + bv[e])));
        ss += v[i][e] * v[i][e];
      }
    }
  }
  ss = block_sum<4>(ss, red);
  const float inv1 = 1.f / sqrtf(ss / (float)W + eps);
  float s2 = 0.f;
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
    const int c = (threadIdx.x + 256 * i) * V;
    if (threadIdx.x + 256 * i < ng) {
      float xv[V], wv[V];
      ldn<float, V>(x + row * W + c, xv);
      ldn<float, V>(wpost + c, wv);
#pragma unroll
      for (int e = 0; e < V; ++e) {
        v[i][e] = xv[e] + v[i][e] * inv1 * wv[e];
        s2 += v[i][e] * v[i][e];
      }
      stn<float, V>(x + row * W + c, v[i]);
    }
  }
  if (!out) return;
  s2 = block_sum<4>(s2, red);
  const float inv2 = 1.f / sqrtf(s2 / (float)W + eps);
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
    const int c = (threadIdx.x + 256 * i) * V;
    if (threadIdx.x + 256 * i < ng) {
      float wv[V], r[V];
      ldn<float, V>(wnext + c, wv);
#pragma unroll
      for (int e = 0; e < V; ++e) r[e] = v[i][e] * inv2 * wv[e];
      stn<T, V>(out + row * os + c, r);
    }
  }
}

// The same for steps of few rows (bf16), whose time is the trips to memory behind each other: everything that a row reads is requested
// before anything waits (columns past the row are its last again, and not used).  With many rows the registers cost more waves than the trips.  CONV: the causal convolution over each sequence's rows
// that the next sublayer opens with (conv_silu_vec_kernel of csrc/ssm.hip with one token per sequence, without activation and bias; the
// normed row as it rounds is its input): its columns are this thread's, so only the weights and the state's rows come on top and a launch less.
struct GatedConv {
  const float* w;     // [W][taps]
  int taps;
  bf16_t* state;      // [slots][taps - 1][W]
  const int* slots;   // per row; < 0: zeros, and no state
  const int* positions;
  bf16_t* out;
  long os;
};
template <int MAXI, int PARTS, bool CONV>
__global__ __launch_bounds__(512) void gated_norm_row_kernel(float* __restrict__ x, const bf16_t* __restrict__ y, long ys,
                                                             const bf16_t* __restrict__ g, long gs, const float* __restrict__ gb,
                                                             const float* __restrict__ wpost, const float* __restrict__ wnext, float eps,
                                                             bf16_t* __restrict__ out, long os, int W, GatedConv cv) {
  __shared__ float red[8];
  const long row = blockIdx.x;
  const int ng = W / 4;
  int col[MAXI];
  bool on[MAXI];
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
    on[i] = (int)threadIdx.x + 512 * i < ng;
    col[i] = 4 * min((int)threadIdx.x + 512 * i, ng - 1);
  }
  short4_t yr[MAXI][PARTS], gr[MAXI], sr[MAXI][3];
  floatx4 bv[MAXI], xv[MAXI], wp[MAXI], wn[MAXI];
  float wk[MAXI][4][4];   // [tap, of four][column]
  int slot = -1, pos = 0;
  const bool w4 = CONV && cv.taps == 4 && (reinterpret_cast<uintptr_t>(cv.w) & 15) == 0;   // a column's taps in one 16-byte load
  if constexpr (CONV) slot = cv.slots[row], pos = cv.positions[row];
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
#pragma unroll
    for (int p = 0; p < PARTS; ++p) yr[i][p] = *reinterpret_cast<const short4_t*>(y + (row * PARTS + p) * ys + col[i]);
    gr[i] = *reinterpret_cast<const short4_t*>(g + row * gs + col[i]);
    bv[i] = *reinterpret_cast<const floatx4*>(gb + col[i]);
    xv[i] = *reinterpret_cast<const floatx4*>(x + row * W + col[i]);
    wp[i] = *reinterpret_cast<const floatx4*>(wpost + col[i]);
    if (out) wn[i] = *reinterpret_cast<const floatx4*>(wnext + col[i]);
    if constexpr (CONV) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (w4) {
          const floatx4 t = *reinterpret_cast<const floatx4*>(cv.w + (long)(col[i] + e) * 4);
#pragma unroll
          for (int k = 0; k < 4; ++k) wk[i][k][e] = t[k];
        } else {
#pragma unroll
          for (int k = 0; k < 4; ++k) wk[i][k][e] = k >= 4 - cv.taps ? cv.w[(long)(col[i] + e) * cv.taps + (k - (4 - cv.taps))] : 0.f;
        }
#pragma unroll
      for (int d = 0; d < 3; ++d) {   // the input 3 - d tokens ago: row taps - 4 + d of the state
        const int si = cv.taps - 4 + d;
        sr[i][d] = short4_t{0, 0, 0, 0};
        if (si >= 0 && slot >= 0) sr[i][d] = *reinterpret_cast<const short4_t*>(cv.state + ((long)slot * (cv.taps - 1) + si) * W + col[i]);
      }
    }
  }
  float ss = 0.f, s2 = 0.f;
  floatx4 v[MAXI];
#pragma unroll
  for (int i = 0; i < MAXI; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float a = bf2f((bf16_t)yr[i][0][e]);
#pragma unroll
      for (int p = 1; p < PARTS; ++p) a += bf2f((bf16_t)yr[i][p][e]);
      const float val = PARTS > 1 ? a * (1.f / (float)PARTS) : a;
      v[i][e] = val / (1.f + expf(-(bf2f((bf16_t)gr[i][e]) + bv[i][e])));
      if (on[i]) ss += v[i][e] * v[i][e];
    }
  ss = block_sum<8>(ss, red);
  const float inv1 = 1.f / sqrtf(ss / (float)W + eps);
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[i][e] = xv[i][e] + v[i][e] * inv1 * wp[i][e];
      if (on[i]) s2 += v[i][e] * v[i][e];
    }
    if (on[i]) *reinterpret_cast<floatx4*>(x + row * W + col[i]) = v[i];
  }
  if (!out) return;
  s2 = block_sum<8>(s2, red);
  const float inv2 = 1.f / sqrtf(s2 / (float)W + eps);
#pragma unroll
  for (int i = 0; i < MAXI; ++i) {
    if (!on[i]) continue;
    const floatx4 r = v[i] * inv2 * wn[i];
    const short4_t h = {(short)f2bf(r[0]), (short)f2bf(r[1]), (short)f2bf(r[2]), (short)f2bf(r[3])};
    *reinterpret_cast<short4_t*>(out + row * os + col[i]) = h;
    if constexpr (CONV) {
      short4_t c = {0, 0, 0, 0};
      if (slot >= 0) {
        if (pos <= 0) sr[i][0] = sr[i][1] = sr[i][2] = c;   // no past
#pragma unroll
        for (int e = 0; e < 4; ++e)
          c[e] = (short)f2bf(wk[i][0][e] * bf2f((bf16_t)sr[i][0][e]) + wk[i][1][e] * bf2f((bf16_t)sr[i][1][e]) + wk[i][2][e] * bf2f((bf16_t)sr[i][2][e]) +
                             wk[i][3][e] * bf2f((bf16_t)h[e]));
#pragma unroll
        for (int d = 0; d < 3; ++d) {
          const int si = cv.taps - 4 + d;
          if (si >= 0) *reinterpret_cast<short4_t*>(cv.state + ((long)slot * (cv.taps - 1) + si) * W + col[i]) = d < 2 ? sr[i][d < 2 ? d + 1 : 2] : h;
        }
      }
      *reinterpret_cast<short4_t*>(cv.out + row * cv.os + col[i]) = c;
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void rms_cols_kernel(const T* __restrict__ u, long us, int n, const float* __restrict__ w, float eps,
                                                       T* __restrict__ out, long os) {
  __shared__ float red[4];
  const long row = blockIdx.x;
  const T* src = u + row * us;
  float ss = 0.f;
  for (int c = threadIdx.x; c < n; c += 256) {
    const float v = ldv<T>(src + c);
    ss += v * v;
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)n + eps);
  for (int c = threadIdx.x; c < n; c += 256) stv<T>(out + row * os + c, ldv<T>(src + c) * inv * w[c]);
}

constexpr int kRotMaxHead = 256;

struct RotParams {
  void* q;
  long qs;
  int H, qdim;
  const void* k;
  long ks;
  int G, kdim;
  const void* sh;   // key part shared by the heads (null: none)
  long shs;
  int sdim;
  const void* v;
  long vs;
  int vdim;
  const void* v2;   // rows of G heads of vdim columns blended into v (null: none): cached = (1 - blend) v + blend v2
  long v2s;
  float blend;
  int rot_off, rot;  // dimensions [rot_off, rot_off + rot) of a query / key head are rotated in adjacent pairs
  const float* freq;
  float mag;
  const int* positions;
  void* kc;
  void* vc;
  const int* slots;
  int BS, KD, VD;
};

// One workgroup per token; its 4 waves take the H + 2 G (head, kind) jobs in turn.  The token's cos and sin
// (accurate sincosf of the f32 angle, times mag) are computed once per pair into LDS and shared by all heads.
// A head's elements and their rotation partners are in registers (up to 4 of each per lane) before anything is
// written, so the in-place q is safe.
template <typename T>
__global__ __launch_bounds__(256) void rot_kv_write_kernel(RotParams p) {
  __shared__ float scs[kRotMaxHead / 2], ssn[kRotMaxHead / 2];
  const long t = blockIdx.x;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int slot = p.slots[t];
  const float pos = (float)p.positions[t];
  for (int i = threadIdx.x; i < p.rot / 2; i += 256) {
    float sn, cs;
    sincosf(pos * p.freq[i], &sn, &cs);
    scs[i] = cs * p.mag;
    ssn[i] = sn * p.mag;
  }
  __syncthreads();
  const long blk = slot >= 0 ? slot / p.BS : 0;
  const int off = slot >= 0 ? slot % p.BS : 0;
  const T* krow = reinterpret_cast<const T*>(p.k) + t * p.ks;
  const T* shrow = p.sh ? reinterpret_cast<const T*>(p.sh) + t * p.shs : nullptr;
  for (int job = w; job < p.H + 2 * p.G; job += 4) {
    if (job < p.H + p.G) {
      const bool isq = job < p.H;
      if (!isq && slot < 0) continue;
      const int hd = isq ? p.qdim : p.KD;   // columns written
      const int kh = job - p.H;
      T* qrow = reinterpret_cast<T*>(p.q) + t * p.qs + (long)job * p.qdim;
      auto src = [&](int c) -> float {
        if (isq) return ldv<T>(qrow + c);
        if (c < p.kdim) return ldv<T>(krow + (long)kh * p.kdim + c);
        if (c < p.kdim + p.sdim) return ldv<T>(shrow + (c - p.kdim));
        return 0.f;
      };
      float own[4], par[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        own[i] = par[i] = 0.f;
        if (c < hd) {
          own[i] = src(c);
          const int r = c - p.rot_off;
          if (r >= 0 && r < p.rot) par[i] = src((r & 1) ? c - 1 : c + 1);
        }
      }
      T* dst = isq ? qrow : reinterpret_cast<T*>(p.kc) + ((blk * p.G + kh) * p.BS + off) * p.KD;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (c < hd) {
          float y = own[i];
          const int r = c - p.rot_off;
          if (r >= 0 && r < p.rot) {
            const float sn = ssn[r >> 1], cs = scs[r >> 1];
            y = (r & 1) ? own[i] * cs + par[i] * sn : own[i] * cs - par[i] * sn;
          }
          stv<T>(dst + c, y);
        }
      }
    } else if (slot >= 0) {
      const int gh = job - p.H - p.G;
      const T* x = reinterpret_cast<const T*>(p.v) + t * p.vs + (long)gh * p.vdim;
      const T* x2 = p.v2 ? reinterpret_cast<const T*>(p.v2) + t * p.v2s + (long)gh * p.vdim : nullptr;
      T* dst = reinterpret_cast<T*>(p.vc) + (blk * p.G + gh) * (long)p.VD * p.BS + off;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = lane + 64 * i;
        if (c < p.VD) {
          float val = c < p.vdim ? ldv<T>(x + c) : 0.f;
          if (x2 && c < p.vdim) val = (1.f - p.blend) * val + p.blend * ldv<T>(x2 + c);
          stv<T>(dst + (long)c * p.BS, val);
        }
      }
    }
  }
}

// The same for bf16 rows whose head sizes and strides are whole 16-byte pieces: R rows and a part of their heads per
// workgroup (kv_rows.h).  grid (rows / R, q / k parts + value parts).  4,096 rows of 16 query and 16 key heads of 192 with
// 16 x 128 values: 77 us with one workgroup per row (2-byte accesses, values in 64 sectors per store) -> 35 us; 64
// decode rows 20 -> 6.4 us.
template <int R, int LPH>
__global__ __launch_bounds__(256) void rot_file_kernel(RotParams p, long rows, int qk_parts) {
  using KT = KvTile<R, LPH>;
  constexpr int SV = R == 1 ? 1 : R;
  __shared__ float2 sct[R][kRotMaxHead / 2];
  __shared__ __attribute__((aligned(16))) bf16_t sv[SV][KT::VCOLS + 2];
  const long t0 = (long)blockIdx.x * R;
  const int tl = (int)min((long)R, rows - t0), part = blockIdx.y;
  if (part >= qk_parts) {
    const int n = p.G * p.VD, c0 = (part - qk_parts) * KT::VCOLS;
    kv_file_values<R, KT::VCOLS>(p.slots, t0, tl, c0, min(n, c0 + KT::VCOLS), p.G, p.VD, p.BS, reinterpret_cast<bf16_t*>(p.vc), sv,
                                 [&](long t, int gh, int d, float (&f)[8]) {
      if (d >= p.vdim) {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = 0.f;
        return;
      }
      load8(reinterpret_cast<const bf16_t*>(p.v) + t * p.vs + (long)gh * p.vdim + d, f);
      if (p.v2) {
        float f2[8];
        load8(reinterpret_cast<const bf16_t*>(p.v2) + t * p.v2s + (long)gh * p.vdim + d, f2);
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = (1.f - p.blend) * f[e] + p.blend * f2[e];
      }
    });
    return;
  }
  const int np = p.rot / 2;
  for (int i = threadIdx.x; i < tl * np; i += 256) {
    const int r = i / np, k = i % np;
    float sn, cs;
    sincosf((float)p.positions[t0 + r] * p.freq[k], &sn, &cs);
    sct[r][k] = make_float2(cs * p.mag, sn * p.mag);
  }
  __syncthreads();
  const int h0 = part * KT::HEADS, nh = min(KT::HEADS, p.H + p.G - h0);
  const int c = (threadIdx.x % LPH) * 8;
  for (int i = threadIdx.x / LPH; i < tl * nh; i += 256 / LPH) {
    const int r = i / nh, job = h0 + i % nh;
    const long t = t0 + r;
    const bool isq = job < p.H;
    const int kh = job - p.H, hd = isq ? p.qdim : p.KD, slot = isq ? 0 : p.slots[t];
    if (c >= hd || slot < 0) continue;
    bf16_t* dst;
    float f[8];
    if (isq) {
      dst = reinterpret_cast<bf16_t*>(p.q) + t * p.qs + (long)job * p.qdim + c;
      load8(dst, f);
    } else {
      dst = reinterpret_cast<bf16_t*>(p.kc) + (((long)(slot / p.BS) * p.G + kh) * p.BS + slot % p.BS) * p.KD + c;
      if (c < p.kdim) load8(reinterpret_cast<const bf16_t*>(p.k) + t * p.ks + (long)kh * p.kdim + c, f);
      else if (c < p.kdim + p.sdim) load8(reinterpret_cast<const bf16_t*>(p.sh) + t * p.shs + (c - p.kdim), f);
      else {
#pragma unroll
        for (int e = 0; e < 8; ++e) f[e] = 0.f;
      }
    }
#pragma unroll
    for (int e = 0; e < 8; e += 2) {
      const int k = c + e - p.rot_off;
      if (k >= 0 && k < p.rot) {
        const float2 cs = sct[r][k >> 1];
        const float a = f[e], b = f[e + 1];
        f[e] = a * cs.x - b * cs.y;
        f[e + 1] = b * cs.x + a * cs.y;
      }
    }
    store8(dst, f);
  }
}

template <int R, int LPH>
void launch_rot_file(const RotParams& p, long T, hipStream_t st) {
  using KT = KvTile<R, LPH>;
  const int qk = (p.H + p.G + KT::HEADS - 1) / KT::HEADS, vp = (p.G * p.VD + KT::VCOLS - 1) / KT::VCOLS;
  rot_file_kernel<R, LPH><<<dim3((unsigned)((T + R - 1) / R), qk + vp), 256, 0, st>>>(p, T, qk);
}

// grid (blocks a sequence may complete in this step, G, sequences).  Sequence s holds ctx cached tokens, the last
// qlen of them new: the blocks past / P .. ctx / P - 1 end on a new position.
template <typename T>
__global__ __launch_bounds__(256) void pool_kv_write_kernel(const T* __restrict__ kc, const T* __restrict__ vc, T* __restrict__ pkc,
                                                            T* __restrict__ pvc, int P, const int* __restrict__ bt, int bt_stride,
                                                            const int* __restrict__ ctx_lens, const int* __restrict__ cu_q,
                                                            const int* __restrict__ slots, int row0, int G, int BS, int dim,
                                                            int vdim) {
  const int s = blockIdx.z, g = blockIdx.y;
  const int first = cu_q ? cu_q[s] : s, qlen = cu_q ? cu_q[s + 1] - first : 1;
  if (qlen <= 0 || slots[row0 + first] < 0) return;
  const int ctx = ctx_lens[s], past = ctx - qlen;
  const int b = past / P + blockIdx.x;
  if (b >= ctx / P) return;
  const int* tb = bt + (long)s * bt_stride;
  const float invp = 1.f / (float)P;
  const long dblk = tb[b / BS];
  const int doff = b % BS;
  for (int d = threadIdx.x; d < dim + vdim; d += 256) {
    float acc = 0.f;
    if (d < dim) {
      for (int i = 0; i < P; ++i) {
        const int pos = b * P + i;
        acc += ldv<T>(kc + (((long)tb[pos / BS] * G + g) * BS + pos % BS) * dim + d);
      }
      stv<T>(pkc + ((dblk * G + g) * BS + doff) * dim + d, acc * invp);
    } else {
      const int dv = d - dim;
      for (int i = 0; i < P; ++i) {
        const int pos = b * P + i;
        acc += ldv<T>(vc + (((long)tb[pos / BS] * G + g) * vdim + dv) * BS + pos % BS);
      }
      stv<T>(pvc + ((dblk * G + g) * vdim + dv) * BS + doff, acc * invp);
    }
  }
}

// The same for bf16 rows in 16-byte pieces (dim, vdim, P and BS multiples of 8): grid.x alternates keys and values.  A thread sums pieces
// a whole workgroup apart, LDS joins them; before, a thread walked a column's P positions one after the other.  64 decode rows of
// which one ends a block of 64: 11.3 us -> 5 us; 4 prompts of 1,024 tokens 28 -> 6 us.
constexpr int kPoolSums = 8192;   // floats of partial sums in LDS

__global__ __launch_bounds__(256) void pool_kv_vec_kernel(const bf16_t* __restrict__ kc, const bf16_t* __restrict__ vc, bf16_t* __restrict__ pkc,
                                                          bf16_t* __restrict__ pvc, int P, const int* __restrict__ bt, int bt_stride,
                                                          const int* __restrict__ ctx_lens, const int* __restrict__ cu_q,
                                                          const int* __restrict__ slots, int row0, int G, int BS, int dim, int vdim) {
  __shared__ float part[kPoolSums];
  const int s = blockIdx.z, g = blockIdx.y;
  const int first = cu_q ? cu_q[s] : s, qlen = cu_q ? cu_q[s + 1] - first : 1;
  if (qlen <= 0 || slots[row0 + first] < 0) return;
  const int ctx = ctx_lens[s], past = ctx - qlen;
  const int b = past / P + (blockIdx.x >> 1);
  if (b >= ctx / P) return;
  const int* tb = bt + (long)s * bt_stride;
  const float invp = 1.f / (float)P;
  const long dblk = tb[b / BS];
  const int doff = b % BS;
  if ((blockIdx.x & 1) == 0) {
    // thread: the 8 dims of piece t % nk, positions t / nk, + R, ..
    const int nk = dim / 8, R = 256 / nk, t = threadIdx.x, r = t / nk, c = t - r * nk;
    float acc[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) acc[e] = 0.f;
    if (r < R) {
      for (int i = r; i < P; i += R) {
        const int pos = b * P + i;
        float f[8];
        load8(kc + (((long)tb[pos / BS] * G + g) * BS + pos % BS) * dim + 8 * c, f);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[e] += f[e];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) part[r * dim + 8 * c + e] = acc[e];
    }
    __syncthreads();
    for (int d = t; d < dim; d += 256) {
      float a = 0.f;
      for (int j = 0; j < R; ++j) a += part[j * dim + d];
      pkc[((dblk * G + g) * BS + doff) * dim + d] = f2bf(a * invp);
    }
  } else {
    // piece q: 8 positions of one value row, the pieces of a cache block in the order of their addresses
    const int cr = P % BS == 0 ? BS / 8 : 1, n = P / 8 * vdim;
    for (int q = threadIdx.x; q < n; q += 256) {
      const int j = q % cr, vd = q / cr % vdim, pos = b * P + (q / (cr * vdim) * cr + j) * 8;
      float f[8];
      load8(vc + (((long)tb[pos / BS] * G + g) * vdim + vd) * BS + pos % BS, f);
      part[q] = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
    }
    __syncthreads();
    for (int vd = threadIdx.x; vd < vdim; vd += 256) {
      float a = 0.f;
      for (int c = 0; c < P / 8; ++c) a += part[(c / cr * vdim + vd) * cr + c % cr];
      pvc[((dblk * G + g) * vdim + vd) * BS + doff] = f2bf(a * invp);
    }
  }
}

template <typename T>
int gated_norm_t(float* x, const void* y, long ys, int parts, const void* g, long gs, const float* gb, const float* wpost,
                 const float* wnext, float eps, void* out, long os, long rows, int W, bool vec, hipStream_t st) {
  const T* yp = reinterpret_cast<const T*>(y);
  const T* gp = reinterpret_cast<const T*>(g);
  T* op = reinterpret_cast<T*>(out);
  if (vec && W <= 4 * 256 * 8)
    stream_gated_norm_kernel<T, 8, 4><<<(unsigned)rows, 256, 0, st>>>(x, yp, ys, parts, gp, gs, gb, wpost, wnext, eps, op, os, W);
  else if (W <= 256 * 16)
    stream_gated_norm_kernel<T, 16, 1><<<(unsigned)rows, 256, 0, st>>>(x, yp, ys, parts, gp, gs, gb, wpost, wnext, eps, op, os, W);
  else
    return -1;
  LK_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// Whether a step of this many rows takes the row kernel.  us before / with it, 2,048 columns in two parts: 64 rows 4.3 / 3.1, 256 4.7 / 3.5, 512 5.3 / 4.7,
// 1,024 7.4 / 6.9, 2,048 12.2 / 12.4; 8,192 columns: 64 9.9 / 6.2, 1,024 23.3 / 22.3, 2,048 40.5 / 40.4.  Up to 1,024 columns, where half of the
// threads or more idle: 64 rows 3.4 / 3.0, 256 3.6 / 3.3, 512 4.1 / 4.3, 1,024 4.8 / 5.7.
bool lk_gated_norm_row(long rows, int W, int parts, int esz) {
  return esz == 2 && rows <= (W > 1024 ? 1024 : 256) && W % 4 == 0 && W >= 4 && W <= 4 * 512 * 4 && (parts == 1 || parts == 2);
}

int lk_stream_gated_norm(float* x, const void* y, long ys, int parts, const void* g, long gs, const float* gb, const float* wpost,
                         const float* wnext, float eps, void* out, long os, long rows, int W, int esz, hipStream_t st, const float* cw, int taps,
                         void* cstate, const int* slots, const int* positions, void* cout, long cos) {
  if (rows <= 0) return 0;
  if (parts < 1 || W < 1 || !y || !g || !gb || !wpost || (out && !wnext)) return -1;
  const auto al = [](const void* p, long stride_bytes, int vec_bytes) {
    return p == nullptr || (reinterpret_cast<uintptr_t>(p) % vec_bytes == 0 && stride_bytes % vec_bytes == 0);
  };
  const int tv = esz == 2 ? 8 : 16;
  const bool vec = W % 4 == 0 && al(x, (long)W * 4, 16) && al(gb, 0, 16) && al(wpost, 0, 16) && al(wnext, 0, 16) &&
                   al(y, ys * (long)esz, tv) && al(g, gs * (long)esz, tv) && al(out, os * (long)esz, tv);
  const bool conv = cout != nullptr;
  if (conv && (!out || !cw || !slots || !positions || taps < 1 || taps > 4 || (taps > 1 && !cstate) || !al(cstate, (long)W * 2, 8) ||
               !al(cout, cos * 2, 8)))
    return -1;
  if (vec && lk_gated_norm_row(rows, W, parts, esz)) {
    const GatedConv cv{cw, taps, (bf16_t*)cstate, slots, positions, (bf16_t*)cout, cos};
#define LK_ROW(I, P, C)                                                                                                                  \
  gated_norm_row_kernel<I, P, C><<<(unsigned)rows, 512, 0, st>>>(x, (const bf16_t*)y, ys, (const bf16_t*)g, gs, gb, wpost, wnext, eps,   \
                                                                 (bf16_t*)out, os, W, cv)
#define LK_ROWS(I)                                              \
  do {                                                          \
    if (parts == 1) { if (conv) LK_ROW(I, 1, true); else LK_ROW(I, 1, false); } \
    else { if (conv) LK_ROW(I, 2, true); else LK_ROW(I, 2, false); }       \
  } while (0)
    if (W <= 2048) LK_ROWS(1);
    else if (W <= 4096) LK_ROWS(2);
    else LK_ROWS(4);
#undef LK_ROWS
#undef LK_ROW
    LK_CHECK_LAUNCH();
    return 0;
  }
  if (conv) return -1;
  return esz == 2 ? gated_norm_t<bf16_t>(x, y, ys, parts, g, gs, gb, wpost, wnext, eps, out, os, rows, W, vec, st)
                  : gated_norm_t<float>(x, y, ys, parts, g, gs, gb, wpost, wnext, eps, out, os, rows, W, vec, st);
}

int lk_rms_cols(const void* u, long us, int n, const float* w, float eps, void* out, long os, long rows, int esz, hipStream_t st) {
  if (rows <= 0) return 0;
  if (n < 1 || !w) return -1;
  if (esz == 2) rms_cols_kernel<bf16_t><<<(unsigned)rows, 256, 0, st>>>((const bf16_t*)u, us, n, w, eps, (bf16_t*)out, os);
  else rms_cols_kernel<float><<<(unsigned)rows, 256, 0, st>>>((const float*)u, us, n, w, eps, (float*)out, os);
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_rot_kv_write(void* q, long qs, int H, int qdim, const void* k, long ks, int G, int kdim, const void* sh, long shs, int sdim,
                    const void* v, long vs, int vdim, int rot_off, int rot, const float* freq, float mag, const int* positions,
                    void* kc, void* vc, const int* slots, int BS, int KD, int VD, long T, const void* v2, long v2s, float blend, int esz,
                    hipStream_t st) {
  if (T <= 0) return 0;
  if (H < 1 || G < 1 || qdim < 1 || kdim < 0 || sdim < 0 || (sdim > 0 && !sh) || vdim < 1 || qdim > kRotMaxHead || KD > kRotMaxHead ||
      VD > kRotMaxHead || kdim + sdim > KD || kdim + sdim < 1 || vdim > VD || rot < 0 || rot % 2 || rot_off < 0 ||
      rot_off + rot > qdim || rot_off + rot > kdim + sdim || (rot > 0 && !freq) || BS < 1)
    return -1;
  RotParams p;
  p.q = q; p.qs = qs; p.H = H; p.qdim = qdim; p.k = k; p.ks = ks; p.G = G; p.kdim = kdim; p.sh = sdim > 0 ? sh : nullptr; p.shs = shs;
  p.sdim = sdim; p.v = v; p.vs = vs; p.vdim = vdim; p.rot_off = rot_off; p.rot = rot; p.freq = freq; p.mag = mag;
  p.positions = positions; p.kc = kc; p.vc = vc; p.slots = slots; p.BS = BS; p.KD = KD; p.VD = VD;
  p.v2 = v2; p.v2s = v2s; p.blend = blend;
  const auto rows16 = [](const void* x, long stride) { return !x || ((reinterpret_cast<uintptr_t>(x) & 15) == 0 && stride % 8 == 0); };
  if (esz == 2 && qdim % 8 == 0 && kdim % 8 == 0 && sdim % 8 == 0 && vdim % 8 == 0 && KD % 8 == 0 && VD % 8 == 0 && rot_off % 2 == 0 &&
      rows16(q, qs) && rows16(kdim > 0 ? k : nullptr, ks) && rows16(p.sh, shs) && rows16(v, vs) && rows16(v2, v2s) && rows16(kc, 0) &&
      (H + G) <= 32768 && (long)G * VD <= 1 << 24) {
    const int lph = kv_lanes(qdim > KD ? qdim : KD);
    const bool few = T < kFileFewRows;
    if (lph == 8) few ? launch_rot_file<1, 8>(p, T, st) : launch_rot_file<kFileRows, 8>(p, T, st);
    else if (lph == 16) few ? launch_rot_file<1, 16>(p, T, st) : launch_rot_file<kFileRows, 16>(p, T, st);
    else few ? launch_rot_file<1, 32>(p, T, st) : launch_rot_file<kFileRows, 32>(p, T, st);
  } else if (esz == 2) rot_kv_write_kernel<bf16_t><<<(unsigned)T, 256, 0, st>>>(p);
  else rot_kv_write_kernel<float><<<(unsigned)T, 256, 0, st>>>(p);
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_pool_kv_write(const void* kc, const void* vc, void* pkc, void* pvc, int P, const int* bt, int bt_stride, const int* ctx_lens,
                     const int* cu_q, const int* slots, int row0, int S, int max_len, int G, int BS, int dim, int vdim, int esz,
                     hipStream_t st) {
  if (S <= 0 || max_len <= 0) return 0;
  if (P < 1 || G < 1 || BS < 1 || dim < 1 || vdim < 1 || S > 65535 || G > 65535) return -1;
  // a run of max_len new positions ends at most (max_len + P - 1) / P blocks (+ 1 when it starts inside one)
  const dim3 grid((unsigned)((max_len + P - 1) / P + 1), (unsigned)G, (unsigned)S);
  const auto a16 = [](const void* x) { return reinterpret_cast<uintptr_t>(x) % 16 == 0; };
  if (esz == 2 && dim % 8 == 0 && vdim % 8 == 0 && P % 8 == 0 && BS % 8 == 0 && dim <= 2048 && (long)P / 8 * vdim <= kPoolSums &&
      a16(kc) && a16(vc))   // (the keys' partial sums, 256 / (dim / 8) rows of dim, are 2,048 floats at most)
    pool_kv_vec_kernel<<<dim3(2 * grid.x, grid.y, grid.z), 256, 0, st>>>((const bf16_t*)kc, (const bf16_t*)vc, (bf16_t*)pkc, (bf16_t*)pvc, P, bt,
                                                                        bt_stride, ctx_lens, cu_q, slots, row0, G, BS, dim, vdim);
  else if (esz == 2)
    pool_kv_write_kernel<bf16_t><<<grid, 256, 0, st>>>((const bf16_t*)kc, (const bf16_t*)vc, (bf16_t*)pkc, (bf16_t*)pvc, P, bt, bt_stride,
                                                       ctx_lens, cu_q, slots, row0, G, BS, dim, vdim);
  else
    pool_kv_write_kernel<float><<<grid, 256, 0, st>>>((const float*)kc, (const float*)vc, (float*)pkc, (float*)pvc, P, bt, bt_stride,
                                                      ctx_lens, cu_q, slots, row0, G, BS, dim, vdim);
  LK_CHECK_LAUNCH();
  return 0;
}
