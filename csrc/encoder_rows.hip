// Encoder layer, few rows: the layer norm and the attention as prologues of the projections behind them.
//
// What bounds a short text's pass is the chain of launches and of memory latencies in each, not its bytes: 88 launches, 24 of them
// norms of 19 rows and 12 attentions of 12 workgroups.  Both read little, so every workgroup of the following product can afford to
// compute all of it again from L2 while its weight rows are on their way:
//   * ln_rows_kernel:   h = LN(s) for the workgroup's rows in LDS, in the order that the fragment reads want, then
//     Y = act(h W^T + b).  Each row of h is stored by one of the workgroups (it is the next residual).  Row tiles of 64; up to 32 rows two
//     tiles of half the rows and 32 columns: a workgroup's norms are arithmetic of 12 waves on 4 SIMDs (1.3 - 1.9 us of 4.6 with all 19 rows,
//     24 rows at once, between 2.2 us of loads and 0.9 of sums and stores), and half of them half as much.
//   * attn_rows_kernel: bidirectional attention of ONE text of up to 32 tokens and heads of 64, then Y = bf16(A W^T + b) + R.  A
//     wave computes one head: S^T = K Q^T leaves each lane four adjacent keys of one query, O^T = V^T P^T takes them as they are
//     (its K order is permuted alike on both sides), and O^T, rounded to bf16 as the attention alone stores it, is the product's X
//     fragment of the head's 64 columns in registers (W is read from LDS in the same permuted order).
// Measured in a pass (19 tokens): launches apart 314 us, fused 295, with two tiles of half the rows 275 (behind a pass over 512 MB 357 -> 300);
// of a launch's 5.6 us 1.5 are the gap before it, 2.2 its first loads.
// One wave per 64 columns of K in both: every load of a workgroup is requested at its start, so a launch waits for memory once.
// The arithmetic and the roundings are those of layernorm_kernel, of flash_prefill (f32 scores and sums, P and A in bf16) and
// of rows_gemm_kernel.
#include "common.h"
#include "kernels.h"
#include "row_ring.h"

namespace {

constexpr int kErRows = 64;      // rows of a workgroup
// Beyond this many rows and up to 32: two tiles of half the rows.  12 layers of 768 (384), cold weights, 8 / 9 / 16 / 19 / 24 / 32 tokens, one tile ->
// two: 250 / 256 / 275 / 295 / 304 / 333 (194 / 199 / 219 / 230 / 246 / 259) -> 255 / 256 / 273 / 271 / 281 / 296 (197 / 197 / 208 / 210 / 216 / 233) us
constexpr int kErHalve = 8;
constexpr int kErWaves = 12;     // 64 columns of K each: a 64-row tile of h and the weight rows in 160 KB

enum { ER_BIAS = 2, ER_GELU = 3, ER_ADD = 5 };

// 16 NT weight rows x this wave's 64 columns
template <int NT = 1>
LK_DEVICE void er_load_w(const bf16_t* W, int n0, int K, int wave, unsigned char* wl) {
  const int lane = threadIdx.x & 63;
  const bf16_t* w = W + (long)(n0 + (lane >> 3)) * K + wave * 64 + rg_lane_col(lane);
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) __builtin_amdgcn_global_load_lds((rg_gptr)(w + (long)i * 8 * K), (rg_lptr)(wl + i * 1024), 16, 0, 2);
}

// The waves' partial tiles through LDS: wave m, m + waves, .. gets tile row m from total(m, sum)
template <int MT, typename F>
LK_DEVICE void er_sums(unsigned char* smem, const floatx4 (&acc)[MT], int wave, int waves, F total) {
  const int lane = threadIdx.x & 63;
  __syncthreads();
  floatx4* part = reinterpret_cast<floatx4*>(smem);
#pragma unroll
  for (int m = 0; m < MT; ++m) part[(wave * MT + m) * 64 + lane] = acc[m];
  __syncthreads();
  for (int m = wave; m < MT; m += waves) {
    floatx4 t = part[m * 64 + lane];
    for (int w = 1; w < waves; ++w) t += part[(w * MT + m) * 64 + lane];
    total(m, t);
  }
}

// the sum over the lane's 32
LK_DEVICE float half_sum(float v) {
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(q[0]) + __uint_as_float(q[1]);
  v += wave_partner<8>(v);
  v += wave_partner<4>(v);
  v += wave_partner<2>(v);
  return v + wave_partner<1>(v);
}

// 4 columns of one row: bias, one rounding; GELU before it, or the residual r and a second rounding behind it
template <int EPI>
LK_DEVICE void er_store(bf16_t* y, const bf16_t* b, const bf16_t* r, floatx4 t) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    t[j] += bf2f(b[j]);
    if constexpr (EPI == ER_GELU) t[j] = lk_gelu_erf(t[j]);
    if constexpr (EPI == ER_ADD) t[j] = bf2f(f2bf(t[j])) + bf2f(r[j]);
  }
  uint2 pk;
  pk.x = pack_bf2(t[0], t[1]);
  pk.y = pack_bf2(t[2], t[3]);
  *reinterpret_cast<uint2*>(y) = pk;
}

// grid (N / (16 NT), tiles of `rows` rows), K / 64 waves; LDS: the tile of s, then of h: K / 64 pieces of [16 MT rows][128 bytes]; the weight rows
template <int MT, int NT, int EPI>
__global__ __launch_bounds__(64 * kErWaves, 1) void ln_rows_kernel(const bf16_t* __restrict__ S, long ss, const bf16_t* __restrict__ lw,
                                                                   const bf16_t* __restrict__ lb, float eps, bf16_t* __restrict__ H,
                                                                   const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias,
                                                                   bf16_t* __restrict__ Y, int M, int N, int K, int rows) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), waves = K / 64;
  const int n0 = blockIdx.x * (16 * NT), m0 = blockIdx.y * rows;
  M = min(M - m0, rows);
  S += (long)m0 * ss;
  H += (long)m0 * K;
  Y += (long)m0 * N;
  unsigned char* wl = smem + (long)waves * MT * 2048 + wave * (NT * 2048);
  unsigned char* sl = smem + (long)wave * MT * 2048;
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i)   // rows past M repeat the last one
    __builtin_amdgcn_global_load_lds((rg_gptr)(S + (long)min(8 * i + (lane >> 3), M - 1) * ss + wave * 64 + rg_lane_col(lane)),
                                     (rg_lptr)(sl + i * 1024), 16, 0, 0);
  er_load_w<NT>(W, n0, K, wave, wl);

  // Half a wave per row; lane l holds the row's 16-byte chunks l, l + 32, l + 64 (K <= 768: 96).  The loop stays rolled: unrolled over
  // the rows it is 12 KB of code that a launch runs once, and fetching that took longer than the arithmetic.
  constexpr int C = kErWaves * 8 / 32;
  const int nvec = K >> 3, l32 = lane & 31;
  uint4_t g[C], be[C];
#pragma unroll
  for (int i = 0; i < C; ++i)
    if (l32 + 32 * i < nvec) {
      g[i] = *reinterpret_cast<const uint4_t*>(lw + (l32 + 32 * i) * 8);
      be[i] = *reinterpret_cast<const uint4_t*>(lb + (l32 + 32 * i) * 8);
    }
  rg_wait<0>();
  __syncthreads();   // everyone's columns of s
#pragma unroll 1
  for (int row = 2 * wave + (lane >> 5); row < M; row += 2 * waves) {
    unsigned char* at[C];
    float v[C][8], s = 0.f, q = 0.f;
#pragma unroll
    for (int i = 0; i < C; ++i) {
      const int c = l32 + 32 * i;
      at[i] = smem + (long)((c >> 3) * (16 * MT) + row) * 128 + (((c & 7) ^ (row & 7)) << 4);
      uint4_t a = {0u, 0u, 0u, 0u};   // a chunk past the row's end counts as zeros
      if (c < nvec) a = *reinterpret_cast<const uint4_t*>(at[i]);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        s += v[i][2 * j] = __uint_as_float(a[j] << 16);
        s += v[i][2 * j + 1] = __uint_as_float(a[j] & 0xffff0000u);
      }
    }
    const float mean = half_sum(s) / (float)K;
#pragma unroll
    for (int i = 0; i < C; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[i][j] -= mean;
        if (l32 + 32 * i < nvec) q += v[i][j] * v[i][j];
      }
    const float inv = rsqrtf(half_sum(q) / (float)K + eps);
#pragma unroll
    for (int i = 0; i < C; ++i) {
      if (l32 + 32 * i >= nvec) continue;
      uint4_t y;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        y[j] = pack_bf2(v[i][2 * j] * inv * __uint_as_float(g[i][j] << 16) + __uint_as_float(be[i][j] << 16),
                        v[i][2 * j + 1] * inv * __uint_as_float(g[i][j] & 0xffff0000u) + __uint_as_float(be[i][j] & 0xffff0000u));
      *reinterpret_cast<uint4_t*>(at[i]) = y;
      if (row % (int)gridDim.x == (int)blockIdx.x) *reinterpret_cast<uint4_t*>(H + (long)row * K + (l32 + 32 * i) * 8) = y;
    }
  }
  __syncthreads();   // everyone's rows of h

  floatx4 acc[MT * NT];
#pragma unroll
  for (int m = 0; m < MT * NT; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int r16 = lane & 15, g4 = lane >> 4;
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = r16 * 128 + (((4 * h + g4) ^ (r16 & 7)) << 4);
    short8 b[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) b[n] = *reinterpret_cast<const short8*>(wl + n * 2048 + at);
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const short8 a = *reinterpret_cast<const short8*>(sl + m * 2048 + at);
#pragma unroll
      for (int n = 0; n < NT; ++n) acc[m * NT + n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[n], a, acc[m * NT + n], 0, 0, 0);
    }
  }
  er_sums<MT * NT>(smem, acc, wave, waves, [&](int i, floatx4 t) {
    const int row = i / NT * 16 + r16, col = n0 + i % NT * 16 + 4 * g4;
    if (row < M) er_store<EPI>(Y + (long)row * N + col, bias + col, nullptr, t);
  });
}

// grid (N / 16, tiles of `rows` queries), nh waves; QKV rows [q | k | v] of nh heads of 64 each; LDS: V [head][16 MT rows][128 bytes], the
// weight rows.  Texts of 9 - 32 tokens as two tiles of half the queries (beyond 16, MQ 1 of MT 2): the softmax and the products of all 19
// queries were 2.4 us of the workgroup's 4.6, and 48 workgroups leave CUs for as many more.
template <int MQ, int MT>
__global__ __launch_bounds__(64 * kErWaves, 1) void attn_rows_kernel(const bf16_t* __restrict__ QKV, long qs, int nh, float scale_log2,
                                                                     const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias,
                                                                     const bf16_t* __restrict__ R, long rs, bf16_t* __restrict__ Y, int M,
                                                                     int N, int rows) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  typedef __attribute__((address_space(3))) short4_t* s4_ptr;
  constexpr int KS = (MT + 1) / 2;   // steps of 32 keys
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int K = nh * 64, n0 = blockIdx.x * 16, q0 = blockIdx.y * rows, MR = min(M - q0, rows);
  R += (long)q0 * rs;
  Y += (long)q0 * N;
  unsigned char* vl = smem + (long)wave * MT * 2048;
  unsigned char* wl = smem + (long)nh * MT * 2048 + wave * 2048;
  // this head's q and k as fragments (16 rows x 64 bytes), V and W through LDS-DMA
  uint4_t qf[MQ][2], kf[MT][2];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const bf16_t *p = QKV + wave * 64 + 8 * g, *k = p + K + (long)min(16 * m + r16, M - 1) * qs;   // rows past the last repeat it
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (m < MQ) qf[m < MQ ? m : 0][s] = *reinterpret_cast<const uint4_t*>(p + (long)(q0 + min(16 * m + r16, MR - 1)) * qs + 32 * s);
      kf[m][s] = *reinterpret_cast<const uint4_t*>(k + 32 * s);
    }
  }
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i)
    __builtin_amdgcn_global_load_lds((rg_gptr)(QKV + (long)min(8 * i + (lane >> 3), M - 1) * qs + 2 * K + wave * 64 + rg_lane_col(lane)),
                                     (rg_lptr)(vl + i * 1024), 16, 0, 0);
  er_load_w(W, n0, K, wave, wl);

  short8 p[MQ][KS];
  float l[MQ];
#pragma unroll
  for (int m = 0; m < MQ; ++m) {   // 16 queries: column r16; keys 16 t + 4 g + j
    floatx4 s[MT];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < MT; ++t) {
      s[t] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int d = 0; d < 2; ++d)
        s[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(short8, kf[t][d]), __builtin_bit_cast(short8, qf[m][d]), s[t], 0, 0, 0);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if (16 * t + 4 * g + j >= M) s[t][j] = -INFINITY;
        mx = fmaxf(mx, s[t][j]);
      }
    }
    mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
    const float base = mx * scale_log2;
    float e[2 * KS][4], sum = 0.f;
#pragma unroll
    for (int t = 0; t < 2 * KS; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        e[t][j] = t < MT ? __builtin_amdgcn_exp2f(__builtin_fmaf(s[t < MT ? t : 0][j], scale_log2, -base)) : 0.f;
        sum += e[t][j];
      }
    sum += __shfl_xor(sum, 16, 64);
    sum += __shfl_xor(sum, 32, 64);
    l[m] = 1.f / sum;
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      uint4_t pk;
#pragma unroll
      for (int j = 0; j < 4; ++j) pk[j] = pack_bf2(e[2 * c + (j >> 1)][2 * (j & 1)], e[2 * c + (j >> 1)][2 * (j & 1) + 1]);
      p[m][c] = __builtin_bit_cast(short8, pk);
    }
  }
  rg_wait<0>();   // this wave's V and W
  __builtin_amdgcn_sched_barrier(0);
  // O^T tile n: dims 16 n + 4 g + j of query r16
  floatx4 o[4][MQ], acc[MQ];
#pragma unroll
  for (int n = 0; n < 4; ++n) {
#pragma unroll
    for (int m = 0; m < MQ; ++m) o[n][m] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int c = 0; c < KS; ++c) {
      const int r0 = 32 * c + 4 * g + (r16 >> 2), r1 = 2 * c + 1 < MT ? r0 + 16 : r0;   // (no second tile: P is zero there, V any row of the text)
      const int ch = 2 * n + ((r16 & 3) >> 1), half = (r16 & 1) * 8;
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s4_ptr)(vl + r0 * 128 + ((ch ^ (r0 & 7)) << 4) + half));
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((s4_ptr)(vl + r1 * 128 + ((ch ^ (r1 & 7)) << 4) + half));
      const short8 a = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
      for (int m = 0; m < MQ; ++m) o[n][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, p[m][c], o[n][m], 0, 0, 0);
    }
  }
  // the product's two steps of 32 columns of this head, columns in O^T's order: 32 s + 4 g + j, then 32 s + 16 + 4 g + j
#pragma unroll
  for (int m = 0; m < MQ; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const unsigned char* wr = wl + r16 * 128 + (g & 1) * 8;
    const short4_t lo = *reinterpret_cast<const short4_t*>(wr + (((4 * s + (g >> 1)) ^ (r16 & 7)) << 4));
    const short4_t hi = *reinterpret_cast<const short4_t*>(wr + (((4 * s + 2 + (g >> 1)) ^ (r16 & 7)) << 4));
    const short8 b = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
    for (int m = 0; m < MQ; ++m) {
      uint4_t a;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        a[j] = pack_bf2(o[2 * s + (j >> 1)][m][2 * (j & 1)] * l[m], o[2 * s + (j >> 1)][m][2 * (j & 1) + 1] * l[m]);
      acc[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, __builtin_bit_cast(short8, a), acc[m], 0, 0, 0);
    }
  }
  er_sums<MQ>(smem, acc, wave, nh, [&](int m, floatx4 t) {
    const int row = m * 16 + r16, col = n0 + 4 * g;
    if (row < MR) er_store<ER_ADD>(Y + (long)row * N + col, bias + col, R + (long)row * rs + col, t);
  });
}

constexpr int er_lds(int MT, int waves, int NT = 1) { return waves * (MT + NT) * 2048; }   // (the sums' MT NT KB per wave lie over it)

template <int MT, int NT, int EPI>
int launch_ln(int rows, const void* s, long ss, const void* lw, const void* lb, float eps, void* h, const void* w, const void* b, void* y, int M, int N,
              int K, hipStream_t st) {
  LK_SET_MAX_LDS((ln_rows_kernel<MT, NT, EPI>), er_lds(MT, kErWaves, NT));
  ln_rows_kernel<MT, NT, EPI><<<dim3(N / (16 * NT), (M + rows - 1) / rows), K, er_lds(MT, K / 64, NT), st>>>(
      (const bf16_t*)s, ss, (const bf16_t*)lw, (const bf16_t*)lb, eps, (bf16_t*)h, (const bf16_t*)w, (const bf16_t*)b, (bf16_t*)y, M, N, K, rows);
  LK_CHECK_LAUNCH();
  return 0;
}

template <int EPI>
int ln_by_rows(const void* s, long ss, const void* lw, const void* lb, float eps, void* h, const void* w, const void* b, void* y, int M, int N,
               int K, hipStream_t st) {
  if (M > kErHalve && M <= 32 && N % 32 == 0) return launch_ln<1, 2, EPI>((M + 1) / 2, s, ss, lw, lb, eps, h, w, b, y, M, N, K, st);
  if (M <= 16) return launch_ln<1, 1, EPI>(kErRows, s, ss, lw, lb, eps, h, w, b, y, M, N, K, st);
  if (M <= 32) return launch_ln<2, 1, EPI>(kErRows, s, ss, lw, lb, eps, h, w, b, y, M, N, K, st);
  if (M <= 48) return launch_ln<3, 1, EPI>(kErRows, s, ss, lw, lb, eps, h, w, b, y, M, N, K, st);
  return launch_ln<4, 1, EPI>(kErRows, s, ss, lw, lb, eps, h, w, b, y, M, N, K, st);
}

template <int MQ, int MT>
int launch_attn(int rows, const void* qkv, long qs, int nh, float scale_log2, const void* w, const void* b, const void* r, long rs, void* y, int M, int N,
                hipStream_t st) {
  LK_SET_MAX_LDS((attn_rows_kernel<MQ, MT>), er_lds(MT, kErWaves));
  attn_rows_kernel<MQ, MT><<<dim3(N / 16, (M + rows - 1) / rows), 64 * nh, er_lds(MT, nh), st>>>((const bf16_t*)qkv, qs, nh, scale_log2, (const bf16_t*)w, (const bf16_t*)b,
                                                                      (const bf16_t*)r, rs, (bf16_t*)y, M, N, rows);
  LK_CHECK_LAUNCH();
  return 0;
}

}  // namespace

bool lk_ln_rows_supported(int M, int N, int K) {
  return M >= 1 && M <= 4096 && K >= 64 && K <= 64 * kErWaves && K % 64 == 0 && N >= 16 && N % 16 == 0;
}

// h [M, K] = LN(s), y [M, N] = act(h w^T + b); act: 0 none, 1 GELU.  h and y are contiguous and overlap no input.
int lk_ln_rows(const void* s, long ss, const void* lw, const void* lb, float eps, void* h, const void* w, const void* b, void* y, int M, int N,
               int K, int gelu, hipStream_t st) {
  if (!lk_ln_rows_supported(M, N, K)) return -1;
  return gelu ? ln_by_rows<ER_GELU>(s, ss, lw, lb, eps, h, w, b, y, M, N, K, st)
              : ln_by_rows<ER_BIAS>(s, ss, lw, lb, eps, h, w, b, y, M, N, K, st);
}

// (64 tokens: every workgroup would fetch 300 KB of q, k and v; 12.2 us against 4.4 + 4 us of the two launches)
bool lk_attn_rows_supported(int M, int nh, int N) { return M >= 1 && M <= 32 && nh >= 1 && nh <= kErWaves && N >= 16 && N % 16 == 0; }

// y [M, N] = bf16(attention(qkv rows of one text) w^T + b) + r, heads of 64; r and y 8-byte aligned with rows of whole 8 bytes
int lk_attn_rows(const void* qkv, long qs, int nh, float scale, const void* w, const void* b, const void* r, long rs, void* y, int M, int N,
                 hipStream_t st) {
  if (!lk_attn_rows_supported(M, nh, N)) return -1;
  const float s2 = scale * 1.4426950408889634f;
  if (M <= 16) return launch_attn<1, 1>(M > kErHalve ? (M + 1) / 2 : 16, qkv, qs, nh, s2, w, b, r, rs, y, M, N, st);
  return launch_attn<1, 2>((M + 1) / 2, qkv, qs, nh, s2, w, b, r, rs, y, M, N, st);
}
