// Per-head products out[t, h, n] = sum_k w[h][n][k] x[t, h * xh + k] (bf16 or f32 rows and weights, f32 accumulation): the
// projections between a head's own space and a latent that all heads share.
//
// Computed transposed (A = weight rows, B = token rows), so a lane ends up with 4 adjacent output columns of one token: one 8- or
// 16-byte store.  Grids run over the heads fastest: rows lie a power of two apart, and neighbours that differ in the head spread over
// the memory channels and keep each XCD on a few heads' weights.
//
// Many rows: a workgroup owns 128 tokens x 128 columns of a head, its 4 waves 64 x 64 quarters; both operands of a 128-byte step of
// the contraction are fetched once per workgroup (the next step's under this step's products) and staged in LDS, rows padded to
// 144 bytes.  Few rows, and sizes the vector loads do not divide: head_linear_few_kernel.
//
// Rows that are attention queries over a cached latent also get their rotated part (RotTail): few rows in workgroups of the products'
// launch behind the columns' (they read nothing that it writes), many in a launch of its own.
#include "common.h"
#include "kernels.h"
#include "attn_frag.h"

namespace {

constexpr int kRotMax = 1024;   // rotated elements per head

// the 4 adjacent columns n .. n + 3 of a token's row
template <typename T>
LK_DEVICE void store4(T* row, int n, int N, int vst, const floatx4& v) {
  if (vst && n + 4 <= N) {
    if constexpr (sizeof(T) == 2) {
      short4_t b;
#pragma unroll
      for (int j = 0; j < 4; ++j) b[j] = (short)f2bf(v[j]);
      *reinterpret_cast<short4_t*>(row + n) = b;
    } else {
      *reinterpret_cast<floatx4*>(row + n) = v;
    }
  } else {
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (n + j < N) El<T>::st(row + n + j, v[j]);
  }
}

// The rotated part of an output row behind its rp columns: the rd elements of the token's input row behind a head's first dim, turned
// by position (pairs i and i + rd / 2, or neighbours), zeros up to RDP.
struct RotTail {
  int dim, rd, rp, RDP, adj;
  float mag;   // times cos and sin
  const float* freq;
  const int* positions;
};

// the pair d of one row and head, by its angle's cos and sin times the magnitude
template <typename T>
LK_DEVICE void rot_pair(const RotTail& p, const T* s, T* o, int d, float cs, float sn) {
  const int ia = p.adj ? 2 * d : d, ib = p.adj ? 2 * d + 1 : p.rd / 2 + d;
  const float a = El<T>::ld(s + ia), b = El<T>::ld(s + ib);
  El<T>::st(o + ia, a * cs - b * sn);
  El<T>::st(o + ib, b * cs + a * sn);
}

LK_DEVICE void rot_angle(const RotTail& p, long t, int d, float& cs, float& sn) {
  sincosf((float)p.positions[t] * p.freq[d], &sn, &cs);
  cs *= p.mag;
  sn *= p.mag;
}

// 16 rows of one head by one workgroup
template <typename T>
LK_DEVICE void rot_tail(const RotTail& p, const T* x, long xs, long xh, T* out, long os, long oh, int h, long t0, long rows) {
  const int half = p.rd / 2, n = half + p.RDP - p.rd;
  for (int i = threadIdx.x; i < 16 * n; i += 256) {
    const long t = t0 + i / n;
    const int d = i % n;
    if (t >= rows) return;
    T* o = out + t * os + h * oh + p.rp;
    if (d >= half) {
      El<T>::st(o + half + d, 0.f);
      continue;
    }
    float cs, sn;
    rot_angle(p, t, d, cs, sn);
    rot_pair<T>(p, x + t * xs + h * xh + p.dim, o, d, cs, sn);
  }
}

// Many rows: one workgroup per token, its angles once for all heads (with an angle per head in the products' launch, 4,096 rows of 16
// heads took 52 us with the products instead of 33.5 + 8.6).
template <typename T>
__global__ __launch_bounds__(256) void latent_rot_kernel(const T* __restrict__ x, long xs, long xh, T* __restrict__ out, long os, long oh, int H,
                                                         RotTail p) {
  __shared__ float cs[kRotMax / 2], sn[kRotMax / 2];
  const long t = blockIdx.x;
  const int half = p.rd / 2, n = half + p.RDP - p.rd;
  for (int i = threadIdx.x; i < half; i += 256) rot_angle(p, t, i, cs[i], sn[i]);
  __syncthreads();
  for (int i = threadIdx.x; i < H * n; i += 256) {
    const int h = i / n, d = i % n;
    T* o = out + t * os + (long)h * oh + p.rp;
    if (d >= half) El<T>::st(o + half + d, 0.f);
    else rot_pair<T>(p, x + t * xs + (long)h * xh + p.dim, o, d, cs[d], sn[d]);
  }
}

// PARTS 2: x holds K columns and K more that add to them (an operand in two bf16 parts), both times the same w; K in whole steps.
template <typename T, int PARTS>
__global__ __launch_bounds__(256) void head_linear_lds_kernel(const T* __restrict__ x, long xs, long xh, const T* __restrict__ w, int N, int K,
                                                              long rows, T* __restrict__ out, long os, long oh, int vst) {
  constexpr int EV = El<T>::V, KS = 8 * EV, TM = 128, TN = 128;
  __shared__ uint4_t sx[2][TM][9];
  __shared__ uint4_t sw[2][TN][9];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.x, c0 = blockIdx.y * TN;
  const long t0 = (long)blockIdx.z * TM;
  const int pr = tid >> 3, ps = tid & 7;   // this thread's pieces: rows pr + 32 i, segment ps
  const T* xp[4];
  const T* wp[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {   // rows behind the end read a valid row whose results are not stored
    xp[i] = x + min(t0 + pr + 32 * i, rows - 1) * xs + h * xh;
    wp[i] = w + ((long)h * N + min(c0 + pr + 32 * i, N - 1)) * K;
  }
  uint4_t rx[4], rw[4];
  auto fetch = [&](int kb) {
    const int k = kb + ps * EV, kw = PARTS == 2 && kb >= K ? k - K : k;
    const bool in = k < PARTS * K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      rx[i] = ld16(xp[i] + (in ? k : 0));
      rw[i] = ld16(wp[i] + (in ? kw : 0));
    }
  };
  auto stage = [&](int buf, int kb) {
    const bool in = kb + ps * EV < PARTS * K;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      sx[buf][pr + 32 * i][ps] = in ? rx[i] : uint4_t{0u, 0u, 0u, 0u};
      sw[buf][pr + 32 * i][ps] = in ? rw[i] : uint4_t{0u, 0u, 0u, 0u};
    }
  };
  const int wt = wv >> 1, wc = wv & 1;
  floatx4 acc[4][4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) acc[r][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  fetch(0);
  stage(0, 0);
  __syncthreads();
  int cur = 0;
  for (int kb = 0; kb < PARTS * K; kb += KS) {
    const bool more = kb + KS < PARTS * K;
    if (more) fetch(kb + KS);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      uint4_t a[4], b[4];
#pragma unroll
      for (int c = 0; c < 4; ++c) a[c] = sw[cur][64 * wc + 16 * c + n16][4 * u + g];
#pragma unroll
      for (int r = 0; r < 4; ++r) b[r] = sx[cur][64 * wt + 16 * r + n16][4 * u + g];
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int c = 0; c < 4; ++c) acc[r][c] = mma_qk<T>(a[c], b[r], acc[r][c]);
    }
    if (more) stage(cur ^ 1, kb + KS);
    __syncthreads();
    cur ^= 1;
  }
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const long t = t0 + 64 * wt + 16 * r + n16;
    if (t >= rows) continue;
#pragma unroll
    for (int c = 0; c < 4; ++c) store4<T>(out + t * os + h * oh, c0 + 64 * wc + 16 * c + 4 * g, N, vst, acc[r][c]);
  }
}

// Few rows: a workgroup owns 16 RT tokens x 32 columns of a head, its 4 waves a quarter of the contraction each (steps of 64 bytes in
// turn), up to 4 steps' fragments requested together straight from memory; the quarters meet in LDS.  At 64 rows the 2 MB of weights are
// a microsecond of bandwidth, so what counts is the chain of waits per wave: one for K 128, one for K 512 (bf16).  A wave over the whole
// contraction of 64 columns waited 8 times at K 512 and left 3 of 4 waves idle below 17 rows: 8.8 -> 5.5 us on average over
// K 128 -> 512 and K 512 -> 128 columns, 16 heads, the rotated part included.
template <typename T, int RT, int PARTS>
__global__ __launch_bounds__(256) void head_linear_few_kernel(const T* __restrict__ x, long xs, long xh, const T* __restrict__ w, int N, int K,
                                                              long rows, T* __restrict__ out, long os, long oh, int vec, int vst, int H, int ncol,
                                                              RotTail rot) {
  constexpr int EV = El<T>::V, STEP = 4 * EV, NT = 2, U = 4;
  static_assert(PARTS == 1 || sizeof(T) == 2, "f32 operands are whole");
  __shared__ floatx4 part[4][RT * NT][64];
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n16 = lane & 15, g = lane >> 4;
  const int h = blockIdx.x % H, cb = blockIdx.x / H, c0 = cb * 16 * NT;
  const long t0 = (long)blockIdx.z * 16 * RT;
  if (cb >= ncol) {   // the whole workgroup
    rot_tail<T>(rot, x, xs, xh, out, os, oh, h, t0 + 16 * (cb - ncol), rows);
    return;
  }
  const T* xr[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) xr[r] = x + min(t0 + 16 * r + n16, rows - 1) * xs + h * xh;
  const T* wr[NT];
#pragma unroll
  for (int c = 0; c < NT; ++c) wr[c] = w + ((long)h * N + min(c0 + 16 * c + n16, N - 1)) * K;
  floatx4 acc[RT][NT];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < NT; ++c) acc[r][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  // step i of this wave: elements (4 i + wv) STEP ..; groups of U whole steps as plain vector loads, then one at a time
  const int whole = vec ? K / STEP : 0, steps = (K + STEP - 1) / STEP;
  int s = wv;
  for (; s + 4 * (U - 1) < whole; s += 4 * U) {
    uint4_t a[U][NT], b[U][PARTS][RT];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int k = (s + 4 * u) * STEP + g * EV;
#pragma unroll
      for (int c = 0; c < NT; ++c) a[u][c] = ld16(wr[c] + k);
#pragma unroll
      for (int q = 0; q < PARTS; ++q)
#pragma unroll
        for (int r = 0; r < RT; ++r) b[u][q][r] = ld16(xr[r] + q * K + k);
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int q = 0; q < PARTS; ++q)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < NT; ++c) acc[r][c] = mma_qk<T>(a[u][c], b[u][q][r], acc[r][c]);
  }
  for (; s < steps; s += 4) {
    const int k = s * STEP + g * EV;
    uint4_t a[NT], b[RT];
#pragma unroll
    for (int c = 0; c < NT; ++c) a[c] = frag<T>(wr[c], k, K, vec);
#pragma unroll
    for (int q = 0; q < PARTS; ++q) {
#pragma unroll
      for (int r = 0; r < RT; ++r) b[r] = frag<T>(xr[r] + q * K, k, K, vec);
#pragma unroll
      for (int r = 0; r < RT; ++r)
#pragma unroll
        for (int c = 0; c < NT; ++c) acc[r][c] = mma_qk<T>(a[c], b[r], acc[r][c]);
    }
  }
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < NT; ++c) part[wv][r * NT + c][lane] = acc[r][c];
  __syncthreads();
  // tile i = (r, c): accumulator j of a lane is output column 16 c + 4 g + j of token 16 r + n16
  for (int i = wv; i < RT * NT; i += 4) {
    floatx4 v = part[0][i][lane];
#pragma unroll
    for (int q = 1; q < 4; ++q) {
      const floatx4 o = part[q][i][lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] += o[j];
    }
    const long t = t0 + 16 * (i / NT) + n16;
    if (t < rows) store4<T>(out + t * os + h * oh, c0 + 16 * (i % NT) + 4 * g, N, vst, v);
  }
}

int cu_count() {
  static const int cus = [] {
    int dev = 0, n = 256;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    return n;
  }();
  return cus;
}

template <typename T, int PARTS>
int head_linear_t(const void* x, long xs, long xh, const void* w, int H, int N, int K, long rows, void* out, long os, long oh, int vec, int vst,
                  const RotTail& rot, hipStream_t st) {
  if (N > 0 && rows > 65535L * 64) return -1;
  const bool fused = rot.RDP > 0 && N > 0 && rows <= 128;
  const int tail = fused ? 1 : 0;   // workgroups of 16 rows each behind the columns'
  // 16-row tiles of a workgroup: up to 4, fewer while that leaves no more than one workgroup per CU (a workgroup's rows come at the rate of
  // its CU; the weights, read once more per halving, out of L2).  16 heads of 128 columns on K 512 in two parts at 64 rows: 4, 2, 1 tiles 8.3,
  // 5.6, 4.7 us, at 128 rows 8.4, 5.7, 6.3; 32 heads at 128 rows (2 tiles: 512 workgroups) 8.8, 8.4, 10.0; in one part at 64 rows 6.0, 4.7, 4.1.
  int rt = rows <= 16 ? 1 : rows <= 32 ? 2 : 4;
  while (rt > 1 && (long)H * ((N + 31) / 32) * ((rows + 8 * rt - 1) / (8 * rt)) <= cu_count()) rt /= 2;
#define LK_HEAD(RT)                                                                                                                          \
  head_linear_few_kernel<T, RT, PARTS><<<dim3((unsigned)((long)H * ((N + 31) / 32 + tail * RT)), 1, (unsigned)((rows + 16 * RT - 1) / (16 * RT))),  \
                                  256, 0, st>>>((const T*)x, xs, xh, (const T*)w, N, K, rows, (T*)out, os, oh, vec, vst, H, (N + 31) / 32, rot)
  if (N == 0)
    ;
  else if (rows > 128 && vec && (PARTS == 1 || K % 64 == 0))
    head_linear_lds_kernel<T, PARTS><<<dim3((unsigned)H, (unsigned)((N + 127) / 128), (unsigned)((rows + 127) / 128)), 256, 0, st>>>(
        (const T*)x, xs, xh, (const T*)w, N, K, rows, (T*)out, os, oh, vst);
  else if (rt == 1)
    LK_HEAD(1);
  else if (rt == 2)
    LK_HEAD(2);
  else
    LK_HEAD(4);
#undef LK_HEAD
  LK_CHECK_LAUNCH();
  if (rot.RDP > 0 && !fused) {
    latent_rot_kernel<T><<<(unsigned)rows, 256, 0, st>>>((const T*)x, xs, xh, (T*)out, os, oh, H, rot);
    LK_CHECK_LAUNCH();
  }
  return 0;
}

// N 0: the rotated part alone
int head_products(const void* x, long xs, long xh, const void* w, int H, int N, int K, long rows, void* out, long os, long oh, int qdim, int dim,
                  int rd, const float* freq, const int* positions, int rp, int RDP, int adj, float mag, int esz, hipStream_t st, int parts) {
  if (rows <= 0) return 0;
  if (H < 1 || H > 65535 || N < 0 || (N > 0 && K < 1) || (N + 63) / 64 > 65535 || (long)H * ((N + 31) / 32 + 4) > 2147483647L) return -1;
  if (rd < 0 || rd % 2 || rd > kRotMax || dim < 0 || dim + rd > qdim || rd > RDP || N > (RDP > 0 ? rp : N) || (rd > 0 && (!freq || !positions))) return -1;
  const int ev = 16 / esz;
  const auto a16 = [](const void* p, int b) { return reinterpret_cast<uintptr_t>(p) % b == 0; };
  const int vec = K % ev == 0 && xs % ev == 0 && xh % ev == 0 && a16(x, 16) && a16(w, 16);
  const int vst = os % 4 == 0 && oh % 4 == 0 && a16(out, 4 * esz);
  const RotTail rot{dim, rd, rp, RDP, adj, mag, freq, positions};
  if (esz != 2) return head_linear_t<float, 1>(x, xs, xh, w, H, N, K, rows, out, os, oh, vec, vst, rot, st);
  return parts == 2 ? head_linear_t<bf16_t, 2>(x, xs, xh, w, H, N, K, rows, out, os, oh, vec, vst, rot, st)
                    : head_linear_t<bf16_t, 1>(x, xs, xh, w, H, N, K, rows, out, os, oh, vec, vst, rot, st);
}

}  // namespace

int lk_head_linear(const void* x, long xs, long xh, const void* w, int H, int N, int K, long rows, void* out, long os, long oh, int esz,
                   hipStream_t st, int parts) {
  if (N < 1 || K < 1 || parts < 1 || parts > 2 || (parts == 2 && esz != 2)) return rows <= 0 ? 0 : -1;
  return head_products(x, xs, xh, w, H, N, K, rows, out, os, oh, 0, 0, 0, nullptr, nullptr, 0, 0, 0, 1.f, esz, st, parts);
}

int lk_latent_query(const void* x, long xs, long xh, const void* w, int H, int N, int K, long rows, void* out, long os, long oh, int qdim, int dim,
                    int rd, const float* freq, const int* positions, int rp, int RDP, int adj, float mag, int esz, hipStream_t st) {
  return head_products(x, xs, xh, w, H, N, K, rows, out, os, oh, qdim, dim, rd, freq, positions, rp, RDP, adj, mag, esz, st, 1);
}
