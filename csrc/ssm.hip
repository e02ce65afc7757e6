// Mamba-2 style selective state-space mixer, token-parallel where it can be and sequential only
// along the recurrence:
//
//   u_t  = [z | x B C | dt]                       the input projection's row (bf16 or f32)
//   xBC  = silu(causal_conv(x B C) + b)           per channel, `taps` wide (act = 0: without the SiLU), the last column is the
//                                                 current token's; the taps - 1 inputs before a chunk
//                                                 come from the sequence's conv state
//   dt   = softplus(dt + dt_bias)                 f32, no clamp
//   S_t  = exp(-exp(A_log) dt) S_{t-1} + dt B_t x_t^T      S: [N, P] per head, f32, carried per sequence
//   y_t  = S_t^T C_t + D x_t                      f32
//   out  = groupRMS(y * silu(z)) * w              the gate comes before the norm
//
// A batch is a list of sequences (prefill chunks of any length, decode rows of length 1): rows
// [cu[s], cu[s+1]) belong to sequence s, whose state lives in slot slots[s] (< 0: a padding row,
// skipped) and starts from zero when its first row sits at position 0.
#include <algorithm>
#include "common.h"
#include "kernels.h"

namespace {

template <typename T>
LK_DEVICE float ldf(const T* p);
template <>
LK_DEVICE float ldf<bf16_t>(const bf16_t* p) { return bf2f(*p); }
template <>
LK_DEVICE float ldf<float>(const float* p) { return *p; }
template <typename T>
LK_DEVICE void stf(T* p, float v);
template <>
LK_DEVICE void stf<bf16_t>(bf16_t* p, float v) { *p = f2bf(v); }
template <>
LK_DEVICE void stf<float>(float* p, float v) { *p = v; }

constexpr int kMaxTaps = 8;
constexpr int kConvRows = 16;  // tokens per workgroup of the convolution (at most)

template <bool EXACT>
LK_DEVICE float silu_f(float x) {
  if constexpr (EXACT) return x / (1.f + expf(-x));
  else return x * __builtin_amdgcn_rcpf(1.f + __expf(-x));
}

// grid (sequence, token tile, channel block): out[row][c] = silu(sum_k w[c][k] in(i - (taps-1) + k) + b[c])
template <typename T>
__global__ __launch_bounds__(256) void conv_silu_kernel(const T* __restrict__ u, long us, int C, int taps,
                                                        const float* __restrict__ w, const float* __restrict__ bias,
                                                        const T* __restrict__ state, const int* __restrict__ cu,
                                                        const int* __restrict__ slots,
                                                        const int* __restrict__ positions, T* __restrict__ out,
                                                        long os, int act) {
  const int s = blockIdx.x, c = blockIdx.z * 256 + threadIdx.x;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  const int i0 = blockIdx.y * kConvRows;
  if (c >= C || i0 >= len) return;
  if (slot < 0) {
    for (int i = i0; i < min(len, i0 + kConvRows); ++i) stf<T>(out + (long)(row0 + i) * os + c, 0.f);
    return;
  }
  const bool past = positions[row0] > 0;
  const T* st = state + (long)slot * (taps - 1) * C + c;
  float wk[kMaxTaps];
#pragma unroll
  for (int k = 0; k < kMaxTaps; ++k) wk[k] = k < taps ? w[(long)c * taps + k] : 0.f;
  const float b = bias ? bias[c] : 0.f;
  for (int i = i0; i < min(len, i0 + kConvRows); ++i) {
    float acc = b;
#pragma unroll
    for (int k = 0; k < kMaxTaps; ++k) {
      if (k < taps) {
        const int idx = i - (taps - 1) + k;
        float v = 0.f;
        if (idx >= 0) v = ldf<T>(u + (long)(row0 + idx) * us + c);
        else if (past) v = ldf<T>(st + (long)(taps - 1 + idx) * C);
        acc += wk[k] * v;
      }
    }
    stf<T>(out + (long)(row0 + i) * os + c, act ? silu_f<sizeof(T) == 4>(acc) : acc);
  }
}

// The same for taps <= 4 with 16-byte accesses: a thread owns EV adjacent channels and walks its `rows`
// tokens with the three previous inputs in registers (weights right-aligned in a 4-tap window, the
// unused leading taps zero), so every input row is read once per tile instead of once per tap.
// Needs C % EV == 0 and 16-byte aligned rows of u, out and the state.  The sequence's first tile also leaves the channels' last inputs
// in the state (nobody else reads it), without a launch of its own.  GR: rows requested together, a group ahead of the one in use (1: steps of
// single tokens; 8 are level, 16 slower by half, from registers).  A thread's weights are 128 bytes from its neighbour's, so that loading them
// cost as much as 8 rows: a tile's come in one sweep and are turned round in LDS.  bf16 x 6,144 channels, before / now, us: four sequences of 1,024
// tokens 28.2 / 23.1 (100 MB: 4.4 TB/s), 32 of 200 45.7 / 37.8, one of 900 15.1 / 11.0, of 60 6.9 / 5.5, 64 single tokens 4.7 / 4.4; x 2,048
// 16.1 / 13.0, 20.2 / 16.9, 8.5 / 5.8, 6.9 / 5.5, 4.2 / 4.1.
template <typename T, int GR>
__global__ __launch_bounds__(256) void conv_silu_vec_kernel(const T* __restrict__ u, long us, int C, int taps,
                                                            const float* __restrict__ w, const float* __restrict__ bias,
                                                            T* state, const int* __restrict__ cu,
                                                            const int* __restrict__ slots,
                                                            const int* __restrict__ positions, T* __restrict__ out,
                                                            long os, int act, int rows) {
  constexpr int EV = 16 / sizeof(T);
  const int s = blockIdx.x, c0 = (blockIdx.z * 256 + threadIdx.x) * EV;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  const int i0 = blockIdx.y * rows;
  if (i0 >= len) return;   // (the whole workgroup)
  const int i1 = min(len, i0 + rows);
  const bool on = c0 < C;
  using Row = std::conditional_t<sizeof(T) == 2, short8, floatx4>;
  auto ldrow = [&](const T* p) { return *reinterpret_cast<const Row*>(p); };
  auto flt = [&](const Row& v, float (&f)[EV]) {
#pragma unroll
    for (int e = 0; e < EV; ++e)
      if constexpr (sizeof(T) == 2) f[e] = bf2f((bf16_t)v[e]);
      else f[e] = v[e];
  };
  auto strow = [&](T* p, const float (&f)[EV]) {
    if constexpr (sizeof(T) == 2) {
      store8(p, f);
    } else {
      *reinterpret_cast<floatx4*>(p) = floatx4{f[0], f[1], f[2], f[3]};
    }
  };
  if (slot < 0) {
    float z[EV];
#pragma unroll
    for (int e = 0; e < EV; ++e) z[e] = 0.f;
    for (int i = i0; i < i1 && on; ++i) strow(out + (long)(row0 + i) * os + c0, z);
    return;
  }
  const bool past = positions[row0] > 0;
  Row cur[GR], old[3], last[3];   // old[3 - d] = the input d tokens before the tile's first; last: the sequence's new state
  const Row zero = {};
  float wk[4][EV], b[EV], win[3][EV];
  const bool w4 = taps == 4 && (reinterpret_cast<uintptr_t>(w) & 15) == 0;   // a channel's taps in one 16-byte load
  auto rows_of = [&](int i) {
#pragma unroll
    for (int x = 0; x < GR; ++x) cur[x] = ldrow(u + (long)(row0 + min(i + x, i1 - 1)) * us + c0);
  };
  if constexpr (GR == 1)
    if (on && w4)
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const floatx4 v = *reinterpret_cast<const floatx4*>(w + (long)(c0 + e) * 4);
#pragma unroll
        for (int k = 0; k < 4; ++k) wk[k][e] = v[k];
      }
  if (on) {
    rows_of(i0);
#pragma unroll
    for (int d = 3; d >= 1; --d) {
      const int idx = i0 - d, si = taps - 1 + idx, at = len - d;
      old[3 - d] = last[3 - d] = zero;
      if (d <= taps - 1) {
        if (idx >= 0) old[3 - d] = ldrow(u + (long)(row0 + idx) * us + c0);
        else if (si >= 0) old[3 - d] = ldrow(state + ((long)slot * (taps - 1) + si) * C + c0);   // (the position may be on its way)
        if (GR > 1 && i0 == 0 && at >= 0) last[3 - d] = ldrow(u + (long)(row0 + at) * us + c0);
      }
    }
  }
  if constexpr (GR > 1) {
    // the block's weights in one sweep, turned round in LDS (9 places for 8, so that the threads' reads, 128 bytes apart, meet different banks)
    __shared__ floatx4 sw[256 * EV + 256 * EV / 8];
    if (w4) {
      const int b0 = blockIdx.z * 256 * EV;
      for (int c = threadIdx.x; c < min(256 * EV, C - b0); c += 256) sw[c + c / 8] = *reinterpret_cast<const floatx4*>(w + (long)(b0 + c) * 4);
      __syncthreads();
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const int c = threadIdx.x * EV + e;
        const floatx4 v = sw[on ? c + c / 8 : 0];
#pragma unroll
        for (int k = 0; k < 4; ++k) wk[k][e] = v[k];
      }
    }
  }
  if (!on) return;
#pragma unroll
  for (int e = 0; e < EV; ++e) {
    b[e] = bias ? bias[c0 + e] : 0.f;
    if (!w4)
#pragma unroll
      for (int k = 0; k < 4; ++k) wk[k][e] = k >= 4 - taps ? w[(long)(c0 + e) * taps + (k - (4 - taps))] : 0.f;
  }
#pragma unroll
  for (int x = 0; x < 3; ++x) {
    if (i0 - 3 + x < 0 && !past) old[x] = zero;
    flt(old[x], win[x]);
  }
  if (i0 == 0) {   // the first tile has read the old state, so it writes the new one: the last taps - 1 of [state, inputs]
#pragma unroll
    for (int x = 0; x < 3; ++x) {
      const int si = taps - 4 + x;   // row of the state: the input 3 - x tokens before the end
      if (si < 0) continue;
      Row v = last[x];
      if (GR == 1) {                 // (one token)
        v = x < 2 ? old[x < 2 ? x + 1 : 2] : cur[0];
      } else if (len - 3 + x < 0) {  // of the old state (len is 1 or 2): old[x + len], a token earlier per input
        v = zero;
#pragma unroll
        for (int n = 1; n < 3; ++n)
          if (len == n && x + n < 3) v = old[x + n < 3 ? x + n : 2];
      }
      *reinterpret_cast<Row*>(state + ((long)slot * (taps - 1) + si) * C + c0) = v;
    }
  }
  // (rows in groups, the next group's requested before this one's are used: the window slides over values in registers)
  for (int i = i0; i < i1; i += GR) {
    Row now[GR];
#pragma unroll
    for (int x = 0; x < GR; ++x) now[x] = cur[x];
    if (i + GR < i1) rows_of(i + GR);
#pragma unroll
    for (int x = 0; x < GR; ++x) {
      if (i + x >= i1) break;
      float r[EV], in[EV];
      flt(now[x], in);
#pragma unroll
      for (int e = 0; e < EV; ++e) {
        const float acc = b[e] + wk[0][e] * win[0][e] + wk[1][e] * win[1][e] + wk[2][e] * win[2][e] + wk[3][e] * in[e];
        r[e] = act ? silu_f<sizeof(T) == 4>(acc) : acc;
        win[0][e] = win[1][e];
        win[1][e] = win[2][e];
        win[2][e] = in[e];
      }
      strow(out + (long)(row0 + i + x) * os + c0, r);
    }
  }
}

// grid (sequence, channel block): the sequence's last taps - 1 inputs become its conv state.
// Runs after conv_silu_kernel (which reads the old state).
template <typename T>
__global__ __launch_bounds__(256) void conv_state_kernel(const T* __restrict__ u, long us, int C, int taps,
                                                         T* __restrict__ state, const int* __restrict__ cu,
                                                         const int* __restrict__ slots,
                                                         const int* __restrict__ positions) {
  const int s = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  if (c >= C || slot < 0 || len <= 0) return;
  const bool past = positions[row0] > 0;
  T* st = state + (long)slot * (taps - 1) * C + c;
  T keep[kMaxTaps];
#pragma unroll
  for (int i = 0; i < kMaxTaps; ++i) {
    if (i < taps - 1) {
      const int idx = len - (taps - 1) + i;
      T v;
      stf<T>(&v, 0.f);
      if (idx >= 0) v = u[(long)(row0 + idx) * us + c];
      else if (past) v = st[(long)(i + len) * C];
      keep[i] = v;
    }
  }
#pragma unroll
  for (int i = 0; i < kMaxTaps; ++i)
    if (i < taps - 1) st[(long)i * C] = keep[i];
}

// Sequential scan.  grid (sequence, head, P / 16): 256 threads = 16 state columns p x 16 slices of
// the N state rows (thread holds rows ns * NR .. ns * NR + NR - 1), so y_t[p] is a 16-lane butterfly.
// Tokens are taken in tiles of kScanTile: the tile's B, C (as f32), x, softplus(dt) and the decay are
// staged in LDS with coalesced loads (16-byte ones when the row layout allows), so the recurrence
// itself runs on LDS reads only -- per-token global loads of a few bytes per lane made the first
// version address-unit bound (18 tiny loads per lane and token).
constexpr int kScanTile = 16;

template <typename T, int NR>
__global__ __launch_bounds__(256) void ssm_scan_kernel(const T* __restrict__ xbc, long xs, const T* __restrict__ dtp,
                                                       long dts, int heads, int P, int N, int groups,
                                                       const float* __restrict__ dt_bias,
                                                       const float* __restrict__ A_log, const float* __restrict__ Dp,
                                                       float* __restrict__ state, const int* __restrict__ cu,
                                                       const int* __restrict__ slots,
                                                       const int* __restrict__ positions, float* __restrict__ y,
                                                       long ys) {
  constexpr int NP = NR * 16;  // padded state rows
  constexpr int EV = 16 / sizeof(T);
  __shared__ __attribute__((aligned(16))) float sB[kScanTile][NP];
  __shared__ __attribute__((aligned(16))) float sC[kScanTile][NP];
  __shared__ float sx[kScanTile][16], sy[kScanTile][16], sdt[kScanTile], sdA[kScanTile];
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x;
  const int ns = tid & 15, pl = tid >> 4, p0 = blockIdx.z * 16, p = p0 + pl;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  if (len <= 0) return;
  const bool pv = p < P;
  if (slot < 0) {
    for (int i = tid; i < len * 16; i += 256)
      if (p0 + (i & 15) < P) y[(long)(row0 + (i >> 4)) * ys + (long)h * P + p0 + (i & 15)] = 0.f;
    return;
  }
  const int inner = heads * P, grp = h / (heads / groups);
  const long xo = (long)h * P + p0, bo = inner + (long)grp * N, co = inner + (long)groups * N + (long)grp * N;
  float* sp = state + (((long)slot * heads + h) * P + (pv ? p : 0)) * N;
  float S[NR];
  const bool past = positions[row0] > 0;
#pragma unroll
  for (int i = 0; i < NR; ++i) {
    const int n = ns * NR + i;
    S[i] = (past && pv && n < N) ? sp[n] : 0.f;
  }
  const float nA = -expf(A_log[h]), db = dt_bias[h], Dh = Dp[h];
  // 16-byte staging loads need every row's B / C run to start on a 16-byte boundary
  const bool vec = N % EV == 0 && xs % EV == 0 && bo % EV == 0 && co % EV == 0 &&
                   (reinterpret_cast<uintptr_t>(xbc) & 15) == 0;
  // vector path: the next tile's global loads are issued before the current tile is computed and
  // land in registers meanwhile (a tile's exposed load latency was ~2/3 of its time otherwise)
  constexpr int NPF = (2 * kScanTile * NP / EV + 255) / 256;
  uint4_t pre[NPF];
  float prex = 0.f, predt = 0.f;
  auto fetch = [&](int t0) {
    const int tl = min(kScanTile, len - t0), cpr = N / EV;
#pragma unroll
    for (int k = 0; k < NPF; ++k) {
      const int i = tid + 256 * k;
      if (i < tl * cpr * 2) {
        const int which = i / (tl * cpr), r = i % (tl * cpr), t = r / cpr, c = r % cpr;
        pre[k] = *reinterpret_cast<const uint4_t*>(xbc + (long)(row0 + t0 + t) * xs + (which ? co : bo) + c * EV);
      }
    }
    const int t = tid >> 4, c = tid & 15;
    prex = (t < tl && p0 + c < P) ? ldf<T>(xbc + (long)(row0 + t0 + t) * xs + xo + c) : 0.f;
    if (tid < tl) predt = ldf<T>(dtp + (long)(row0 + t0 + tid) * dts + h);
  };
  if (vec) fetch(0);
  for (int t0 = 0; t0 < len; t0 += kScanTile) {
    const int tl = min(kScanTile, len - t0);
    __syncthreads();  // the previous tile's sy / sB readers are done
    float dtraw = 0.f;
    if (vec) {
      const int cpr = N / EV;
#pragma unroll
      for (int k = 0; k < NPF; ++k) {
        const int i = tid + 256 * k;
        if (i < tl * cpr * 2) {
          const int which = i / (tl * cpr), r = i % (tl * cpr), t = r / cpr, c = r % cpr;
          float* dst = (which ? sC[t] : sB[t]) + c * EV;
          if constexpr (sizeof(T) == 2) {
            const short8 v = __builtin_bit_cast(short8, pre[k]);
#pragma unroll
            for (int e = 0; e < 8; ++e) dst[e] = bf2f((bf16_t)v[e]);
          } else {
            *reinterpret_cast<uint4_t*>(dst) = pre[k];
          }
        }
      }
      if ((tid >> 4) < tl) sx[tid >> 4][tid & 15] = prex;
      dtraw = predt;
    } else {
      for (int i = tid; i < tl * N * 2; i += 256) {
        const int which = i / (tl * N), r = i % (tl * N), t = r / N, n = r % N;
        (which ? sC[t] : sB[t])[n] = ldf<T>(xbc + (long)(row0 + t0 + t) * xs + (which ? co : bo) + n);
      }
      const int t = tid >> 4, c = tid & 15;  // 16 tokens x 16 columns: one x each
      if (t < tl) sx[t][c] = p0 + c < P ? ldf<T>(xbc + (long)(row0 + t0 + t) * xs + xo + c) : 0.f;
      if (tid < tl) dtraw = ldf<T>(dtp + (long)(row0 + t0 + tid) * dts + h);
    }
    if (N < NP)
      for (int i = tid; i < tl * (NP - N); i += 256) {
        const int t = i / (NP - N), n = N + i % (NP - N);
        sB[t][n] = 0.f;
        sC[t][n] = 0.f;
      }
    if (tid < tl) {
      const float a = dtraw + db;
      const float dt = a > 20.f ? a : log1pf(expf(a));
      sdt[tid] = dt;
      sdA[tid] = expf(nA * dt);
    }
    __syncthreads();
    if (vec && t0 + kScanTile < len) fetch(t0 + kScanTile);
    auto token = [&](int t) {
      const float x = sx[t][pl], dA = sdA[t], dx = sdt[t] * x;
      float acc = 0.f;
#pragma unroll
      for (int k = 0; k < NR; ++k) {
        S[k] = dA * S[k] + dx * sB[t][ns * NR + k];
        acc += S[k] * sC[t][ns * NR + k];
      }
      acc += __shfl_xor(acc, 1, 64);
      acc += __shfl_xor(acc, 2, 64);
      acc += __shfl_xor(acc, 4, 64);
      acc += __shfl_xor(acc, 8, 64);
      if (ns == 0) sy[t][pl] = acc + Dh * x;
    };
    if (tl == kScanTile) {  // whole tile: unrolled, so a token's LDS reads issue under its predecessor's reduction
#pragma unroll
      for (int t = 0; t < kScanTile; ++t) token(t);
    } else {
      for (int t = 0; t < tl; ++t) token(t);
    }
    __syncthreads();
    {
      const int t = tid >> 4, c = tid & 15;
      if (t < tl && p0 + c < P) y[(long)(row0 + t0 + t) * ys + (long)h * P + p0 + c] = sy[t][c];
    }
  }
  if (pv) {
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const int n = ns * NR + i;
      if (n < N) sp[n] = S[i];
    }
  }
}

// four adjacent values, zero where the lane has none; vec: the address is aligned to all four
template <typename T>
LK_DEVICE void ld4s(const T* p, bool on, bool vec, float (&f)[4]) {
  if (on && vec) {
    if constexpr (sizeof(T) == 2) {
      const short4_t v = *reinterpret_cast<const short4_t*>(p);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = bf2f((bf16_t)v[e]);
    } else {
      const floatx4 v = *reinterpret_cast<const floatx4*>(p);
#pragma unroll
      for (int e = 0; e < 4; ++e) f[e] = v[e];
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; ++e) f[e] = on ? ldf<T>(p + e) : 0.f;
  }
}

// the value of lane ^ O, by the vector unit's lane moves
template <int O>
LK_DEVICE float lane_xor(float v) {
  static_assert(O == 1 || O == 2 || O == 4 || O == 8);
  const int i = (int)__float_as_uint(v);
  if constexpr (O == 4) {  // ^ 3, then ^ 7 (the half row mirrored)
    const int q = __builtin_amdgcn_update_dpp(0, i, 0x1b, 0xf, 0xf, true);
    return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, q, 0x141, 0xf, 0xf, true));
  } else {  // quad_perm [1, 0, 3, 2], [2, 3, 0, 1]; row_ror 8
    return __uint_as_float((unsigned)__builtin_amdgcn_update_dpp(0, i, O == 1 ? 0xb1 : O == 2 ? 0x4e : 0x128, 0xf, 0xf, true));
  }
}
// butterfly over the distances O, 2 O, .. below END
template <int O, int END>
LK_DEVICE float group_sum(float v) {
  if constexpr (O >= END) {
    return v;
  } else if constexpr (O < 16) {
    return group_sum<2 * O, END>(v + lane_xor<O>(v));
  } else {
    const unsigned u = __float_as_uint(v);
    if constexpr (O == 16) {
      const auto h = __builtin_amdgcn_permlane16_swap(u, u, false, false);
      return group_sum<2 * O, END>(__uint_as_float(h[0]) + __uint_as_float(h[1]));
    } else {
      const auto h = __builtin_amdgcn_permlane32_swap(u, u, false, false);
      return __uint_as_float(h[0]) + __uint_as_float(h[1]);
    }
  }
}

// One token per sequence (decode): grid (sequence, head).  All a step does is pass over the state once
// (read, decay, add, write: 8 bytes per element), so HBM is the bound and the kernel is laid out for it:
// LPR = N / 4 lanes hold one state row [n] as 16-byte vectors, a wave covers 64 / LPR rows per access and
// requests RB of them together.  y_p is the row's sum over its lanes: the RB rows' sums are halved against
// each other first (log2 RB exchanges leave one row per lane group), then finished inside the group.
// FULL: N = 4 LPR, P whole passes, rows aligned.  Then nothing is tested per row, and a wave's rows lie at immediates from one address:
// 69 registers instead of 142, so that 7 waves and not 3 per SIMD keep requests in flight; the exchanges are lane moves of the vector
// unit instead of the LDS unit's.  64 sequences x 64 heads x [64, 128]: 143 us as a one-token run of ssm_scan_kernel (256 threads for 16
// rows, positions before the state is requested) -> 67 us (without FULL) -> 48 us, 5.6 TB/s; a bare pass over the state takes 43.
template <typename T, int LPR, int RB, bool FULL>
__global__ __launch_bounds__(256) void ssm_step_kernel(const T* __restrict__ xbc, long xs, const T* __restrict__ dtp, long dts,
                                                       int heads, int P, int N, int groups, const float* __restrict__ dt_bias,
                                                       const float* __restrict__ A_log, const float* __restrict__ Dp,
                                                       float* __restrict__ state, const int* __restrict__ cu,
                                                       const int* __restrict__ slots, const int* __restrict__ positions,
                                                       float* __restrict__ y, long ys) {
  constexpr int RPA = 64 / LPR;  // rows per access of a wave
  const int s = blockIdx.x, h = blockIdx.y, lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int row0 = cu[s], row1 = cu[s + 1], slot = slots[s];
  if (row1 <= row0) return;
  const int sub = lane / LPR, nl = lane % LPR, n0 = nl * 4;
  if (slot < 0) {
    for (int row = row0; row < row1; ++row)
      for (int p = threadIdx.x; p < P; p += 256) y[(long)row * ys + (long)h * P + p] = 0.f;
    return;
  }
  const int inner = heads * P, grp = h / (heads / groups);
  const bool nv = FULL || n0 < N;
  bool past = positions[row0] > 0;
  const float nA = -expf(A_log[h]), db = dt_bias[h], Dh = Dp[h];
  const bool vec = FULL || ((reinterpret_cast<uintptr_t>(xbc) | xs * sizeof(T) | inner * sizeof(T)) & (4 * sizeof(T) - 1)) == 0;
  float* sp = state + ((long)slot * heads + h) * P * N;
  const int ld = FULL ? 4 * LPR : N;
  for (int row = row0; row < row1; ++row) {  // (a longer sequence comes back to the rows that this thread has written)
    const T* in = xbc + (long)row * xs;
    const T* xp = in + (long)h * P;
    float* yr = y + (long)row * ys + (long)h * P;
    float B[4], C[4];
    ld4s<T>(in + inner + (long)grp * N + n0, nv, vec, B);
    ld4s<T>(in + inner + (long)(groups + grp) * N + n0, nv, vec, C);
    const float a = ldf<T>(dtp + (long)row * dts + h) + db;
    const float dt = a > 20.f ? a : log1pf(expf(a));
    const float dA = expf(nA * dt);
    for (int p0 = w * RPA * RB; p0 < P; p0 += 4 * RPA * RB) {
      floatx4 S[RB];
      float x[RB], acc[RB];
      float* const s0 = sp + (long)(p0 + sub) * ld + n0;
      const T* const x0 = xp + p0 + sub;
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const bool on = FULL || p0 + i * RPA + sub < P;
        // (requested whether the sequence has a past or not: the position is still on its way)
        S[i] = nv && on ? __builtin_nontemporal_load(reinterpret_cast<const floatx4*>(s0 + (long)i * RPA * ld)) : (floatx4){0.f, 0.f, 0.f, 0.f};
        x[i] = on ? ldf<T>(x0 + i * RPA) : 0.f;
      }
#pragma unroll
      for (int i = 0; i < RB; ++i) {
        const float dx = dt * x[i];
        acc[i] = 0.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          S[i][e] = dA * (past ? S[i][e] : 0.f) + dx * B[e];
          acc[i] += S[i][e] * C[e];
        }
        if (nv && (FULL || p0 + i * RPA + sub < P)) __builtin_nontemporal_store(S[i], reinterpret_cast<floatx4*>(s0 + (long)i * RPA * ld));
      }
      // halve the rows against the lanes of a group: an exchange at distance o leaves each lane with the half
      // of the rows that bit o of its number names
      int base = 0;  // first row of the block that acc[0] stands for
      auto halve = [&](auto k_t) {
        constexpr int k = decltype(k_t)::value, o = RB / 2 / k;
        const bool up = nl & o;
#pragma unroll
        for (int i = 0; i < k; ++i) {
          const float mine = up ? acc[i + k] : acc[i], give = up ? acc[i] : acc[i + k];
          acc[i] = mine + lane_xor<o>(give);
        }
        base += up ? k : 0;
      };
      if constexpr (RB >= 8) halve(std::integral_constant<int, 4>{});
      if constexpr (RB >= 4) halve(std::integral_constant<int, 2>{});
      if constexpr (RB >= 2) halve(std::integral_constant<int, 1>{});
      acc[0] = group_sum<RB, LPR>(acc[0]);
      const int p = p0 + base * RPA + sub;
      if (nl < RB && (FULL || p < P)) yr[p] = acc[0] + Dh * ldf<T>(xp + p);
    }
    past = true;
  }
}

// Chunked (matrix-form) scan for prompt portions: the recurrence is unrolled over chunks of 16
// tokens and every product runs on true-f32 MFMAs (v_mfma_f32_16x16x4_f32), the state staying in
// the accumulators' layout from chunk to chunk.  With a_t = -exp(A_log) dt_t, c_t = a_1 + .. + a_t
// inside the chunk and S the state before it:
//   y_t  = exp(c_t) C_t^T S  +  sum_{s<=t} exp(c_t - c_s) dt_s (C_t . B_s) x_s  +  D x_t
//   S'   = exp(c_L) S  +  sum_s exp(c_L - c_s) dt_s B_s x_s^T
// grid (sequence, head, P / 64): wave w owns the 16 state columns p0 + 16 w .. +15 (all N rows:
// N / 16 accumulator tiles).  Per chunk a wave issues about 12 + 4 N / 16 ... MFMAs instead of
// 16 x 2 N / 16 scalar FMA rounds per lane; tokens past the end of the last chunk get dt = a = 0,
// so they neither decay nor feed the state.  Operand orders are permuted as in attn_sigmoid.hip so
// that accumulators feed the next MFMA without shuffles.
template <typename T, int NR>
__global__ __launch_bounds__(256) void ssm_chunk_kernel(const T* __restrict__ xbc, long xs, const T* __restrict__ dtp,
                                                        long dts, int heads, int P, int N, int groups,
                                                        const float* __restrict__ dt_bias,
                                                        const float* __restrict__ A_log, const float* __restrict__ Dp,
                                                        float* __restrict__ state, const int* __restrict__ cu,
                                                        const int* __restrict__ slots,
                                                        const int* __restrict__ positions, float* __restrict__ y,
                                                        long ys) {
  constexpr int NP = NR * 16, LD = NP + 4, L = 16;
  constexpr int EV = 16 / sizeof(T);
  __shared__ __attribute__((aligned(16))) float sB[L][LD];
  __shared__ __attribute__((aligned(16))) float sC[L][LD];
  __shared__ float sx[L][64], sdt[L], sa[L];
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, p0 = blockIdx.z * 64;
  const int lane = tid & 63, w = tid >> 6, n16 = lane & 15, g = lane >> 4;
  const int pcol = p0 + 16 * w + n16;
  const bool pv = pcol < P;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  if (len <= 0) return;
  if (slot < 0) {
    for (int i = tid; i < len * 64; i += 256)
      if (p0 + (i & 63) < P) y[(long)(row0 + (i >> 6)) * ys + (long)h * P + p0 + (i & 63)] = 0.f;
    return;
  }
  const int inner = heads * P, grp = h / (heads / groups);
  const long xo = (long)h * P + p0, bo = inner + (long)grp * N, co = inner + (long)groups * N + (long)grp * N;
  float* sp = state + (((long)slot * heads + h) * P + (pv ? pcol : 0)) * N;
  const bool past = positions[row0] > 0;
  floatx4 S[NR];
#pragma unroll
  for (int nt = 0; nt < NR; ++nt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = nt * 16 + 4 * g + j;
      S[nt][j] = (past && pv && n < N) ? sp[n] : 0.f;
    }
  const float nA = -expf(A_log[h]), db = dt_bias[h], Dh = Dp[h];
  const bool vec = N % EV == 0 && xs % EV == 0 && bo % EV == 0 && co % EV == 0 &&
                   (reinterpret_cast<uintptr_t>(xbc) & 15) == 0;
  // vector path: the next chunk's operands are requested before this chunk's products are issued
  constexpr int NPF = (2 * L * NP / EV + 255) / 256;
  uint4_t pre[NPF];
  float prex[4], predt = 0.f;
  auto fetch = [&](int t0) {
    const int tl = min(L, len - t0), cpr = NP / EV, ncpr = N / EV;
#pragma unroll
    for (int k = 0; k < NPF; ++k) {
      const int i = tid + 256 * k;
      pre[k] = uint4_t{0u, 0u, 0u, 0u};
      if (i < L * cpr * 2) {
        const int which = i / (L * cpr), r = i % (L * cpr), t = r / cpr, c = r % cpr;
        if (t < tl && c < ncpr)
          pre[k] = *reinterpret_cast<const uint4_t*>(xbc + (long)(row0 + t0 + t) * xs + (which ? co : bo) + c * EV);
      }
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int i = tid + 256 * k, t = i >> 6, c = i & 63;
      prex[k] = (t < tl && p0 + c < P) ? ldf<T>(xbc + (long)(row0 + t0 + t) * xs + xo + c) : 0.f;
    }
    predt = tid < tl ? ldf<T>(dtp + (long)(row0 + t0 + tid) * dts + h) : 0.f;
  };
  if (vec) fetch(0);
  for (int t0 = 0; t0 < len; t0 += L) {
    const int tl = min(L, len - t0);
    __syncthreads();
    float dtraw = 0.f;
    if (vec) {
      const int cpr = NP / EV;
#pragma unroll
      for (int k = 0; k < NPF; ++k) {
        const int i = tid + 256 * k;
        if (i < L * cpr * 2) {
          const int which = i / (L * cpr), r = i % (L * cpr), t = r / cpr, c = r % cpr;
          float* dst = (which ? sC[t] : sB[t]) + c * EV;
          if constexpr (sizeof(T) == 2) {
            const short8 v = __builtin_bit_cast(short8, pre[k]);
#pragma unroll
            for (int e = 0; e < 8; ++e) dst[e] = bf2f((bf16_t)v[e]);
          } else {
            *reinterpret_cast<uint4_t*>(dst) = pre[k];
          }
        }
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int i = tid + 256 * k;
        sx[i >> 6][i & 63] = prex[k];
      }
      dtraw = predt;
    } else {
      for (int i = tid; i < L * NP * 2; i += 256) {
        const int which = i / (L * NP), r = i % (L * NP), t = r / NP, n = r % NP;
        (which ? sC[t] : sB[t])[n] =
            (t < tl && n < N) ? ldf<T>(xbc + (long)(row0 + t0 + t) * xs + (which ? co : bo) + n) : 0.f;
      }
      for (int i = tid; i < L * 64; i += 256) {
        const int t = i >> 6, c = i & 63;
        sx[t][c] = (t < tl && p0 + c < P) ? ldf<T>(xbc + (long)(row0 + t0 + t) * xs + xo + c) : 0.f;
      }
      if (tid < tl) dtraw = ldf<T>(dtp + (long)(row0 + t0 + tid) * dts + h);
    }
    if (tid < L) {
      float dt = 0.f;
      if (tid < tl) {
        const float a = dtraw + db;
        dt = a > 20.f ? a : log1pf(expf(a));
      }
      sdt[tid] = dt;
      sa[tid] = nA * dt;
    }
    __syncthreads();
    if (vec && t0 + L < len) fetch(t0 + L);
    // inclusive prefix of the log-decays inside every 16-lane group: lane n16 ends up with c_(n16)
    float cum = sa[n16];
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const float v = __shfl_up(cum, o, 16);
      if (n16 >= o) cum += v;
    }
    // G^T: lane (t = n16, g) gets G[t][s = 4g + j] = C_t . B_s
    floatx4 gt = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nb = 0; nb < NR; ++nb) {
      const floatx4 a4 = *reinterpret_cast<const floatx4*>(&sB[n16][nb * 16 + 4 * g]);
      const floatx4 b4 = *reinterpret_cast<const floatx4*>(&sC[n16][nb * 16 + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) gt = __builtin_amdgcn_mfma_f32_16x16x4f32(a4[j], b4[j], gt, 0, 0, 0);
    }
    const float ct = cum, cl = __shfl(cum, 15, 16);
    float M[4], xv[4], wv[4], ec[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int sj = 4 * g + j;
      const float cs = __shfl(cum, sj, 16), ds = sdt[sj];
      M[j] = sj <= n16 ? gt[j] * expf(ct - cs) * ds : 0.f;
      xv[j] = sx[sj][16 * w + n16];
      wv[j] = expf(cl - cs) * ds;
      ec[j] = expf(cs);
    }
    // y: rows t = 4g + j, column p = n16 of this wave's tile
    floatx4 ya = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nt = 0; nt < NR; ++nt) {
      const floatx4 c4 = *reinterpret_cast<const floatx4*>(&sC[n16][nt * 16 + 4 * g]);
#pragma unroll
      for (int j = 0; j < 4; ++j) ya = __builtin_amdgcn_mfma_f32_16x16x4f32(c4[j], S[nt][j], ya, 0, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) ya[j] *= ec[j];
#pragma unroll
    for (int j = 0; j < 4; ++j) ya = __builtin_amdgcn_mfma_f32_16x16x4f32(M[j], xv[j], ya, 0, 0, 0);
    if (pv) {
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int t = 4 * g + j;
        if (t < tl) y[(long)(row0 + t0 + t) * ys + (long)h * P + pcol] = ya[j] + Dh * xv[j];
      }
    }
    // state: rows n = 16 nt + 4g + j, column p = n16
    const float dec = expf(cl);
#pragma unroll
    for (int nt = 0; nt < NR; ++nt) {
#pragma unroll
      for (int j = 0; j < 4; ++j) S[nt][j] *= dec;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        S[nt] = __builtin_amdgcn_mfma_f32_16x16x4f32(sB[4 * g + j][nt * 16 + n16] * wv[j], xv[j], S[nt], 0, 0, 0);
    }
  }
  if (pv) {
#pragma unroll
    for (int nt = 0; nt < NR; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int n = nt * 16 + 4 * g + j;
        if (n < N) sp[n] = S[nt][j];
      }
  }
}

// The same matrix form for bf16 rows in chunks of 64 tokens on bf16 MFMAs (v_mfma_f32_16x16x32_bf16).  B, C and x ARE bf16, so
// products of them lose nothing; what is f32 -- the state, the masked and decayed C.B matrix M, the weighted x of the state update --
// enters a product as three bf16 parts (8 + 8 + 8 mantissa bits, an f32), summed in the f32 accumulators.  A sequence's chunks are a
// serial chain, so what bounds the kernel is the time of one chunk: 64 tokens take 130 products of 16 cycles per wave instead of
// 4 x 100 of 32 (16x16x4 f32), with two barriers instead of eight.  4 x 1,024 tokens, 64 heads of [64, 128]: 351 us (f32
// products, chunks of 16) -> 126 us (now ssm_pipe_kernel's, which takes states of 33 - 128 columns: lk_ssm_piped); 4 x 512, 32 heads of [64, 256] 75 us.
// Error against f64 9e-8 (f32 products: 2.2e-7).
// grid (sequence, head, P / 64): wave w owns state columns p0 + 16 w .. +15 (all N rows as accumulators S[n][p]: lane p = l & 15,
// rows 16 nt + 4 (l >> 4) + j) and computes M's rows of token tile w for everybody.  y is accumulated transposed (lane: one token,
// four adjacent columns).  The order of n inside a 32-step is (4g + j, 16 + 4g + j), so that the accumulators are operands as they lie.
struct BfParts {
  short8 p[3];
};
LK_DEVICE BfParts bf_split3(const float (&v)[8]) {
  BfParts r;
  float rest[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) rest[e] = v[e];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    uint4_t u;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      u[e] = pack_bf2(rest[2 * e], rest[2 * e + 1]);
      rest[2 * e] -= __uint_as_float(u[e] << 16);
      rest[2 * e + 1] -= __uint_as_float(u[e] & 0xffff0000u);
    }
    r.p[k] = __builtin_bit_cast(short8, u);
  }
  return r;
}

// exp of a sum carried in f64: the rounding of the argument to f32 is put back to first order
LK_DEVICE float exp_f64sum(double c) {
  const float hi = (float)c, e = expf(hi);
  return fmaf(e, (float)(c - hi), e);
}

template <int NR>
constexpr int ssm_chunk_lds() {
  return 2 * 64 * (NR * 16 + 8) * 2 + NR * 16 * 72 * 2 + 64 * 72 * 2 + 3 * 64 * 72 * 2 + 5 * 64 * 4;
}

// the lanes' doubles moved by one DPP control (0 where a lane has no source or its row is masked out)
template <int CTRL, int ROWS>
LK_DEVICE double dpp64(double v) {
  const int2 a = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, make_int2(__builtin_amdgcn_update_dpp(0, a.x, CTRL, ROWS, 0xf, ROWS == 0xf),
                                              __builtin_amdgcn_update_dpp(0, a.y, CTRL, ROWS, 0xf, ROWS == 0xf)));
}

template <int NR>
__global__ __launch_bounds__(256, 1) void ssm_chunk_bf16_kernel(const bf16_t* __restrict__ xbc, long xs, const bf16_t* __restrict__ dtp,
                                                                long dts, int heads, int P, int N, int groups,
                                                                const float* __restrict__ dt_bias, const float* __restrict__ A_log,
                                                                const float* __restrict__ Dp, float* __restrict__ state,
                                                                const int* __restrict__ cu, const int* __restrict__ slots,
                                                                const int* __restrict__ positions, float* __restrict__ y, long ys) {
  constexpr int L = 64, NP = NR * 16, LN = NP + 8, LT = L + 8;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* const sB = reinterpret_cast<bf16_t*>(smem);  // [t][n]
  bf16_t* const sC = sB + L * LN;                      // [t][n]
  bf16_t* const sBt = sC + L * LN;                     // [n][t]
  bf16_t* const sXt = sBt + NP * LT;                   // [p][t]
  bf16_t* const sM = sXt + 64 * LT;                    // [part][t][s]
  float* const sc = reinterpret_cast<float*>(sM + 3 * L * LT);
  float *const sdt = sc + L, *const sec = sdt + L, *const swv = sec + L, *const scl = swv + L;
  const int s = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, p0 = blockIdx.z * 64;
  const int lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), r16 = lane & 15, g = lane >> 4;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  if (len <= 0) return;
  if (slot < 0) {
    for (int i = tid; i < len * 64; i += 256)
      if (p0 + (i & 63) < P) y[(long)(row0 + (i >> 6)) * ys + (long)h * P + p0 + (i & 63)] = 0.f;
    return;
  }
  const int inner = heads * P, grp = h / (heads / groups);
  const bf16_t* const bx = xbc + (long)row0 * xs + (long)h * P + p0;
  const bf16_t* const bb = xbc + (long)row0 * xs + inner + (long)grp * N;
  const bf16_t* const bc = bb + (long)groups * N;
  const int pcol = p0 + 16 * w + r16;
  const bool pv = pcol < P, past = positions[row0] > 0;
  float* const sp = state + (((long)slot * heads + h) * P + (pv ? pcol : 0)) * N;
  floatx4 S[NR];
#pragma unroll
  for (int nt = 0; nt < NR; ++nt) {
    const int n = nt * 16 + 4 * g;
    S[nt] = (past && pv && n < N) ? *reinterpret_cast<const floatx4*>(sp + n) : (floatx4){0.f, 0.f, 0.f, 0.f};
  }
  const float nA = -expf(A_log[h]), db = dt_bias[h], Dh = Dp[h];

  // a chunk's rows, requested one chunk ahead: B and x as 4 tokens x 4 columns per thread (filed in both orders), C as 16 bytes
  constexpr int NB = NP / 64 > 0 ? NP / 64 : 1, NC = NP / 32;
  short4_t fb[NB][4], fx[4];
  uint4_t fc[NC];
  bf16_t fdt = 0;
  const short4_t z4 = {0, 0, 0, 0};
  auto fetch = [&](int t0) {
    const int tl = len - t0;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int b = tid + 256 * k, n = (b % (NP / 4)) * 4, t = (b / (NP / 4)) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        fb[k][i] = (t + i < min(tl, L) && n < N) ? *reinterpret_cast<const short4_t*>(bb + (long)(t0 + t + i) * xs + n) : z4;
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int b = tid + 256 * k, n = (b % (NP / 8)) * 8, t = b / (NP / 8);
      fc[k] = (t < tl && n < N) ? *reinterpret_cast<const uint4_t*>(bc + (long)(t0 + t) * xs + n) : (uint4_t){0u, 0u, 0u, 0u};
    }
    const int xp = (tid & 15) * 4, xt = (tid >> 4) * 4;
#pragma unroll
    for (int i = 0; i < 4; ++i)
      fx[i] = (xt + i < tl && p0 + xp < P) ? *reinterpret_cast<const short4_t*>(bx + (long)(t0 + xt + i) * xs + xp) : z4;
    // (kept as it lies: converted here, every load above would be waited for at once, 2 us of a chunk)
    fdt = dtp[(long)(row0 + t0 + min(lane, tl - 1)) * dts + h];
  };
  // a transposed row's groups of 8 tokens are turned by the row: threads file rows four apart, which lay in the same banks (16 deep)
  auto at_t = [&](int row, int t) { return row * LT + (((t >> 3) ^ ((row >> 3) & 7)) << 3) + (t & 7); };
  fetch(0);
  for (int t0 = 0; t0 < len; t0 += L) {
    const int tl = min(L, len - t0);
    __syncthreads();  // the previous chunk's readers are done
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int b = tid + 256 * k, n = (b % (NP / 4)) * 4, t = (b / (NP / 4)) * 4;
      if (t < L) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          *reinterpret_cast<short4_t*>(sB + (t + i) * LN + n) = fb[k][i];
          *reinterpret_cast<short4_t*>(sBt + at_t(n + i, t)) = (short4_t){fb[k][0][i], fb[k][1][i], fb[k][2][i], fb[k][3][i]};
        }
      }
    }
#pragma unroll
    for (int k = 0; k < NC; ++k) {
      const int b = tid + 256 * k;
      *reinterpret_cast<uint4_t*>(sC + (b / (NP / 8)) * LN + (b % (NP / 8)) * 8) = fc[k];
    }
    {
      const int xp = (tid & 15) * 4, xt = (tid >> 4) * 4;
#pragma unroll
      for (int i = 0; i < 4; ++i)
        *reinterpret_cast<short4_t*>(sXt + at_t(xp + i, xt)) = (short4_t){fx[0][i], fx[1][i], fx[2][i], fx[3][i]};
    }
    // lane = token: c, the running sum of the log-decays (every wave computes and files the same values)
    float dec;
    {
      const float a = bf2f(fdt) + db;
      const float dt = lane < tl ? (a > 20.f ? a : log1pf(expf(a))) : 0.f;
      // (the sum over 64 tokens in f64 and as two floats: a difference of two of them keeps an f32's relative error, as the
      // 16-token chunks' sums did)
      double c = (double)nA * dt;
      c += dpp64<0x111, 0xf>(c);   // row_shr 1, 2, 4, 8: inside 16 lanes (by the LDS unit, 14 exchanges deep, it was a tenth of a chunk)
      c += dpp64<0x112, 0xf>(c);
      c += dpp64<0x114, 0xf>(c);
      c += dpp64<0x118, 0xf>(c);
      c += dpp64<0x142, 0xa>(c);   // row_bcast 15 to the second and fourth 16, 31 to the upper half
      c += dpp64<0x143, 0xc>(c);
      const int2 last = __builtin_bit_cast(int2, c);
      const double cld = __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(last.x, 63), __builtin_amdgcn_readlane(last.y, 63)));
      const float hi = (float)c;
      sc[lane] = hi;
      scl[lane] = (float)(c - hi);
      sdt[lane] = dt;
      sec[lane] = exp_f64sum(c);
      swv[lane] = exp_f64sum(cld - c) * dt;
      dec = exp_f64sum(cld);
    }
    __syncthreads();
    if (t0 + L < len) fetch(t0 + L);

    // M^T tiles: columns t of tile w, rows s of the tiles up to it (one tile of zeros completes a 32-step)
    {
      const int t = 16 * w + r16;
      const float ct = sc[t], ctl = scl[t];
      short8 cf[NR / 2];
#pragma unroll
      for (int kk = 0; kk < NR / 2; ++kk) cf[kk] = *reinterpret_cast<const short8*>(sC + t * LN + 32 * kk + 8 * g);
      // (all four tiles in every wave, side by side: those behind t's are zeros, and the wave with four of them is the one waited for)
      floatx4 m[4];
#pragma unroll
      for (int kk = 0; kk < NR / 2; ++kk)
#pragma unroll
        for (int st = 0; st < 4; ++st) {
          const short8 a = *reinterpret_cast<const short8*>(sB + (16 * st + r16) * LN + 32 * kk + 8 * g);
          m[st] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, cf[kk], kk == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : m[st], 0, 0, 0);
        }
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        const floatx4 cs = *reinterpret_cast<const floatx4*>(sc + 16 * st + 4 * g);
        const floatx4 cw = *reinterpret_cast<const floatx4*>(scl + 16 * st + 4 * g);
        const floatx4 ds = *reinterpret_cast<const floatx4*>(sdt + 16 * st + 4 * g);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int sj = 16 * st + 4 * g + j;
          m[st][j] = sj < t ? m[st][j] * expf((ct - cs[j]) + (ctl - cw[j])) * ds[j]
                            : (sj == t ? m[st][j] * ds[j] + Dh : 0.f);  // the skip D x on the diagonal
        }
      }
#pragma unroll
      for (int st = 0; st < 4; ++st) {
        if (st > (w | 1)) break;   // (the 32-steps behind t's are not read)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          uint2 u;
          u.x = pack_bf2(m[st][0], m[st][1]);
          u.y = pack_bf2(m[st][2], m[st][3]);
          *reinterpret_cast<uint2*>(sM + (k * L + t) * LT + 16 * st + 4 * g) = u;
          m[st][0] -= __uint_as_float(u.x << 16);
          m[st][1] -= __uint_as_float(u.x & 0xffff0000u);
          m[st][2] -= __uint_as_float(u.y << 16);
          m[st][3] -= __uint_as_float(u.y & 0xffff0000u);
        }
      }
    }
    // y^T[p][t] from the state: exp(c_t) S^T C
    floatx4 ya[4];
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) ya[tt] = (floatx4){0.f, 0.f, 0.f, 0.f};
    if (past || t0 > 0) {
#pragma unroll
      for (int kk = 0; kk < NR / 2; ++kk) {
        float v[8];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          v[j] = S[2 * kk][j];
          v[4 + j] = S[2 * kk + 1][j];
        }
        const BfParts q = bf_split3(v);
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) {
          const bf16_t* cp = sC + (16 * tt + r16) * LN + 32 * kk + 4 * g;
          const short4_t lo = *reinterpret_cast<const short4_t*>(cp), hi = *reinterpret_cast<const short4_t*>(cp + 16);
          const short8 c = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
#pragma unroll
          for (int k = 2; k >= 0; --k) ya[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(q.p[k], c, ya[tt], 0, 0, 0);
        }
      }
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) ya[tt] *= sec[16 * tt + r16];
    }
    __syncthreads();  // M is complete
    // (xe: without the second tile of a 32-step, whose M rows are zeros for an even token tile: an infinity or NaN among its x would
    // reach outputs up to 31 tokens before it, not only those of its own 16 as in chunks of 16)
    short8 xf[2], xe[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      xf[kk] = *reinterpret_cast<const short8*>(sXt + at_t(16 * w + r16, 32 * kk + 8 * g));
      xe[kk] = g < 2 ? xf[kk] : (short8){0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) {
#pragma unroll
      for (int kk = 0; kk <= tt / 2; ++kk)
#pragma unroll
        for (int k = 2; k >= 0; --k) {
          const short8 m = *reinterpret_cast<const short8*>(sM + (k * L + 16 * tt + r16) * LT + 32 * kk + 8 * g);
          ya[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(2 * kk == tt ? xe[kk] : xf[kk], m, ya[tt], 0, 0, 0);
        }
      const int t = 16 * tt + r16, p = p0 + 16 * w + 4 * g;
      if (t < tl && p < P) *reinterpret_cast<floatx4*>(y + (long)(row0 + t0 + t) * ys + (long)h * P + p) = ya[tt];
    }
    // S' = exp(c_L) S + B (w x)^T
#pragma unroll
    for (int nt = 0; nt < NR; ++nt) S[nt] *= dec;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float v[8];
      const floatx4 w0 = *reinterpret_cast<const floatx4*>(swv + 32 * kk + 8 * g), w1 = *reinterpret_cast<const floatx4*>(swv + 32 * kk + 8 * g + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = bf2f((bf16_t)xf[kk][e]) * (e < 4 ? w0[e & 3] : w1[e & 3]);
      const BfParts q = bf_split3(v);
#pragma unroll
      for (int nt = 0; nt < NR; ++nt) {
        const short8 b = *reinterpret_cast<const short8*>(sBt + at_t(16 * nt + r16, 32 * kk + 8 * g));
#pragma unroll
        for (int k = 2; k >= 0; --k) S[nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b, q.p[k], S[nt], 0, 0, 0);
      }
    }
  }
  if (pv) {
#pragma unroll
    for (int nt = 0; nt < NR; ++nt) {
      const int n = nt * 16 + 4 * g;
      if (n < N) *reinterpret_cast<floatx4*>(sp + n) = S[nt];
    }
  }
}

// The same for states of 33 - 128 columns and prompts, as a pipeline of 16 waves in one workgroup.  A chunk's chain is latency, not work (with four
// waves, one to a SIMD, 12 k cycles for 4.6 k of vector and 2 k of matrix instructions per SIMD), and half of it does not depend on the state: eight waves
// file the next chunk's rows, its decays and then its M, eight carry the state and y behind them, so that every SIMD has four waves to take
// turns.  Those eight hold half of N each (nh), exchange their halves of S^T C through LDS and finish two token tiles each.
// 64 heads of [64, 128], in four waves / here (us): 4 sequences of 1,024 111 / 61 (y writes 67 MB and the rows read 50: 24), one of 2,000 203 / 99,
// of 300 35 / 19, of 8 10.4 / 7.4, 64 of 8 133 / 95, 512 rows and 64 decode rows 189 / 126; 32 heads of [64, 64], 4 of 1,024 77 / 41.
// Error against f64 as there: 0.9e-7.
template <int NR>
constexpr int ssm_pipe_lds() {
  return 2 * 64 * (NR * 16 + 8) * 2 + 3 * 64 * 72 * 2 + 2 * (NR * 16 * 72 * 2 + 64 * 72 * 2 + 6 * 64 * 4) + 16 * 64 * 16;
}

template <int NR>
__global__ __launch_bounds__(1024) void ssm_pipe_kernel(const bf16_t* __restrict__ xbc, long xs, const bf16_t* __restrict__ dtp, long dts,
                                                        int heads, int P, int N, int groups, const float* __restrict__ dt_bias,
                                                        const float* __restrict__ A_log, const float* __restrict__ Dp,
                                                        float* __restrict__ state, const int* __restrict__ cu,
                                                        const int* __restrict__ slots, const int* __restrict__ positions,
                                                        float* __restrict__ y, long ys) {
  constexpr int L = 64, NP = NR * 16, LN = NP + 8, LT = L + 8, BT = NP * LT, XT = 64 * LT, W = 6 * L, NH = NR / 2;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  bf16_t* const sB = reinterpret_cast<bf16_t*>(smem);  // [t][n]
  bf16_t* const sC = sB + L * LN;                      // [t][n]
  bf16_t* const sM = sC + L * LN;                      // [part][t][s]
  bf16_t* const sBt0 = sM + 3 * L * LT;                // [chunk & 1][n][t]
  bf16_t* const sXt0 = sBt0 + 2 * BT;                  // [chunk & 1][p][t]
  floatx4* const sY = reinterpret_cast<floatx4*>(sXt0 + 2 * XT);   // [column tile][token tile][lane]: the other half's part of S^T C
  float* const sw0 = reinterpret_cast<float*>(sY + 16 * 64);       // [chunk & 1][c, dt, 2^c, weight, c's low part, 2^c_L]
  const int s = blockIdx.x, h = blockIdx.y, p0 = blockIdx.z * 64;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  const int w = wave & 3, half = (wave >> 2) & 1;
  const bool files = wave >= 8;
  const int row0 = cu[s], len = cu[s + 1] - row0, slot = slots[s];
  if (len <= 0) return;
  if (slot < 0) {
    for (int i = threadIdx.x; i < len * 64; i += 1024)
      if (p0 + (i & 63) < P) y[(long)(row0 + (i >> 6)) * ys + (long)h * P + p0 + (i & 63)] = 0.f;
    return;
  }
  // a transposed row's groups of 8 tokens are turned by two in every second tile of 16 rows: 32 lanes file 8 rows four apart at 4 tokens each
  auto at_t = [](int row, int t) { return row * LT + (((t >> 3) ^ ((row >> 3) & 2)) << 3) + (t & 7); };

  if (files) {
    const int inner = heads * P, grp = h / (heads / groups), q = wave - 8;
    const bf16_t* const bx = xbc + (long)row0 * xs + (long)h * P + p0;
    const bf16_t* const bb = xbc + (long)row0 * xs + inner + (long)grp * N;
    const bf16_t* const bc = bb + (long)groups * N;
    const double nA = -1.4426950408889634 * expf(A_log[h]);   // (decays as powers of two: in M one instruction where expf is 13)
    const float db = dt_bias[h], Dh = Dp[h];
    // what a thread files: B as 4 tokens x 4 columns (in both orders), x so too (the upper four waves), C in pieces of 16 bytes
    constexpr int BN = NP / 32, NC = NP / 64;   // (waves across B's columns; pieces of C)
    const bool hasb = q < 2 * BN, hasx = q >= 4;
    const int bn = q % BN * 32 + (lane & 7) * 4, bt = q / BN % 2 * 32 + (lane >> 3) * 4;
    const int xp = (q & 1) * 32 + (lane & 7) * 4, xt = (q >> 1 & 1) * 32 + (lane >> 3) * 4;
    const bool vb = bn < N, vx = p0 + xp < P;
    const int pt = threadIdx.x - 512, cn = pt % (NP / 8) * 8, ct = pt / (NP / 8);
    constexpr int CR = 512 / (NP / 8);   // rows of C between a thread's pieces
    const bool vc = cn < N;
    short4_t fb[4], fx[4];
    uint4_t fc[NC];
    bf16_t fdt = 0;
    // a chunk's rows, requested one chunk ahead (rows and columns that are not there: others again, and zeros when they are filed)
    auto fetch = [&](int t0) {
      const int last = min(len - t0, L) - 1;
      if (q == 4) fdt = dtp[(long)(row0 + t0 + min(lane, last)) * dts + h];
      const bf16_t *const cb = bb + (long)t0 * xs, *const cc = bc + (long)t0 * xs, *const cx = bx + (long)t0 * xs;
      const unsigned st = (unsigned)xs;
      if (hasb) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fb[i] = *reinterpret_cast<const short4_t*>(cb + ((unsigned)min(bt + i, last) * st + (vb ? bn : 0)));
      }
      if (hasx) {
#pragma unroll
        for (int i = 0; i < 4; ++i) fx[i] = *reinterpret_cast<const short4_t*>(cx + ((unsigned)min(xt + i, last) * st + (vx ? xp : 0)));
      }
#pragma unroll
      for (int k = 0; k < NC; ++k) fc[k] = *reinterpret_cast<const uint4_t*>(cc + ((unsigned)min(ct + k * CR, last) * st + (vc ? cn : 0)));
    };
    auto file = [&](int t0, int odd) {
      const int tl = min(L, len - t0);
      const short4_t z4 = {0, 0, 0, 0};
      if (tl < L || N < NP || P - p0 < 64) {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          fb[i] = (bt + i < tl && vb) ? fb[i] : z4;
          fx[i] = (xt + i < tl && vx) ? fx[i] : z4;
        }
#pragma unroll
        for (int k = 0; k < NC; ++k) fc[k] = (ct + k * CR < tl && vc) ? fc[k] : (uint4_t){0u, 0u, 0u, 0u};
      }
      if (hasb) {
        bf16_t* const sBt = sBt0 + odd * BT;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          *reinterpret_cast<short4_t*>(sB + (bt + i) * LN + bn) = fb[i];
          *reinterpret_cast<short4_t*>(sBt + at_t(bn + i, bt)) = (short4_t){fb[0][i], fb[1][i], fb[2][i], fb[3][i]};
        }
      }
      if (hasx) {
        bf16_t* const sXt = sXt0 + odd * XT;
#pragma unroll
        for (int i = 0; i < 4; ++i) *reinterpret_cast<short4_t*>(sXt + at_t(xp + i, xt)) = (short4_t){fx[0][i], fx[1][i], fx[2][i], fx[3][i]};
      }
#pragma unroll
      for (int k = 0; k < NC; ++k) *reinterpret_cast<uint4_t*>(sC + (ct + k * CR) * LN + cn) = fc[k];
    };
    // lane = token: c, the running sum of the log-decays (one wave, of the two that have no tile of M)
    auto decays = [&](int t0, int odd) {
      const int tl = min(L, len - t0);
      float* const sw = sw0 + odd * W;
      const float a = bf2f(fdt) + db;
      const float dt = lane < tl ? (a > 20.f ? a : log1pf(expf(a))) : 0.f;
      // (the sum over 64 tokens in f64 and as two floats: a difference of two of them keeps an f32's relative error, as the
      // 16-token chunks' sums did)
      double c = nA * dt;
      c += dpp64<0x111, 0xf>(c);   // row_shr 1, 2, 4, 8: inside 16 lanes (by the LDS unit, 14 exchanges deep, it was a tenth of a chunk)
      c += dpp64<0x112, 0xf>(c);
      c += dpp64<0x114, 0xf>(c);
      c += dpp64<0x118, 0xf>(c);
      c += dpp64<0x142, 0xa>(c);   // row_bcast 15 to the second and fourth 16, 31 to the upper half
      c += dpp64<0x143, 0xc>(c);
      const int2 last = __builtin_bit_cast(int2, c);
      const double cld = __builtin_bit_cast(double, make_int2(__builtin_amdgcn_readlane(last.x, 63), __builtin_amdgcn_readlane(last.y, 63)));
      constexpr double kLn2 = 0.6931471805599453;
      const float hi = (float)c;
      sw[lane] = hi;
      sw[L + lane] = dt;
      sw[2 * L + lane] = exp_f64sum(c * kLn2);
      sw[3 * L + lane] = exp_f64sum((cld - c) * kLn2) * dt;
      sw[4 * L + lane] = (float)(c - hi);
      sw[5 * L + lane] = exp_f64sum(cld * kLn2);
    };
    // M^T tiles: columns t of tile w, rows s of the half's two tiles (one tile of zeros completes a 32-step; the 32-steps behind t's are not read)
    auto scores = [&](int odd) {
      const float *const sc = sw0 + odd * W, *const sdt = sc + L, *const scl = sc + 4 * L;
      const int t = 16 * w + r16;
      const float ct = sc[t], ctl = scl[t];
      floatx4 m[2], cs[2], cw[2], ds[2];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int o = 32 * half + 16 * u + 4 * g;
        cs[u] = *reinterpret_cast<const floatx4*>(sc + o);
        cw[u] = *reinterpret_cast<const floatx4*>(scl + o);
        ds[u] = *reinterpret_cast<const floatx4*>(sdt + o);
      }
#pragma unroll
      for (int kk = 0; kk < NR / 2; ++kk) {
        const short8 cf = *reinterpret_cast<const short8*>(sC + t * LN + 32 * kk + 8 * g);
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const short8 a = *reinterpret_cast<const short8*>(sB + (32 * half + 16 * u + r16) * LN + 32 * kk + 8 * g);
          m[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, cf, kk == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : m[u], 0, 0, 0);
        }
      }
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const int st = 2 * half + u;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          float below = m[u][j] * (__builtin_amdgcn_exp2f((ct - cs[u][j]) + (ctl - cw[u][j])) * ds[u][j]);
          if (st < w) {
            m[u][j] = below;
          } else {
            const int sj = 16 * st + 4 * g + j;
            asm volatile("" : "+v"(below));   // (side by side: a branch for each otherwise)
            m[u][j] = sj < t ? below : (sj == t ? m[u][j] * ds[u][j] + Dh : 0.f);   // the skip D x on the diagonal
          }
        }
      }
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          uint2 v;
          v.x = pack_bf2(m[u][0], m[u][1]);
          v.y = pack_bf2(m[u][2], m[u][3]);
          *reinterpret_cast<uint2*>(sM + (k * L + t) * LT + 32 * half + 16 * u + 4 * g) = v;
          m[u][0] -= __uint_as_float(v.x << 16);
          m[u][1] -= __uint_as_float(v.x & 0xffff0000u);
          m[u][2] -= __uint_as_float(v.y << 16);
          m[u][3] -= __uint_as_float(v.y & 0xffff0000u);
        }
    };
    fetch(0);
    file(0, 0);
    if (q == 4) decays(0, 0);
    if (L < len) fetch(L);
    __syncthreads();
    int odd = 0;
    for (int t0 = 0; t0 < len; t0 += L, odd ^= 1) {
      if (!half || w >= 2) scores(odd);
      else if (q == 4 && t0 + L < len) decays(t0 + L, odd ^ 1);
      __syncthreads();  // M is complete; B and C by rows are read
      if (t0 + L < len) {
        file(t0 + L, odd ^ 1);
        if (t0 + 2 * L < len) fetch(t0 + 2 * L);
      }
      __syncthreads();  // the next chunk is filed; M and this chunk's columns are read
    }
    return;
  }

  const int pcol = p0 + 16 * w + r16;
  const bool pv = pcol < P, past = positions[row0] > 0;
  float* const sp = state + (((long)slot * heads + h) * P + (pv ? pcol : 0)) * N;
  floatx4 S[NH], ya[4];   // (rows 16 (NH half + j) + 4 g + ..)
#pragma unroll
  for (int j = 0; j < NH; ++j) {
    const int n = (half * NH + j) * 16 + 4 * g;
    S[j] = (past && pv && n < N) ? *reinterpret_cast<const floatx4*>(sp + n) : (floatx4){0.f, 0.f, 0.f, 0.f};
  }
  // y^T[p][t] from the state: 2^c_t S^T C over the half's rows; the token tiles that the other half finishes go to it
  auto from_state = [&](int odd) {
    const float* const sec = sw0 + odd * W + 2 * L;
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) ya[tt] = (floatx4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kk = 0; kk < NH / 2; ++kk) {
      float v[8];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        v[j] = S[2 * kk][j];
        v[4 + j] = S[2 * kk + 1][j];
      }
      const BfParts b = bf_split3(v);
      short8 c[4];
#pragma unroll
      for (int tt = 0; tt < 4; ++tt) {
        const bf16_t* cp = sC + (16 * tt + r16) * LN + 32 * (half * (NH / 2) + kk) + 4 * g;
        const short4_t lo = *reinterpret_cast<const short4_t*>(cp), hi = *reinterpret_cast<const short4_t*>(cp + 16);
        c[tt] = (short8){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      }
#pragma unroll
      for (int k = 2; k >= 0; --k)
#pragma unroll
        for (int tt = 0; tt < 4; ++tt) ya[tt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b.p[k], c[tt], ya[tt], 0, 0, 0);
    }
#pragma unroll
    for (int tt = 0; tt < 4; ++tt) ya[tt] *= sec[16 * tt + r16];
    sY[(w * 4 + 1 - half) * 64 + lane] = half ? ya[0] : ya[1];
    sY[(w * 4 + 2 + half) * 64 + lane] = half ? ya[3] : ya[2];
  };
  // .. and from the chunk's own tokens, for tiles T0 and T1
  auto finish = [&](int t0, int odd, bool both, auto T0, auto T1) {
    const int tl = min(L, len - t0);
    const bf16_t* const sXt = sXt0 + odd * XT;
    constexpr int tts[2] = {decltype(T0)::value, decltype(T1)::value};
    floatx4 a[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) a[i] = both ? ya[tts[i]] + sY[(w * 4 + tts[i]) * 64 + lane] : ya[tts[i]];
    // (xe: without the second tile of a 32-step, whose M rows are zeros for an even token tile: an infinity or NaN among its x would
    // reach outputs up to 31 tokens before it, not only those of its own 16 as in chunks of 16)
    short8 xf[2], xe[2];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      xf[kk] = *reinterpret_cast<const short8*>(sXt + at_t(16 * w + r16, 32 * kk + 8 * g));
      xe[kk] = g < 2 ? xf[kk] : (short8){0, 0, 0, 0, 0, 0, 0, 0};
    }
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
#pragma unroll
      for (int k = 2; k >= 0; --k)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          if (kk > tts[i] / 2) continue;
          const short8 m = *reinterpret_cast<const short8*>(sM + (k * L + 16 * tts[i] + r16) * LT + 32 * kk + 8 * g);
          a[i] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(2 * kk == tts[i] ? xe[kk] : xf[kk], m, a[i], 0, 0, 0);
        }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int t = 16 * tts[i] + r16, p = p0 + 16 * w + 4 * g;
      if (t < tl && p < P) *reinterpret_cast<floatx4*>(y + (long)(row0 + t0 + t) * ys + (long)h * P + p) = a[i];
    }
    // S' = 2^c_L S + B (w x)^T
    const bf16_t* const sBt = sBt0 + odd * BT;
    const float* const swv = sw0 + odd * W + 3 * L;
    const float dec = swv[2 * L];
#pragma unroll
    for (int j = 0; j < NH; ++j) S[j] *= dec;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      float v[8];
      const floatx4 w0 = *reinterpret_cast<const floatx4*>(swv + 32 * kk + 8 * g), w1 = *reinterpret_cast<const floatx4*>(swv + 32 * kk + 8 * g + 4);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = bf2f((bf16_t)xf[kk][e]) * (e < 4 ? w0[e & 3] : w1[e & 3]);
      const BfParts b = bf_split3(v);
#pragma unroll
      for (int k = 2; k >= 0; --k)
#pragma unroll
        for (int j = 0; j < NH; ++j) {
          const short8 a = *reinterpret_cast<const short8*>(sBt + at_t(16 * (half * NH + j) + r16, 32 * kk + 8 * g));
          S[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b.p[k], S[j], 0, 0, 0);
        }
    }
  };
  __syncthreads();
  int odd = 0;
  for (int t0 = 0; t0 < len; t0 += L, odd ^= 1) {
    const bool both = past || t0 > 0;
    if (both) from_state(odd);
    else ya[0] = ya[1] = ya[2] = ya[3] = (floatx4){0.f, 0.f, 0.f, 0.f};
    __syncthreads();
    if (half == 0) finish(t0, odd, both, std::integral_constant<int, 0>{}, std::integral_constant<int, 3>{});
    else finish(t0, odd, both, std::integral_constant<int, 1>{}, std::integral_constant<int, 2>{});
    __syncthreads();
  }
  if (pv) {
#pragma unroll
    for (int j = 0; j < NH; ++j) {
      const int n = (half * NH + j) * 16 + 4 * g;
      if (n < N) *reinterpret_cast<floatx4*>(sp + n) = S[j];
    }
  }
}

// grid (row, norm group): out = (y * silu(z)) / sqrt(mean_group((y silu z)^2) + eps) * w
template <typename T>
__global__ __launch_bounds__(256) void gated_group_rmsnorm_kernel(const float* __restrict__ y, long ys,
                                                                  const T* __restrict__ z, long zs,
                                                                  const float* __restrict__ w, int gs, float eps,
                                                                  T* __restrict__ out, long os) {
  __shared__ float red[4];
  const long row = blockIdx.x;
  const int c0 = blockIdx.y * gs;
  float ss = 0.f;
  for (int c = threadIdx.x; c < gs; c += 256) {
    const float v = y[row * ys + c0 + c] * silu_f<sizeof(T) == 4>(ldf<T>(z + row * zs + c0 + c));
    ss += v * v;
  }
  ss = block_sum<4>(ss, red);
  const float inv = 1.f / sqrtf(ss / (float)gs + eps);
  for (int c = threadIdx.x; c < gs; c += 256) {
    const float v = y[row * ys + c0 + c] * silu_f<sizeof(T) == 4>(ldf<T>(z + row * zs + c0 + c));
    stf<T>(out + row * os + c0 + c, v * inv * w[c0 + c]);
  }
}

// The same for bf16 z and groups of up to 512 V columns in whole 16-byte pieces: one wave per (row, group), the products in
// registers between the two uses (one pass over y and z instead of two, no barrier).  4,096 x 4,096 in groups of 512: 52 us ->
// 23 us, 117 MB.
template <int V>
__global__ __launch_bounds__(256) void gated_group_rmsnorm_wave_kernel(const float* __restrict__ y, long ys, const bf16_t* __restrict__ z,
                                                                       long zs, const float* __restrict__ w, int gs, int ngroups, long n,
                                                                       float eps, bf16_t* __restrict__ out, long os) {
  const long job = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (job >= n) return;
  const long row = job / ngroups;
  const int lane = threadIdx.x & 63, c0 = (int)(job % ngroups) * gs;
  float v[V][8], ss = 0.f;
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = (lane + 64 * i) * 8;
    if (c < gs) {
      const floatx4* yp = reinterpret_cast<const floatx4*>(y + row * ys + c0 + c);
      const floatx4 a = yp[0], b = yp[1];
      float f[8];
      load8(z + row * zs + c0 + c, f);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        v[i][e] = (e < 4 ? a[e & 3] : b[e & 3]) * silu_f<false>(f[e]);
        ss += v[i][e] * v[i][e];
      }
    }
  }
  const float inv = 1.f / sqrtf(wave_sum(ss) / (float)gs + eps);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    const int c = (lane + 64 * i) * 8;
    if (c < gs) {
      const floatx4* wp = reinterpret_cast<const floatx4*>(w + c0 + c);
      const floatx4 a = wp[0], b = wp[1];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[i][e] *= inv * (e < 4 ? a[e & 3] : b[e & 3]);
      store8(out + row * os + c0 + c, v[i]);
    }
  }
}

// prompt portions (some sequence of the step has >= kChunkMin rows): the chunked MFMA kernel, for the step's other sequences too.  What
// decides in short portions and decode rows is the pass over the state, so the 64-token chunks lead there as well; us, chunks of 16 ->
// of 64, 64 heads of [64, 128]: 512 rows and 64 decode rows 322 -> 126, 8 and 64 177 -> 102, 64 portions of 8 170 -> 95, one of 8 14.4 -> 7.4.
// With up to 32 state columns that pass is short and a chunk's own work decides: there portions of up to 16 tokens stay with chunks of 16
// (16 heads of [128, 16]: 32 portions of 16 10.3 against 15.0, 8 and 64 decode rows 17.4 / 24.8; 17 tokens 7.5 / 7.1).
constexpr int kChunkMin = 8;

int cu_count() {
  static const int cus = [] {
    int dev = 0, n = 256;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 1) n = 256;
    return n;
  }();
  return cus;
}

template <typename T>
int scan_t(const T* xbc, long xs, const T* dtp, long dts, long rows, int S, int heads, int P, int N, int groups,
           const float* dt_bias, const float* A_log, const float* D, float* state, const int* cu, const int* slots,
           const int* positions, float* y, long ys, int max_len, hipStream_t st) {
  if (max_len >= kChunkMin) {
    dim3 cgrid(S, heads, (P + 63) / 64);
    if constexpr (sizeof(T) == 2) {
      // 16-byte loads of B, C and the state's rows, 8-byte ones of x, 16-byte stores of y
      const auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
      if (!(N <= 32 && max_len <= 16) && N % 8 == 0 && N <= 256 && xs < (1L << 25) && P % 4 == 0 && ((long)heads * P) % 8 == 0 && xs % 8 == 0 && ys % 4 == 0 && a16(xbc) && a16(state) && a16(y)) {
#define LK_CHUNK64(NR)                                                                                                             \
  do {                                                                                                                             \
    LK_SET_MAX_LDS((ssm_chunk_bf16_kernel<NR>), (ssm_chunk_lds<NR>()));                                                            \
    ssm_chunk_bf16_kernel<NR><<<cgrid, 256, ssm_chunk_lds<NR>(), st>>>(xbc, xs, dtp, dts, heads, P, N, groups, dt_bias, A_log, D,  \
                                                                      state, cu, slots, positions, y, ys);                        \
  } while (0)
#define LK_PIPE(NR)                                                                                                            \
  do {                                                                                                                         \
    LK_SET_MAX_LDS((ssm_pipe_kernel<NR>), (ssm_pipe_lds<NR>()));                                                               \
    ssm_pipe_kernel<NR><<<cgrid, 1024, ssm_pipe_lds<NR>(), st>>>(xbc, xs, dtp, dts, heads, P, N, groups, dt_bias, A_log, D,    \
                                                                 state, cu, slots, positions, y, ys);                          \
  } while (0)
        if (N <= 32) LK_CHUNK64(2);
        else if (N <= 64 && lk_ssm_piped(S, heads, P, N, max_len, rows, cu_count())) LK_PIPE(4);
        else if (N <= 64) LK_CHUNK64(4);
        else if (N <= 128) LK_PIPE(8);
        else LK_CHUNK64(16);   // (two chunks' columns of 256 do not fit the LDS)
#undef LK_CHUNK64
#undef LK_PIPE
        LK_CHECK_LAUNCH();
        return 0;
      }
    }
#define LK_CHUNK(NR)                                                                                                   \
  ssm_chunk_kernel<T, NR><<<cgrid, 256, 0, st>>>(xbc, xs, dtp, dts, heads, P, N, groups, dt_bias, A_log, D, state, cu, \
                                                 slots, positions, y, ys)
    if (N <= 16) LK_CHUNK(1);
    else if (N <= 32) LK_CHUNK(2);
    else if (N <= 64) LK_CHUNK(4);
    else if (N <= 128) LK_CHUNK(8);
    else if (N <= 256) LK_CHUNK(16);
    else return -1;
#undef LK_CHUNK
    LK_CHECK_LAUNCH();
    return 0;
  }
  if (max_len == 1 && N % 4 == 0 && N >= 16 && N <= 256 && (reinterpret_cast<uintptr_t>(state) & 15) == 0) {
    dim3 sgrid(S, heads);
    const bool vec = ((reinterpret_cast<uintptr_t>(xbc) | xs * sizeof(T) | (size_t)heads * P * sizeof(T)) & (4 * sizeof(T) - 1)) == 0;
#define LK_STEP_(LPR, RB, FULL)                                                                                                  \
  ssm_step_kernel<T, LPR, RB, FULL><<<sgrid, 256, 0, st>>>(xbc, xs, dtp, dts, heads, P, N, groups, dt_bias, A_log, D, state, cu, \
                                                           slots, positions, y, ys)
#define LK_STEP(LPR, RB)                                                       \
  do {                                                                         \
    if (vec && N == 4 * LPR && P % (64 / LPR * (RB)) == 0) LK_STEP_(LPR, (RB), true); \
    else LK_STEP_(LPR, (RB), false);                                           \
  } while (0)
    // rows per lane group of a pass: 8, or what gives all four waves a part of P.  One sequence, 32 heads of [64, 32] / [64, 64]:
    // 5.2 / 5.5 us with 8 (one and two of the four waves at work) -> 3.6 / 4.3; 16 sequences 6.1 / 7.1 -> 4.5 / 5.9
#define LK_STEPS(LPR)                                       \
  do {                                                      \
    if (P * LPR > 1024) LK_STEP(LPR, (LPR > 4 ? 8 : 4));    \
    else if (P * LPR > 512) LK_STEP(LPR, 4);                \
    else if (P * LPR > 256) LK_STEP(LPR, 2);                \
    else LK_STEP(LPR, 1);                                   \
  } while (0)
    if (N <= 16) LK_STEPS(4);
    else if (N <= 32) LK_STEPS(8);
    else if (N <= 64) LK_STEPS(16);
    else if (N <= 128) LK_STEPS(32);
    else LK_STEPS(64);
#undef LK_STEPS
#undef LK_STEP
#undef LK_STEP_
    LK_CHECK_LAUNCH();
    return 0;
  }
  dim3 grid(S, heads, (P + 15) / 16);
#define LK_SCAN(NR)                                                                                                 \
  ssm_scan_kernel<T, NR><<<grid, 256, 0, st>>>(xbc, xs, dtp, dts, heads, P, N, groups, dt_bias, A_log, D, state, cu, \
                                               slots, positions, y, ys)
  if (N <= 16) LK_SCAN(1);
  else if (N <= 32) LK_SCAN(2);
  else if (N <= 64) LK_SCAN(4);
  else if (N <= 128) LK_SCAN(8);
  else if (N <= 256) LK_SCAN(16);
  else return -1;
#undef LK_SCAN
  LK_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// Tokens per workgroup of the convolution, which walks them in fours behind each other: 4 or 8 where that leaves about a workgroup or two to a CU, 16
// where shorter tiles would not all be on the chip at once.  bf16 x 6,144 channels, us, what is taken / 8 / 32 tokens: one sequence of 60
// 5.5 / 6.6 / 13.5, of 300 5.9 / 7.0 / 13.8, of 900 11.0 / 11.0 / 15.1, of 2,000 16.1 / 16.5 / 17.1, four of 1,024 23.1 / 26.3 / 24.4, 32 of 200
// 37.8 / 40.8 / 35.9; x 2,048, four of 1,024 13.0 / 13.1 / 16.2; x 512 5.9 / 5.9 / 12.4
int lk_conv_rows(int S, int cblocks, int max_len, int cus) {
  const auto groups = [&](int r) { return (long)S * cblocks * ((max_len + r - 1) / r); };
  return groups(4) * 256 <= 300L * cus ? 4 : groups(8) * 256 <= 600L * cus ? 8 : kConvRows;
}

int lk_conv_silu(const void* u, long us, int C, int taps, const float* w, const float* bias, void* state, const int* cu,
                 const int* slots, const int* positions, int S, int max_len, void* out, long os, int act, int esz,
                 hipStream_t st) {
  if (S <= 0 || max_len <= 0) return 0;
  if (taps < 1 || taps > kMaxTaps || C <= 0) return -1;
  dim3 grid(S, (max_len + kConvRows - 1) / kConvRows, (C + 255) / 256), g2(S, (C + 255) / 256);
  const int ev = 16 / esz;
  const auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (taps <= 4 && C % ev == 0 && us % ev == 0 && os % ev == 0 && a16(u) && a16(out) && a16(state)) {
    const int cblocks = (C / ev + 255) / 256;
    const int rows = lk_conv_rows(S, cblocks, max_len, cu_count());
    dim3 gv(S, (max_len + rows - 1) / rows, cblocks);
#define LK_CONV(T, GR) conv_silu_vec_kernel<T, GR><<<gv, 256, 0, st>>>((const T*)u, us, C, taps, w, bias, (T*)state, cu, slots, positions, (T*)out, os, act, rows)
    if (max_len == 1) {
      if (esz == 2) LK_CONV(bf16_t, 1);
      else LK_CONV(float, 1);
    } else {
      if (esz == 2) LK_CONV(bf16_t, 4);
      else LK_CONV(float, 4);
    }
#undef LK_CONV
    LK_CHECK_LAUNCH();
    return 0;
  }
  if (esz == 2) {
    conv_silu_kernel<bf16_t><<<grid, 256, 0, st>>>((const bf16_t*)u, us, C, taps, w, bias, (const bf16_t*)state, cu,
                                                   slots, positions, (bf16_t*)out, os, act);
    LK_CHECK_LAUNCH();
    if (taps > 1) conv_state_kernel<bf16_t><<<g2, 256, 0, st>>>((const bf16_t*)u, us, C, taps, (bf16_t*)state, cu, slots, positions);
  } else {
    conv_silu_kernel<float><<<grid, 256, 0, st>>>((const float*)u, us, C, taps, w, bias, (const float*)state, cu, slots,
                                                  positions, (float*)out, os, act);
    LK_CHECK_LAUNCH();
    if (taps > 1) conv_state_kernel<float><<<g2, 256, 0, st>>>((const float*)u, us, C, taps, (float*)state, cu, slots, positions);
  }
  LK_CHECK_LAUNCH();
  return 0;
}

// Whether 64-token chunks of 33 - 128 state columns run as the pipeline of 16 waves, one workgroup to a CU, or (up to 64 columns, whose
// LDS leaves room for two) in four waves.  The pipeline shortens a sequence's chain; where workgroups queue for the CUs what decides is how long one
// of one chunk holds its place, and that is shorter in four waves.  us: the longest sequence alone, then each further round of workgroups with
// its average chunks; within 6 % (rms) of 126 launches (6 layouts of 33 - 64 columns, 1 - 257 sequences of 8 - 2,000 tokens), and the slower of the
// two for two of them (10 %).  32 heads of [64, 64], four waves / pipeline: 16 x 8 tokens 10.7 / 12.9, 64 x 8 33.5 / 42.6, 64 x 64 34.0 / 43.5,
// 64 x 128 55.4 / 62.3, 16 x 256 30.1 / 28.7, 8 x 512 42.4 / 25.9, 4 x 8 8.7 / 7.0, 8 and 256 decode rows 110 / 160, 512 and 64 65.2 / 60.8.
int lk_ssm_piped(int S, int heads, int P, int N, int max_len, long rows, int cus) {
  if (N > 64) return 1;
  const long wgs = (long)S * heads * ((P + 63) / 64);
  const double later = (max_len + 63) / 64 - 1, each = std::min(later, rows / 64.0 / S), queue = (double)((wgs + cus - 1) / cus - 1);
  return 7.0 + 2.2 * later + queue * (4.9 + 2.6 * each) < 8.1 + 4.4 * later + queue * (3.3 + 2.3 * each);
}

int lk_ssm_scan(const void* xbc, long xs, const void* dt, long dts, long rows, int S, int heads, int P, int N, int groups,
                const float* dt_bias, const float* A_log, const float* D, float* state, const int* cu, const int* slots,
                const int* positions, float* y, long ys, int max_len, int esz, hipStream_t st) {
  if (S <= 0) return 0;
  if (heads <= 0 || groups <= 0 || heads % groups || P <= 0 || N <= 0) return -1;
  return esz == 2 ? scan_t<bf16_t>((const bf16_t*)xbc, xs, (const bf16_t*)dt, dts, rows, S, heads, P, N, groups, dt_bias,
                                   A_log, D, state, cu, slots, positions, y, ys, max_len, st)
                  : scan_t<float>((const float*)xbc, xs, (const float*)dt, dts, rows, S, heads, P, N, groups, dt_bias, A_log,
                                  D, state, cu, slots, positions, y, ys, max_len, st);
}

int lk_gated_group_rmsnorm(const float* y, long ys, const void* z, long zs, const float* w, long rows, int inner,
                           int ngroups, float eps, void* out, long os, int esz, hipStream_t st) {
  if (rows <= 0) return 0;
  if (ngroups <= 0 || inner % ngroups) return -1;
  dim3 grid((unsigned)rows, ngroups);
  const int gs = inner / ngroups;
  const auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; };
  if (esz == 2 && gs % 8 == 0 && gs <= 2048 && ys % 4 == 0 && zs % 8 == 0 && os % 8 == 0 && a16(y) && a16(z) && a16(w) && a16(out)) {
    const long n = rows * ngroups;
#define LK_GGN(V)                                                                                                                    \
  gated_group_rmsnorm_wave_kernel<V><<<(unsigned)((n + 3) / 4), 256, 0, st>>>(y, ys, (const bf16_t*)z, zs, w, gs, ngroups, n, eps, \
                                                                              (bf16_t*)out, os)
    if (gs <= 512) LK_GGN(1);
    else if (gs <= 1024) LK_GGN(2);
    else LK_GGN(4);
#undef LK_GGN
  } else if (esz == 2)
    gated_group_rmsnorm_kernel<bf16_t><<<grid, 256, 0, st>>>(y, ys, (const bf16_t*)z, zs, w, inner / ngroups, eps,
                                                             (bf16_t*)out, os);
  else
    gated_group_rmsnorm_kernel<float><<<grid, 256, 0, st>>>(y, ys, (const float*)z, zs, w, inner / ngroups, eps,
                                                            (float*)out, os);
  LK_CHECK_LAUNCH();
  return 0;
}
