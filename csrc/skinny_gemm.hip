// K2, decode regime: Y[M,N] = X[M,K] . W[N,K]^T for M <= 128 rows (one decode
// token per running sequence), optionally with the SwiGLU epilogue fused.
//
// At M <= 128 every Llama linear is HBM-bound on the weight stream (O-proj at
// M=64: 32 MiB of W vs 2 GFLOP), so the kernel is built to keep all 256 CUs
// pulling W at full rate rather than to maximise MFMA reuse:
//   * block = 4 waves owning BN = 16*NTW output columns and ALL M rows; the
//     4 waves split the block's K range (intra-block split-K), so every W and
//     X element a block needs is loaded exactly once, straight to VGPRs in the
//     MFMA fragment layout (no LDS round trip on the way in: the "GEMV / M<=16"
//     rule of the CDNA4 playbook, extended to M<=128 because X is tiny and
//     L2-resident).
//   * blocks split K further (S-way) when N/BN alone would leave CUs idle
//     (QKV/O/down at 64-96 column tiles); S partial slabs go to an f32
//     workspace and a 16-B-vectorised reduce kernel sums them (with the SwiGLU
//     epilogue when fused).  gate_up (448 tiles) and the LM head run S=1 with
//     the epilogue in the GEMM itself.
//   * W is read with non-temporal loads (streamed once; keeps X in L2), one
//     64-deep K step of fragments in flight under the current step's MFMAs.
//   * v_mfma_f32_16x16x32_bf16: lane l holds A = X[16m + (l&15)][k0 + 8(l>>4) + j]
//     and B = W[n0 + (l&15)][k0 + 8(l>>4) + j]: both are 16-B row-contiguous
//     loads, two K sub-steps cover each 128-B line of W exactly.
//   * the 4 waves' f32 tiles are summed through LDS (rows padded by 4 floats so
//     the 4 lane groups hit different banks) and stored coalesced.
// SwiGLU fusion: block t owns gate columns [t*BN/2, (t+1)*BN/2) and the matching
// up columns I + [...]; out[m][j] = bf16(silu(bf16(g)) ) * bf16(u), rounded like
// the unfused linear -> silu_mul path (bit-identical to it).
#include <algorithm>
#include <cstdlib>
#include <map>
#include <mutex>
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace {

constexpr int kSkW = 4;  // waves per block

LK_DEVICE float silu_f(float x) { return x / (1.f + __expf(-x)); }
LK_DEVICE float rbf(float x) { return bf2f(f2bf(x)); }

constexpr int kSysCoherent = 1 | 16;  // buffer cache policy sc0 | sc1: past L1 and L2

// Fused split-K tail of the weight-streaming GEMM (kind != 0).  Every split workgroup writes its
// f32 partial through to memory and takes a ticket; the LAST one to finish reduces the slabs
// itself, so no reduce kernel is launched after the GEMM (at decode sizes a reduce launch is a
// ~5 us step of the critical path per projection):
//   kind 1: RoPE + paged-KV write, one ticket per column tile = one head (BN == D): the qkv rows
//           exactly as lk_splitk_rope_kv leaves them (q rotated, k rotated in the cache and in
//           the row only with write_k_inplace, v copied);
//   kind 2: residual add + RMSNorm, one ticket for the whole grid (few rows: the last workgroup
//           normalises every row), exactly as lk_splitk_rmsnorm.
// Tickets are zero-initialised int32 counters reset by their last taker.
struct WsTail {
  int kind = 0;
  int* tickets = nullptr;
  bf16_t* out = nullptr;  // 1: qkv rows; 2: normed rows
  long os = 0;
  const int* positions = nullptr;
  const float* cos_sin = nullptr;
  int Hq = 0, Hkv = 0, D = 0;
  bf16_t* kc = nullptr;
  bf16_t* vc = nullptr;
  const int* slots = nullptr;
  int BS = 1, neox = 0, write_k_inplace = 0;
  bf16_t* residual = nullptr;
  long rs = 0;
  const bf16_t* norm_w = nullptr;
  float eps = 0.f;
};

// Consumer-side prologue of the weight-streaming GEMM (kind != 0, <= 64 rows): before its K walk
// every workgroup computes the X rows of its K slice itself and stages them from the scratch
// rows `x` it wrote, so the launch that would have produced X disappears from the decode step
// (its W prefetch is issued before the prologue and flies under it):
//   kind 1: x = RMSNorm(bf16(sum of the producer's split-K slabs) + res) * gamma -- exactly the
//           rmsnorm_kernel<_, 4, S> arithmetic (256 threads slicing the row the same way, same
//           block_sum), so the values are bit-identical to lk_splitk_rmsnorm; workgroup 0 also
//           writes the summed residual row(s) to res_out (a buffer other than res: the other
//           workgroups still read res);
//   kind 2: the flash-decoding merge of a split-K paged-decode step's partials, exactly as
//           decode_reduce_kernel, for the rows with more than one split (the others the
//           attention kernel wrote into x itself).
struct WsPro {
  int kind = 0;
  bf16_t* x = nullptr;  // [M, K] scratch rows (row stride K): written here, then staged as X
  const float* part = nullptr;  // 1: producer slabs [S][M][K]
  int S = 0;
  long slab = 0;
  const bf16_t* res = nullptr;
  bf16_t* res_out = nullptr;
  long rs = 0;  // row stride of res and res_out
  const bf16_t* gamma = nullptr;
  float eps = 0.f;
  const float* po = nullptr;   // 2: [(row * Hq + qh) * max_splits + s][D]
  const float* pml = nullptr;  // 2: [(row * Hq + qh) * max_splits + s][2]
  const int* ctx = nullptr;
  int Hq = 0, D = 0, max_splits = 0, split = 0;
};

template <int KIND>
LK_DEVICE void ws_prologue(const WsPro& pr, int M, int K, long kbase, int ks) {
  if constexpr (KIND == 1) {
    __shared__ float red[4];
    const int nvec = K >> 3;
    for (int m = 0; m < M; ++m) {
      float v[4][8];
      float ss = 0.f;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = threadIdx.x + i * 256;
        if (c < nvec) {
          const float* pp = pr.part + (long)m * K + c * 8;
          floatx4 a = *reinterpret_cast<const floatx4*>(pp), b = *reinterpret_cast<const floatx4*>(pp + 4);
          for (int q = 1; q < pr.S; ++q) {
            a += *reinterpret_cast<const floatx4*>(pp + q * pr.slab);
            b += *reinterpret_cast<const floatx4*>(pp + q * pr.slab + 4);
          }
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            v[i][j] = bf2f(f2bf(a[j]));
            v[i][j + 4] = bf2f(f2bf(b[j]));
          }
          float r[8];
          load8(pr.res + (long)m * pr.rs + c * 8, r);
#pragma unroll
          for (int j = 0; j < 8; ++j) v[i][j] = bf2f(f2bf(v[i][j] + r[j]));
          if (blockIdx.x == 0) store8(pr.res_out + (long)m * pr.rs + c * 8, v[i]);
#pragma unroll
          for (int j = 0; j < 8; ++j) ss += v[i][j] * v[i][j];
        }
      }
      ss = block_sum<4>(ss, red);
      const float inv = rsqrtf(ss / (float)K + pr.eps);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int c = threadIdx.x + i * 256;
        if (c < nvec && c * 8 >= kbase && c * 8 < kbase + ks) {
          float g[8], y[8];
          load8(pr.gamma + c * 8, g);
#pragma unroll
          for (int j = 0; j < 8; ++j) y[j] = bf2f(f2bf(v[i][j] * inv)) * g[j];
          store8(pr.x + (long)m * K + c * 8, y);
        }
      }
    }
  } else if constexpr (KIND == 2) {
    for (int m = 0; m < M; ++m) {
      const int nsplit = max(0, min((pr.ctx[m] + pr.split - 1) / pr.split, pr.max_splits));
      if (nsplit <= 1) continue;  // (uniform) the attention kernel wrote this row into x
      for (int e = threadIdx.x; e < ks; e += 256) {
        const long col = kbase + e;
        const int qh = (int)(col / pr.D), d = (int)(col - (long)qh * pr.D);
        const long base = ((long)m * pr.Hq + qh) * pr.max_splits;
        float Mx = -INFINITY;
        for (int q = 0; q < nsplit; ++q) Mx = fmaxf(Mx, pr.pml[(base + q) * 2]);
        if (Mx == -INFINITY) Mx = 0.f;
        float den = 0.f, num = 0.f;
        for (int q = 0; q < nsplit; ++q) {
          const float f = exp2f(pr.pml[(base + q) * 2] - Mx);
          den += f * pr.pml[(base + q) * 2 + 1];
          num += f * pr.po[(base + q) * pr.D + d];
        }
        pr.x[(long)m * K + col] = f2bf(den > 0.f ? num / den : 0.f);
      }
    }
  }
}

// 8 consecutive columns of one row: the S slabs summed in slab order, rounded to bf16 (the values
// the unfused reduce stores); partials read past L1 / L2 (other workgroups wrote them through)
LK_DEVICE void tail_ld8(__amdgpu_buffer_rsrc_t prs, int S, long slab, long off, float* f) {
  floatx4 a = floatx4{0.f, 0.f, 0.f, 0.f}, b = a;
  for (int q0 = 0; q0 < S; q0 += 4) {  // 4 slabs in flight at a time (registers: the tail shares the kernel's)
    floatx4 pa[4], pb[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q0 + q < S) {
        const unsigned o = (unsigned)((off + (q0 + q) * slab) * 4);
        pa[q] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(prs, o, 0, kSysCoherent));
        pb[q] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(prs, o + 16, 0, kSysCoherent));
      }
#pragma unroll
    for (int q = 0; q < 4; ++q)
      if (q0 + q < S) {
        a += pa[q];
        b += pb[q];
      }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    f[j] = bf2f(f2bf(a[j]));
    f[j + 4] = bf2f(f2bf(b[j]));
  }
}

// kind 1: head = column tile t of the fused [(Hq + 2 Hkv) * D] projection, all M rows
LK_DEVICE void tail_rope_kv(const WsTail& tl, __amdgpu_buffer_rsrc_t prs, int S, int M, long ld, int head) {
  const int D = tl.D, half = D >> 1;
  const long slab = (long)M * ld;
  const bool rot = head < tl.Hq + tl.Hkv;
  const int ipr = rot ? (tl.neox ? (D >> 4) : (D >> 3)) : (D >> 3);
  const bool is_k = head >= tl.Hq && rot;
  const bool store_src = !is_k || tl.write_k_inplace;
  for (int it = threadIdx.x; it < M * ipr; it += blockDim.x) {
    const int row = it / ipr, v = it - row * ipr;
    bf16_t* hp = tl.out + (long)row * tl.os + (long)head * D;
    const long pbase = (long)row * ld + (long)head * D;
    const int slot = tl.slots ? tl.slots[row] : -1;
    const long blk = slot >= 0 ? slot / tl.BS : 0;
    const int off = slot >= 0 ? slot % tl.BS : 0;
    if (!rot) {  // V: copy into the row and the cache
      const int c = v * 8, h = head - tl.Hq - tl.Hkv;
      float f[8];
      tail_ld8(prs, S, slab, pbase + c, f);
      store8(hp + c, f);
      if (tl.vc && slot >= 0) store8(tl.vc + ((blk * tl.Hkv + h) * tl.BS + off) * D + c, f);
      continue;
    }
    const float* cs = tl.cos_sin + (long)tl.positions[row] * D;  // [cos(D/2) | sin(D/2)]
    bf16_t* kdst = (is_k && tl.kc && slot >= 0) ? tl.kc + ((blk * tl.Hkv + (head - tl.Hq)) * tl.BS + off) * D : nullptr;
    if (tl.neox) {
      const int i0 = v * 8;
      float x1[8], x2[8], y1[8], y2[8];
      tail_ld8(prs, S, slab, pbase + i0, x1);
      tail_ld8(prs, S, slab, pbase + half + i0, x2);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const float c = cs[i0 + j], sn = cs[half + i0 + j];
        y1[j] = rot_lo(x1[j], x2[j], c, sn);
        y2[j] = rot_hi(x1[j], x2[j], c, sn);
      }
      store8(hp + i0, store_src ? y1 : x1);
      store8(hp + half + i0, store_src ? y2 : x2);
      if (kdst) {
        store8(kdst + i0, y1);
        store8(kdst + half + i0, y2);
      }
    } else {
      const int e0 = v * 8;  // elements e0..e0+7 = pairs e0/2 .. e0/2+3
      float x[8], y[8];
      tail_ld8(prs, S, slab, pbase + e0, x);
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const float c = cs[(e0 >> 1) + p], sn = cs[half + (e0 >> 1) + p];
        y[2 * p] = rot_lo(x[2 * p], x[2 * p + 1], c, sn);
        y[2 * p + 1] = rot_hi(x[2 * p], x[2 * p + 1], c, sn);
      }
      store8(hp + e0, store_src ? y : x);
      if (kdst) store8(kdst + e0, y);
    }
  }
}

// kind 2: rows 0..M-1 of N = ld columns: residual += bf16(sum of slabs); out = RMSNorm(residual) * w
LK_DEVICE void tail_rmsnorm(const WsTail& tl, __amdgpu_buffer_rsrc_t prs, int S, int M, long ld, float* red) {
  const int nvec = (int)(ld >> 3);
  const long slab = (long)M * ld;
  const int nw = blockDim.x >> 6, lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  for (int row = 0; row < M; ++row) {
    float ss = 0.f;
    for (int c = threadIdx.x; c < nvec; c += blockDim.x) {
      float v[8], r[8];
      tail_ld8(prs, S, slab, (long)row * ld + c * 8, v);
      bf16_t* rr = tl.residual + (long)row * tl.rs + c * 8;
      load8(rr, r);
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        v[j] = bf2f(f2bf(v[j] + r[j]));  // the new residual stream: the bf16-rounded sum
        ss += v[j] * v[j];
      }
      store8(rr, v);
    }
    ss = wave_sum(ss);
    __syncthreads();  // (the previous row's reads of red are done)
    if (lane == 0) red[wv] = ss;
    __syncthreads();
    float tot = 0.f;
    for (int i = 0; i < nw; ++i) tot += red[i];
    const float inv = rsqrtf(tot / (float)ld + tl.eps);
    for (int c = threadIdx.x; c < nvec; c += blockDim.x) {
      float v[8], g[8], y[8];
      load8(tl.residual + (long)row * tl.rs + c * 8, v);  // (this thread's own stores above)
      load8(tl.norm_w + c * 8, g);
#pragma unroll
      for (int j = 0; j < 8; ++j) y[j] = v[j] * inv * g[j];
      store8(tl.out + (long)row * tl.os + c * 8, y);
    }
  }
}

// after the epilogue, by ALL threads of the workgroup (uniform control flow: it has barriers).
// lds: the kernel's dynamic LDS, dead once the K loop is done (no static LDS here: the ring
// already fills the 160 KB)
__attribute__((noinline)) __device__ void ws_tail(const WsTail& tl, float* part, int M, long ld, int S, int t, int n_tiles, unsigned char* lds) {
  int* is_last = reinterpret_cast<int*>(lds);
  float* red = reinterpret_cast<float*>(lds + 64);
  __builtin_amdgcn_s_waitcnt(0);  // this thread's write-through partial stores acknowledged
  __syncthreads();                // (and every wave is done with the LDS ring)
  if (threadIdx.x == 0) {
    int* tk = tl.tickets + (tl.kind == 1 ? t : 0);
    const int need = tl.kind == 1 ? S : S * n_tiles;
    const int old = __hip_atomic_fetch_add(tk, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    const int last = old == need - 1;
    if (last) __hip_atomic_store(tk, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    *is_last = last;
  }
  __syncthreads();
  if (!*is_last) return;
  const long bytes = (long)S * M * ld * 4;
  const __amdgpu_buffer_rsrc_t prs =
      __builtin_amdgcn_make_buffer_rsrc((void*)part, (short)0, (int)min(bytes, 0x7FFFFFF0L), 0x00020000);
  if (tl.kind == 1) tail_rope_kv(tl, prs, S, M, ld, t);
  else tail_rmsnorm(tl, prs, S, M, ld, red);
}

template <int MT, int NTW, bool SWIGLU>
__global__ __launch_bounds__(256) void skinny_gemm_kernel(
    const bf16_t* __restrict__ X, long ldx, const bf16_t* __restrict__ W, int M, int K, int ks,
    int n_tiles, int swiglu_I, bf16_t* __restrict__ out, long ldo, float* __restrict__ part,
    long part_ld) {
  constexpr int BN = 16 * NTW;
  constexpr int ROWS = 16 * MT;
  constexpr int LDR = BN + 4;
  extern __shared__ float red[];  // [kSkW][ROWS][LDR]

  const int t = blockIdx.x % n_tiles, s = blockIdx.x / n_tiles;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int kw = ks / kSkW;
  const long kbase = (long)s * ks + (long)w * kw + 8 * g;

  auto ncol = [&](int c) -> long {  // global W row (output column) of column tile c, lane r
    if constexpr (SWIGLU) {
      constexpr int H = NTW / 2;
      return c < H ? (long)t * (BN / 2) + 16 * c + r : (long)swiglu_I + (long)t * (BN / 2) + 16 * (c - H) + r;
    } else {
      return (long)t * BN + 16 * c + r;
    }
  };

  const bf16_t* wp[NTW];
#pragma unroll
  for (int c = 0; c < NTW; ++c) wp[c] = W + ncol(c) * K + kbase;
  const bf16_t* xp[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int row = min(16 * m + r, M - 1);
    xp[m] = X + (long)row * ldx + kbase;
  }

  floatx4 acc[MT][NTW];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < NTW; ++c) acc[m][c] = floatx4{0.f, 0.f, 0.f, 0.f};

  short8 wa[NTW][2], xa[MT][2], wb[NTW][2], xb[MT][2];
  auto load = [&](short8 (&wf)[NTW][2], short8 (&xf)[MT][2], int k) {
#pragma unroll
    for (int c = 0; c < NTW; ++c)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        wf[c][h] = __builtin_nontemporal_load(reinterpret_cast<const short8*>(wp[c] + k + 32 * h));
#pragma unroll
    for (int m = 0; m < MT; ++m)
#pragma unroll
      for (int h = 0; h < 2; ++h) xf[m][h] = *reinterpret_cast<const short8*>(xp[m] + k + 32 * h);
    __builtin_amdgcn_sched_barrier(0);  // keep the prefetch issued ahead of the MFMAs below
  };
  auto compute = [&](const short8 (&wf)[NTW][2], const short8 (&xf)[MT][2]) {
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int c = 0; c < NTW; ++c)
          acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xf[m][h], wf[c][h], acc[m][c], 0, 0, 0);
  };

  // ping-pong register sets, no copies (a copy of a just-loaded register makes the
  // compiler wait for that load and serialises the stream): step i+1 is in flight
  // under step i's MFMAs.
  const int nsteps = kw / 64;
  load(wa, xa, 0);
  int i = 0;
  for (; i + 2 < nsteps; i += 2) {
    load(wb, xb, (i + 1) * 64);
    compute(wa, xa);
    load(wa, xa, (i + 2) * 64);
    compute(wb, xb);
  }
  if (nsteps - i == 2) {
    load(wb, xb, (i + 1) * 64);
    compute(wa, xa);
    compute(wb, xb);
  } else {
    compute(wa, xa);
  }

  // ---- intra-block split-K reduction through LDS
  float* mine = red + w * ROWS * LDR;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int c = 0; c < NTW; ++c)
#pragma unroll
      for (int i = 0; i < 4; ++i) mine[(16 * m + 4 * g + i) * LDR + 16 * c + r] = acc[m][c][i];
  __syncthreads();

  auto sum4 = [&](int row, int col) -> floatx4 {
    floatx4 v = *reinterpret_cast<const floatx4*>(red + row * LDR + col);
#pragma unroll
    for (int ww = 1; ww < kSkW; ++ww) {
      const floatx4 u = *reinterpret_cast<const floatx4*>(red + ww * ROWS * LDR + row * LDR + col);
      v += u;
    }
    return v;
  };

  const bool split = part != nullptr;
  if (SWIGLU && !split) {
    constexpr int HB = BN / 2, Q = HB / 4;
    for (int idx = threadIdx.x; idx < ROWS * Q; idx += 256) {
      const int row = idx / Q, c4 = (idx % Q) * 4;
      if (row >= M) continue;
      const floatx4 gv = sum4(row, c4), uv = sum4(row, HB + c4);
      float y[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) y[i] = rbf(silu_f(rbf(gv[i]))) * rbf(uv[i]);
      uint2 pk;
      pk.x = pack_bf2(y[0], y[1]);
      pk.y = pack_bf2(y[2], y[3]);
      *reinterpret_cast<uint2*>(out + (long)row * ldo + (long)t * HB + c4) = pk;
    }
  } else {
    constexpr int Q = BN / 4;
    for (int idx = threadIdx.x; idx < ROWS * Q; idx += 256) {
      const int row = idx / Q, c4 = (idx % Q) * 4;
      if (row >= M) continue;
      const floatx4 v = sum4(row, c4);
      if (split) {
        long n;
        if constexpr (SWIGLU) {
          n = c4 < BN / 2 ? (long)t * (BN / 2) + c4 : (long)swiglu_I + (long)t * (BN / 2) + c4 - BN / 2;
        } else {
          n = (long)t * BN + c4;
        }
        *reinterpret_cast<floatx4*>(part + (long)s * M * part_ld + (long)row * part_ld + n) = v;
      } else {
        uint2 pk;
        pk.x = pack_bf2(v[0], v[1]);
        pk.y = pack_bf2(v[2], v[3]);
        *reinterpret_cast<uint2*>(out + (long)row * ldo + (long)t * BN + c4) = pk;
      }
    }
  }
}

// sum S f32 slabs [S][M][ld] -> bf16 out (optionally SwiGLU over [gate | up])
template <bool SWIGLU>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(const float* __restrict__ part, int S, int M,
                                                            long ld, int n_out, int swiglu_I,
                                                            bf16_t* __restrict__ out, long ldo) {
  const int q = n_out / 4;
  const long total = (long)M * q;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < total; i += (long)gridDim.x * 256) {
    const int row = (int)(i / q), c4 = (int)(i % q) * 4;
    const float* p = part + (long)row * ld + c4;
    floatx4 v = *reinterpret_cast<const floatx4*>(p);
    for (int s = 1; s < S; ++s) v += *reinterpret_cast<const floatx4*>(p + (long)s * M * ld);
    float y[4];
    if constexpr (SWIGLU) {
      floatx4 u = *reinterpret_cast<const floatx4*>(p + swiglu_I);
      for (int s = 1; s < S; ++s) u += *reinterpret_cast<const floatx4*>(p + (long)s * M * ld + swiglu_I);
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = rbf(silu_f(rbf(v[j]))) * rbf(u[j]);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) y[j] = v[j];
    }
    uint2 pk;
    pk.x = pack_bf2(y[0], y[1]);
    pk.y = pack_bf2(y[2], y[3]);
    *reinterpret_cast<uint2*>(out + (long)row * ldo + c4) = pk;
  }
}

// ---------------------------------------------------------------------------------
// Weight-streaming GEMM for 64 < M <= 256 rows ("wsgemm").  The fragment-shaped loads
// of skinny_gemm_kernel touch 16 rows x 64 B per wave instruction, which caps the
// per-CU load rate once X (re-read by every column block) grows with M.  Here both
// operands are staged through LDS by 16-B LDS-DMA: every wave
// instruction moves 8 rows x one full 128-B line, lane-linear into LDS, with the
// (row>>1)&7 XOR chunk swizzle applied on the SOURCE address so the MFMA fragment
// reads (ds_read_b128, 16 rows x 16 B per lane group) are bank-conflict free.
//   * block = 4 waves, tile = all M rows (16*MT) x BN columns, BK = 64 per stage, as many stages as 160 KB of LDS hold, the walk below;
//   * W rows are streamed once with the non-temporal policy;
//   * split-K over blocks (S) when N/BN leaves CUs idle; partial slabs -> the same
//     reduce / SwiGLU kernel as skinny_gemm; S = 1 writes bf16 (or SwiGLU) directly.
// What bounds it: at 128 rows the chip's matrix rate (20 us for 28672 x 4096) is half of the weight's stream (38 us at 6.1 TB/s), so
// neither hides a wait that the other has.  A CU takes 125 - 150 KB/us out of its L2 (X) and, with 256 of them at it, 24 from memory (W);
// four waves with 8 KB each in flight reach that.  Waves that each took all columns of a quarter of the rows read 20 fragments a stage in three
// groups, each waited for before its MFMAs, 0.64 us a stage with W out of L2; a 2 x 2 grid of waves reads 16, under the MFMAs of the stage
// before: 0.5.  Cold, us (one ring / loader waves before -> now): 120 rows: gate / up 28672 x 4096 47.9 / 48.4 -> 46.7, 32768 x 4096
// 51.0 / 48.8 -> 47.7, 6144 x 4096 15.6 / 16.2 -> 14.5, 4096 x 4096 12.5 / 13.2 -> 11.7, 4096 x 14336 27.9 / 27.7 -> 27.5; 256 rows:
// 77 / 71 -> 59, 82 / 77 -> 62, 22.5 / 23.0 -> 20.0, 18.0 / 19.6 -> 17.5, 40.5 / 38.7 -> 34.7.
template <int N>
LK_DEVICE void wait_vmcnt() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}

typedef __attribute__((address_space(3))) void* lds_void_ptr;

typedef const __attribute__((address_space(3))) short8* lds_frag_t;
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

LK_DEVICE int wsz(int row) { return (row >> 1) & 7; }
template <class Fn, int... I>
LK_DEVICE void ws_unroll_impl(Fn&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class Fn>
LK_DEVICE void ws_unroll(Fn&& f) {
  ws_unroll_impl(f, std::make_integer_sequence<int, N>{});
}
LK_DEVICE unsigned ws_rfl(unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); }
LK_DEVICE u32x4_t ws_srd(const void* p, long bytes) {  // buffer descriptor words, wave-uniform
  const unsigned long a = reinterpret_cast<unsigned long>(p);
  return u32x4_t{ws_rfl((unsigned)a), ws_rfl((unsigned)(a >> 32)), ws_rfl((unsigned)max(0L, min(bytes, 0xFFFFFFF0L))), 0x00020000u};
}

// A byte offset behind every operand's range, also with an offset along K (less than 32 MB) on top of it.  Host: ws_too_far.
constexpr unsigned kWsPast = 0xFC000000u;

// ring depth: as many stages as 160 KB of LDS hold
// (PRO: a WsPro prologue computes X first -- the LDS ring leaves room for its static scratch)
constexpr int ws_stages_pro(int MT, int BN, int PRO) {
  const int sb = (16 * MT + BN) * 128;
  const int n = (163840 - (PRO ? 1024 : 0)) / sb;
  return n > 8 ? 8 : (n < 3 ? 3 : n);
}

// The walk of one workgroup over its stages (64 columns of K): four waves in a 2 x 2 grid, a wave (ROWS / 2) rows x (BN / 2) columns.
// The fragments of the next stage go to a second set of registers under this stage's MFMAs, so a stage is one barrier that says at once
// "the next stage has landed" and "everyone holds this one in registers: its slot may be requested again", and no MFMA waits for LDS.
// Stages past the last come from a descriptor without range (zeros nobody uses), so that every stage is the same code.
// NSX / NSW: stages of X's and of W's ring.  LOADERS waves more than the four request W (0: the four do).
template <int MT, int BN, bool SWIGLU, int NSX, int NSW, int LOADERS>
struct WsWalk {
  static constexpr int MW = MT / 2, NW = BN / 32;                     // 16 x 16 tiles of a wave; also the four waves' LDS-DMA pieces (8 rows) per stage
  static constexpr int PW = LOADERS ? BN / 8 / LOADERS : NW;          // W pieces per stage of a wave that requests them
  static constexpr int WSTEP = LOADERS ? LOADERS : 4;                 // its pieces are so many apart
  static constexpr int XB = 16 * MT * 128, WB = BN * 128, L = MW + NW;
  static constexpr int NM = 2 * MW * NW, NR = 2 * L;                  // MFMAs and fragment reads of a wave and stage
  static constexpr int OPS = LOADERS ? MW : L;                        // requests per stage of one of the four
  static_assert(LOADERS || NSX == NSW, "one ring");
  static_assert((NSX - 1) * OPS < 64 && (NSW - 1) * PW < 64, "vmcnt");
  unsigned xo[MW], wo[PW];
  unsigned ldsx, ldsw, bx[2], bw[2];
  u32x4_t xs, ws[2];
  int nst, last, at, kofs;      // at: the next stage to request; kofs: its byte offset in a row
  floatx4 acc[MW][NW];
  short8 fx[2][2][MW], fw[2][2][NW];

  // first row of column tile n in the tile's W rows as they lie in LDS, from the wave's first; SwiGLU: gate rows, then up rows
  static constexpr int col(int n) { return SWIGLU ? (n < NW / 2 ? 16 * n : BN / 2 + 16 * (n - NW / 2)) : 16 * n; }
  // piece i of a wave that requests W is one of up rows
  static constexpr bool up(int i) { return SWIGLU && i >= PW / 2; }

  // wave q of those that request W
  LK_DEVICE void begin(const unsigned char* smem, const bf16_t* X, long ldx, const bf16_t* W, const bf16_t* W2, long wrows, int M, int K,
                       long kbase, int stages, int rot) {
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 15, g = lane >> 4, lrow = lane >> 3, q = LOADERS ? w - 4 : w;
    // from the first row's start to the last one's end, whatever lies between two rows' starts (0: one row M times; less than K: windows)
    xs = ws_srd(X + kbase, ((long)(M - 1) * ldx + K - kbase) * 2);
    ws[0] = ws_srd(W + kbase, wrows * K * 2 - kbase * 2);
    ws[1] = SWIGLU ? ws_srd(W2 + kbase, wrows * K * 2 - kbase * 2) : ws[0];
    nst = stages;
    at = 0;
    last = stages * 128;
    kofs = rot * 128;
    // piece p: rows 8 p .., lane l the chunk (l & 7) ^ ((row >> 1) & 7) of row l >> 3; a wave's pieces are an even number apart
    const int ch = (lane & 7) ^ (lrow >> 1);
#pragma unroll
    for (int i = 0; i < MW; ++i) {
      const int row = 8 * (4 * i + w) + lrow;   // rows past M: zeros
      xo[i] = row < M ? (unsigned)row * (unsigned)(ldx * 2) + (unsigned)((ch ^ (4 * (w & 1))) * 16) : kWsPast;
    }
#pragma unroll
    for (int i = 0; i < PW; ++i)
      wo[i] = (unsigned)(8 * (WSTEP * (SWIGLU ? i % (PW / 2) : i) + q) + lrow) * (unsigned)(K * 2) + (unsigned)((ch ^ (4 * (q & 1))) * 16);
    const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((lds_void_ptr)smem);
    ldsx = lds0 + w * 1024;
    ldsw = lds0 + NSX * XB + q * 1024;
    const int wr = w >> 1, wc = w & 1;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned b = lds0 + (((4 * h + g) ^ wsz(r)) << 4) + r * 128;
      bx[h] = b + wr * (8 * MT) * 128;
      bw[h] = b + NSX * XB + wc * (SWIGLU ? BN / 4 : BN / 2) * 128;
    }
#pragma unroll
    for (int m = 0; m < MW; ++m)
#pragma unroll
      for (int n = 0; n < NW; ++n) acc[m][n] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  // piece i of the stage to request next, into the ring slot at `slot`
  template <int I>
  LK_DEVICE void dma_x(unsigned slot) {
    asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
                 ::"v"(xo[I]), "s"(xs), "s"(kofs), "s"(ldsx + slot), "i"(I * 4096) : "memory", "m0", "scc");
  }
  template <int I>
  LK_DEVICE void dma_w(unsigned slot) {
    asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen nt lds"
                 ::"v"(wo[I]), "s"(ws[up(I)]), "s"(kofs), "s"(ldsw + slot), "i"(I * WSTEP * 1024) : "memory", "m0", "scc");
  }
  LK_DEVICE void advance() {   // to the stage after `at`: past the last no descriptor has a range
    kofs = kofs + 128 == last ? 0 : kofs + 128;
    if (++at == nst) xs.z = ws[0].z = ws[1].z = 0;
  }
  template <bool X, bool W>
  LK_DEVICE void request(unsigned xslot, unsigned wslot) {
    if constexpr (X) ws_unroll<MW>([&](auto j_t) { dma_x<decltype(j_t)::value>(xslot); });
    if constexpr (W) ws_unroll<PW>([&](auto j_t) { dma_w<decltype(j_t)::value>(wslot); });
  }
  // fragment j of the stage whose reads start at ax / aw: the first half of K, then the second; X, then W
  template <int P>
  LK_DEVICE void read(int j, const unsigned (&ax)[2], const unsigned (&aw)[2]) {
    const int h = j / L, q = j % L;
    if (q < MW) fx[P][h][q] = *reinterpret_cast<lds_frag_t>(ax[h] + q * 2048);
    else fw[P][h][q - MW] = *reinterpret_cast<lds_frag_t>(aw[h] + col(q - MW) * 128);
  }
  struct Slots { unsigned x, w; };
  LK_DEVICE static void step(Slots& s) {
    s.x = s.x + XB == (unsigned)(NSX * XB) ? 0 : s.x + XB;
    s.w = s.w + WB == (unsigned)(NSW * WB) ? 0 : s.w + WB;
  }
  LK_DEVICE void addresses(Slots s, unsigned (&ax)[2], unsigned (&aw)[2]) const {
#pragma unroll
    for (int h = 0; h < 2; ++h) {   // (opaque: the rest of every address stays the instruction's immediate)
      ax[h] = bx[h] + s.x;
      aw[h] = bw[h] + s.w;
      asm volatile("" : "+v"(ax[h]), "+v"(aw[h]));
    }
  }
  // stage in register set P; cur: its slots, requested again; nxt: the next one's, read into the other set
  template <int P>
  LK_DEVICE void stage(Slots cur, Slots nxt) {
    unsigned ax[2], aw[2];
    addresses(nxt, ax, aw);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4));   // lgkmcnt(0)
    wait_vmcnt<(NSX - 2) * OPS>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    ws_unroll<NM>([&](auto i_t) {
      constexpr int i = decltype(i_t)::value, h = i / (MW * NW), m = i % MW, n = i / MW % NW;
      // the reads over the first two thirds of the MFMAs, the requests over all
#pragma unroll
      for (int j = 0; j < NR; ++j)
        if (j * NM * 2 / (NR * 3) == i) read<P ^ 1>(j, ax, aw);
      ws_unroll<OPS>([&](auto j_t) {
        constexpr int j = decltype(j_t)::value;
        if constexpr (j * NM / OPS + (NM > OPS ? 1 : 0) == i) {
          if constexpr (j < MW) dma_x<j>(cur.x);
          else dma_w<j - MW>(cur.w);
        }
      });
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (LOADERS) asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc[m][n]) : "v"(fw[P][h][n]), "v"(fx[P][h][m]));
      else asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc[m][n]) : "v"(fw[P][h][n]), "v"(fx[P][h][m]));
      __builtin_amdgcn_sched_barrier(0);
    });
    advance();
  }
  // the first NSX stages have been requested, in order, into the slots from 0 on (W's by the loaders)
  LK_DEVICE void walk() {
    wait_vmcnt<(NSX - 1) * OPS>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    Slots cur{0, 0}, nxt{0, 0};
    unsigned ax[2], aw[2];
    addresses(cur, ax, aw);
#pragma unroll
    for (int j = 0; j < NR; ++j) read<0>(j, ax, aw);
    step(nxt);
    for (int st = 0;; st += 2) {
      stage<0>(cur, nxt);
      cur = nxt;
      step(nxt);
      if (st + 1 >= nst) break;
      stage<1>(cur, nxt);
      cur = nxt;
      step(nxt);
      if (st + 2 >= nst) break;
    }
    wait_vmcnt<0>();   // the last requests land before the workgroup's LDS is used again or released
    // (the MFMAs are asm: the wait between the last ones and the first use of their results is ours)
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
#pragma unroll
    for (int m = 0; m < MW; ++m)
#pragma unroll
      for (int n = 0; n < NW; ++n) {
        if constexpr (LOADERS) asm volatile("" : "+v"(acc[m][n]));
        else asm volatile("" : "+a"(acc[m][n]));
      }
  }
  // a loader wave's part: as many barriers as walk() has
  LK_DEVICE void load() {
    for (int p = 0; p < NSW; ++p) {
      request<false, true>(0, p * WB);
      advance();
    }
    wait_vmcnt<(NSW - 1) * PW>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    unsigned slot = 0;
    for (int st = 0; st < nst; ++st) {
      wait_vmcnt<(NSW - 2) * PW>();   // the next stage has landed
      __builtin_amdgcn_s_barrier();   // ... and this one is in everyone's registers
      __builtin_amdgcn_sched_barrier(0);
      request<false, true>(0, slot);
      advance();
      slot = slot + WB == (unsigned)(NSW * WB) ? 0 : slot + WB;
    }
    wait_vmcnt<0>();
  }
};

// The epilogue of tile t (split s of `splits`), straight from the accumulators (W fragment as the MFMA's A operand): a lane holds row
// 16 m + r of its wave's rows, 4 consecutive columns 16 n + 4 g .. + 3, so it writes 16 B (f32 partials) / 8 B (bf16).
template <int MT, int BN, bool SWIGLU, bool TAIL>
LK_DEVICE void ws_store(const floatx4 (&acc)[MT / 2][BN / 32], int t, int s, int M, int splits, int swiglu_I, bf16_t* __restrict__ out, long ldo,
                        float* __restrict__ part, long part_ld, long n_rows) {
  constexpr int MW = MT / 2, NW = BN / 32;
  const long first = (long)t * (SWIGLU ? BN / 2 : BN);
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4, wr = w >> 1, wc = w & 1;
  const bool split = part != nullptr;
  const bool part_vec = split && part_ld % 4 == 0 && reinterpret_cast<uintptr_t>(part) % 16 == 0;
  // (fused tail: the partial slabs through a buffer resource, written past L1 / L2)
  const __amdgpu_buffer_rsrc_t tprs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)part, (short)0, (int)min((long)splits * M * part_ld * 4, 0x7FFFFFF0L), 0x00020000);
  const bool out_vec = ldo % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0;
#pragma unroll
  for (int m = 0; m < MW; ++m) {
    const int row = wr * (8 * MT) + 16 * m + r;
    if (row >= M) continue;
    if (SWIGLU && !split) {
#pragma unroll
      for (int n = 0; n < NW / 2; ++n) {
        float y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) y[i] = rbf(silu_f(rbf(acc[m][n][i]))) * rbf(acc[m][n + NW / 2][i]);
        bf16_t* dst = out + (long)row * ldo + first + wc * (BN / 4) + 16 * n + 4 * g;
        if (out_vec) {
          uint2 pk;
          pk.x = pack_bf2(y[0], y[1]);
          pk.y = pack_bf2(y[2], y[3]);
          *reinterpret_cast<uint2*>(dst) = pk;
        } else {
#pragma unroll
          for (int i = 0; i < 4; ++i) dst[i] = f2bf(y[i]);
        }
      }
    } else {
#pragma unroll
      for (int n = 0; n < NW; ++n) {
        // first of this lane's 4 columns (W rows): a SwiGLU tile's second half are the up rows
        const long col = first + (SWIGLU ? wc * (BN / 4) + 16 * (n % (NW / 2)) + (n < NW / 2 ? 0 : swiglu_I) : wc * (BN / 2) + 16 * n) + 4 * g;
        const floatx4 v = acc[m][n];
        if (split) {
          float* dst = part + (long)s * M * part_ld + (long)row * part_ld + col;
          if (TAIL) {  // fused tail: through to memory (full 16-B tiles: checked on the host)
            __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(uint4_t, v), tprs,
                                                   (unsigned)(((long)s * M + row) * part_ld + col) * 4u, 0, kSysCoherent);
          } else if (part_vec && col + 3 < n_rows) {
            *reinterpret_cast<floatx4*>(dst) = v;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (col + i < n_rows) dst[i] = v[i];
          }
        } else {
          bf16_t* dst = out + (long)row * ldo + col;
          if (out_vec && col + 3 < n_rows) {
            uint2 pk;
            pk.x = pack_bf2(v[0], v[1]);
            pk.y = pack_bf2(v[2], v[3]);
            *reinterpret_cast<uint2*>(dst) = pk;
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
              if (col + i < n_rows) dst[i] = f2bf(v[i]);
          }
        }
      }
    }
  }
}

template <int MT, int BN, bool SWIGLU, bool TAIL, int PRO = 0, int DEPTH = ws_stages_pro(MT, BN, PRO)>
__global__ __launch_bounds__(256, 1) void wsgemm_kernel(const bf16_t* __restrict__ X, long ldx,
                                                        const bf16_t* __restrict__ W, int M, int K, int ks,
                                                        int n_tiles, int swiglu_I, bf16_t* __restrict__ out,
                                                        long ldo, float* __restrict__ part, long part_ld,
                                                        long n_rows, int rot_mul, WsTail tl, WsPro pr) {
  // n_rows: valid W rows (the last column tile may be partial: kNN over a corpus of
  // any size); rows past them read as zeros, stores are masked
  constexpr int NS = DEPTH;  // stages of the ring
  using Walk = WsWalk<MT, BN, SWIGLU, NS, NS, 0>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int t = blockIdx.x % n_tiles, s = blockIdx.x / n_tiles;
  const long kbase = (long)s * ks;
  const int nst = ks / 64;
  // K-step rotation: column tile t starts its K walk at step (t * rot_mul) % nst, so the
  // blocks streaming at the same moment read different 128-B columns of X (every block
  // reads all of X: in lockstep they would all hit the same few L2 channels)
  const int rot = rot_mul ? (int)(((long)t * rot_mul) % nst) : 0;
  const long first = (long)t * (SWIGLU ? BN / 2 : BN);   // the tile's first W row (SwiGLU: gate row; up: + I)
  Walk k;
  k.begin(smem, X, ldx, W + first * K, W + (first + swiglu_I) * K, SWIGLU ? (long)BN / 2 : min(n_rows - first, (long)BN), M, K, kbase, nst, rot);
  if constexpr (PRO != 0) {
    // W of the first stages streams in while the workgroup computes its X slice; then X's
    // first stages come from the rows just written (every wave waits for its own DMAs, the
    // walk's barrier for everyone's)
    const Walk k0 = k;
    for (int p = 0; p < NS; ++p) {
      k.template request<false, true>(0, p * Walk::WB);
      k.advance();
    }
    ws_prologue<PRO>(pr, M, K, kbase, ks);
    wait_vmcnt<0>();
    __syncthreads();
    k = k0;
    for (int p = 0; p < NS; ++p) {
      k.template request<true, false>(p * Walk::XB, 0);
      k.advance();
    }
    wait_vmcnt<0>();
  } else {
    for (int p = 0; p < NS; ++p) {
      k.template request<true, true>(p * Walk::XB, p * Walk::WB);
      k.advance();
    }
  }
  k.walk();

  ws_store<MT, BN, SWIGLU, TAIL>(k.acc, t, s, M, K / ks, swiglu_I, out, ldo, part, part_ld, n_rows);
  if constexpr (TAIL) ws_tail(tl, part, M, part_ld, K / ks, t, n_tiles, smem);
}

// Two products of one X in one launch: tiles of BN output columns of x w1^T, then tiles of BN / 2 columns of silu(x wg^T) * (x wu^T), each
// the whole of K.
template <int MT, int BN, int NS>
__global__ __launch_bounds__(256, BN == 64 ? 2 : 1) void ws_beside_kernel(const bf16_t* __restrict__ X, long ldx, int M, int K,
                                                                          const bf16_t* __restrict__ W1, bf16_t* __restrict__ out1, long ld1,
                                                                          int tiles1, const bf16_t* __restrict__ W2, int I,
                                                                          bf16_t* __restrict__ out2, long ld2) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  auto tile = [&](auto swiglu_t, int t) {
    constexpr bool SW = decltype(swiglu_t)::value;
    using Walk = WsWalk<MT, BN, SW, NS, NS, 0>;
    const int nst = K / 64;
    const long first = (long)t * (SW ? BN / 2 : BN);
    const bf16_t* W = SW ? W2 : W1;
    Walk k;
    k.begin(smem, X, ldx, W + first * K, W + (first + I) * K, SW ? BN / 2 : BN, M, K, 0, nst, (int)((long)t * 5 % nst));
    for (int p = 0; p < NS; ++p) {
      k.template request<true, true>(p * Walk::XB, p * Walk::WB);
      k.advance();
    }
    k.walk();
    ws_store<MT, BN, SW, false>(k.acc, t, 0, M, 1, I, SW ? out2 : out1, SW ? ld2 : ld1, nullptr, 0, 1L << 40);
  };
  if ((int)blockIdx.x < tiles1) tile(std::false_type{}, blockIdx.x);
  else tile(std::true_type{}, blockIdx.x - tiles1);
}

// ---------------------------------------------------------------------------------
// Loader-wave variant of the weight-streaming GEMM ("lw").  s_waitcnt vmcnt retires a wave's vector-memory ops in issue order, so where the
// same waves request X and W, the W prefetch runs only as far ahead as their common ring.  Here the W stream has waves of its own (2 loader
// waves, their own vmcnt): 4 compute waves stage X through a short ring (L2-resident, 3 stages) and compute;
// the loader waves keep the remaining LDS of W stages in flight.  Same walk, tile, K rotation and epilogue, so the same bits.  Up to 128 rows: it is
// the faster one by up to 3 % where few workgroups of 128 columns leave CUs idle (120 x 4096 x 4096 in 4 parts of K 15.0 -> 14.7 us), and
// beyond, two sets of fragments for six waves do not fit the registers (the one ring runs).
constexpr int kWsLoaderRows = 128;
constexpr int lw_nsx(int) { return 3; }
constexpr int lw_nsw(int MT, int BN) {
  const int n = (163840 - lw_nsx(MT) * 16 * MT * 128) / (BN * 128);
  return n > 12 ? 12 : n;
}

template <int MT, int BN, bool SWIGLU, bool TAIL>
__global__ __launch_bounds__(384, 1) void wsgemm_lw_kernel(const bf16_t* __restrict__ X, long ldx,
                                                           const bf16_t* __restrict__ W, int M, int K, int ks,
                                                           int n_tiles, int swiglu_I, bf16_t* __restrict__ out,
                                                           long ldo, float* __restrict__ part, long part_ld,
                                                           long n_rows, int rot_mul, WsTail tl) {
  using Walk = WsWalk<MT, BN, SWIGLU, lw_nsx(MT), lw_nsw(MT, BN), 2>;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int t = blockIdx.x % n_tiles, s = blockIdx.x / n_tiles;
  const long kbase = (long)s * ks;
  const int nst = ks / 64;
  const int rot = rot_mul ? (int)(((long)t * rot_mul) % nst) : 0;
  const long first = (long)t * (SWIGLU ? BN / 2 : BN);
  Walk k;
  k.begin(smem, X, ldx, W + first * K, W + (first + swiglu_I) * K, SWIGLU ? (long)BN / 2 : min(n_rows - first, (long)BN), M, K, kbase, nst, rot);
  if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >= 4) {
    k.load();
  } else {
    for (int p = 0; p < lw_nsx(MT); ++p) {
      k.template request<true, false>(p * Walk::XB, 0);
      k.advance();
    }
    k.walk();
    ws_store<MT, BN, SWIGLU, TAIL>(k.acc, t, s, M, K / ks, swiglu_I, out, ldo, part, part_ld, n_rows);
  }
  if constexpr (TAIL) ws_tail(tl, part, M, part_ld, K / ks, t, n_tiles, smem);  // every wave: it has barriers
}

// K-step rotation multiplier: -1 = policy (5 for unsplit-K grids -- the long-K gate_up
// + SwiGLU and LM-head shapes, 4-8 % faster on MI355X; off for split-K grids, where it
// measured neutral to 30 % slower: benchmarks/ws_rot_probe.py), >= 0 forces it
int g_ws_rot_mul = -1;

template <int MT, int BN, bool SWIGLU>
void launch_ws(const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int ks, int S, int n_tiles, int I,
               bf16_t* out, long ldo, float* part, long part_ld, long n_rows, hipStream_t st, const WsTail& tl) {
  constexpr size_t lds = (size_t)ws_stages_pro(MT, BN, 0) * (16 * MT * 128 + BN * 128);
  // (the fused-tail instantiation only where a tail runs: the plain kernel keeps its registers)
  auto kern = tl.kind ? wsgemm_kernel<MT, BN, SWIGLU, true> : wsgemm_kernel<MT, BN, SWIGLU, false>;
  if (tl.kind) LK_SET_MAX_LDS((wsgemm_kernel<MT, BN, SWIGLU, true>), (int)lds);
  else LK_SET_MAX_LDS((wsgemm_kernel<MT, BN, SWIGLU, false>), (int)lds);
  // kNN scores (n_rows given: a corpus, not a weight) walk K in one order in every tile, so
  // equal corpus rows score bit-identically and ties keep the stable id order
  const int rot_mul = n_rows < (1L << 40) ? 0 : g_ws_rot_mul >= 0 ? g_ws_rot_mul : (S == 1 ? 5 : 0);
  kern<<<n_tiles * S, 256, lds, st>>>(x, ldx, w, M, K, ks, n_tiles, I, out, ldo, part, part_ld, n_rows, rot_mul, tl,
                                      WsPro{});
}

// the prologue instantiations (one LDS ring, 16-row tiles: M <= 64)
template <int BN, bool SWIGLU, int PRO>
void launch_ws_pro(const bf16_t* x, const bf16_t* w, int M, int K, int ks, int S, int n_tiles, int I, bf16_t* out,
                   long ldo, float* part, long part_ld, hipStream_t st, const WsPro& pr) {
  constexpr int MT = 4;
  constexpr size_t lds = (size_t)ws_stages_pro(MT, BN, PRO) * (16 * MT * 128 + BN * 128);
  LK_SET_MAX_LDS((wsgemm_kernel<MT, BN, SWIGLU, false, PRO>), (int)lds);
  const int rot_mul = g_ws_rot_mul >= 0 ? g_ws_rot_mul : (S == 1 ? 5 : 0);
  wsgemm_kernel<MT, BN, SWIGLU, false, PRO><<<n_tiles * S, 256, lds, st>>>(
      x, K, w, M, K, ks, n_tiles, I, out, ldo, part, part_ld, 1L << 40, rot_mul, WsTail{}, pr);
}

template <int MT, int BN, bool SWIGLU>
void launch_ws_lw(const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int ks, int S, int n_tiles, int I,
                  bf16_t* out, long ldo, float* part, long part_ld, long n_rows, hipStream_t st, const WsTail& tl) {
  constexpr size_t lds = (size_t)lw_nsx(MT) * 16 * MT * 128 + (size_t)lw_nsw(MT, BN) * BN * 128;
  auto kern = tl.kind ? wsgemm_lw_kernel<MT, BN, SWIGLU, true> : wsgemm_lw_kernel<MT, BN, SWIGLU, false>;
  if (tl.kind) LK_SET_MAX_LDS((wsgemm_lw_kernel<MT, BN, SWIGLU, true>), (int)lds);
  else LK_SET_MAX_LDS((wsgemm_lw_kernel<MT, BN, SWIGLU, false>), (int)lds);
  const int rot_mul = n_rows < (1L << 40) ? 0 : g_ws_rot_mul >= 0 ? g_ws_rot_mul : (S == 1 ? 5 : 0);
  kern<<<n_tiles * S, 384, lds, st>>>(x, ldx, w, M, K, ks, n_tiles, I, out, ldo, part, part_ld, n_rows, rot_mul, tl);
}

// a tile's rows are reached by 32-bit offsets from its first: up to 256 of X, up to 128 of W
bool ws_too_far(int M, long ldx, int K) { return ((M - 1) * ldx + K) * 2 > (long)kWsPast || (long)K * 256 > (long)kWsPast; }

template <bool SWIGLU>
int dispatch_ws(int MT, int BN, const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int ks, int S,
                int n_tiles, int I, bf16_t* out, long ldo, float* part, long part_ld, hipStream_t st,
                long n_rows = 1L << 40, int variant = 0, const WsTail& tl = WsTail{}) {
  if (ws_too_far(M, ldx, K)) return -1;
#define LK_WS(mt, bn)                                                                                          \
  if (MT == mt && BN == bn) {                                                                                  \
    if constexpr (16 * mt <= kWsLoaderRows) {                                                                  \
      if (variant == 1) {                                                                                      \
        launch_ws_lw<mt, bn, SWIGLU>(x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, part, part_ld, n_rows, st, tl); \
        return 0;                                                                                              \
      }                                                                                                        \
    }                                                                                                          \
    launch_ws<mt, bn, SWIGLU>(x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, part, part_ld, n_rows, st, tl);    \
    return 0;                                                                                                  \
  }
  LK_WS(4, 64) LK_WS(4, 128) LK_WS(8, 64) LK_WS(8, 128) LK_WS(12, 64) LK_WS(12, 128) LK_WS(16, 64) LK_WS(16, 128)
  if constexpr (!SWIGLU) {  // 96-column tiles: projections whose N / 128 tiles leave CUs idle
    LK_WS(4, 96) LK_WS(8, 96) LK_WS(12, 96) LK_WS(16, 96)
  }
#undef LK_WS
  return -2;
}

template <int MT, int NTW, bool SWIGLU>
void launch_skinny(const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int ks, int S, int n_tiles,
                   int I, bf16_t* out, long ldo, float* part, long part_ld, hipStream_t st) {
  const size_t lds = sizeof(float) * kSkW * 16 * MT * (16 * NTW + 4);
  auto kern = skinny_gemm_kernel<MT, NTW, SWIGLU>;
  LK_SET_MAX_LDS(kern, (int)lds);
  kern<<<n_tiles * S, 256, lds, st>>>(x, ldx, w, M, K, ks, n_tiles, I, out, ldo, part, part_ld);
}

template <bool SWIGLU>
int dispatch_mt(int MT, const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int ks, int S, int n_tiles,
                int I, bf16_t* out, long ldo, float* part, long part_ld, hipStream_t st) {
  switch (MT) {
    case 1: launch_skinny<1, 4, SWIGLU>(x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, part, part_ld, st); break;
    case 2: launch_skinny<2, 4, SWIGLU>(x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, part, part_ld, st); break;
    case 4: launch_skinny<4, 4, SWIGLU>(x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, part, part_ld, st); break;
    case 8: launch_skinny<8, 4, SWIGLU>(x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, part, part_ld, st); break;
    default: return -2;
  }
  return 0;
}

}  // namespace

template <int MT, int BN>
static int launch_beside(const bf16_t* x, long ldx, int M, int K, const bf16_t* w1, int N1, bf16_t* out1, long ld1, const bf16_t* w2, int I,
                         bf16_t* out2, long ld2, hipStream_t st) {
  // 64 columns: two workgroups per CU
  constexpr int SB = (16 * MT + BN) * 128, FIT = (BN == 64 ? 81920 : 163840) / SB, NS = FIT > 8 ? 8 : FIT;
  LK_SET_MAX_LDS((ws_beside_kernel<MT, BN, NS>), NS * SB);
  ws_beside_kernel<MT, BN, NS><<<N1 / BN + I / (BN / 2), 256, NS * SB, st>>>(x, ldx, M, K, w1, out1, ld1, N1 / BN, w2, I, out2, ld2);
  LK_CHECK_LAUNCH();
  return 0;
}

int lk_ws_beside(const bf16_t* x, long ldx, int M, int K, const bf16_t* w1, int N1, bf16_t* out1, long ld1, const bf16_t* w2, int I,
                 bf16_t* out2, long ld2, int bn, hipStream_t st) {
  if ((bn != 64 && bn != 128) || M < 1 || M > 128 || K < 64 || K % 64 || N1 < bn || N1 % bn || I < bn / 2 || I % (bn / 2) || ws_too_far(M, ldx, K))
    return -1;
  if (bn == 64) return (M <= 64 ? launch_beside<4, 64> : launch_beside<8, 64>)(x, ldx, M, K, w1, N1, out1, ld1, w2, I, out2, ld2, st);
  return (M <= 64 ? launch_beside<4, 128> : launch_beside<8, 128>)(x, ldx, M, K, w1, N1, out1, ld1, w2, I, out2, ld2, st);
}

// padded row tiles of the weight-streaming GEMM: 16-row MFMA tiles, 4 waves splitting M
// (the X bytes every column block stages grow with the padding: 192 rows for M 129-192
// instead of 256)
static int ws_mt(int M) { return M <= 64 ? 4 : M <= 128 ? 8 : M <= 192 ? 12 : 16; }

// wsgemm launch plan for (M, N, K): BN (64/128) and split S maximising CU occupancy
// (1 block per CU: its LDS ring is 72-144 KB), fewest partial slabs on ties.
void lk_wsgemm_plan(int M, int N, int K, int swiglu, int* bn_out, int* s_out) {
  // Rule fitted to the exhaustive (BN, S) sweep on MI355X (profiles/r1_ws_sweep.md):
  // one block per CU, so fill <= 256 CUs in ONE round; prefer BN = 128 (half the X
  // re-reads through L2) and split K only while every block keeps >= 16 stages;
  // fall back to BN = 64 when BN = 128 leaves more than 30 % of the CUs idle and 64 fewer,
  // and where as many 64-column tiles do without a sum behind them, of short K: the chain of
  // the whole K has to stay below that of two parts and the sum (2.5 us).  Two parts of 128
  // columns / 64 whole, us, 16 / 64 / 128 / 256 rows: SwiGLU 11008 x 2048 13.7 / 17.9 / 23.3 / 29.9
  // -> 11.4 / 14.6 / 18.1 / 26.3, 10240 x 3072 17.3 / 22.2 / 29.2 / 35.9 -> 15.7 / 20.1 / 27.2 / 37.6, 8960 x 4096
  // 20.8 / 25.2 / 31.9 / 39.0 -> 18.3 / 23.8 / 30.7 / 46.2, 9472 x 7168 29.6 / 36.9 / 47.2 / 57.6 -> 30.8 / 40.1 / 52.8 /
  // 78.1, 11008 x 14336 55.6 / 68.7 / 85.2 / 102.8 -> 57.8 / 77.2 / 102.6 / 188; with parts on both sides
  // (5120 x 11008, four of 128 / two of 64) 27.2 / 33.2 / 39.6 / 49.7 -> 30.4 / 37.1 / 49.8 / 66.5.
  auto plan = [&](int BN, int* S_out) -> double {
    const int cols = swiglu ? N / 2 : N, per = swiglu ? BN / 2 : BN;
    if (cols % per) return -1.0;
    const int tiles = cols / per;
    int S = 1;
    while (tiles * S * 2 <= 256 && K % (S * 2 * 64) == 0 && K / (S * 2) >= 1024) S *= 2;
    *S_out = S;
    const int blocks = tiles * S, rounds = (blocks + 255) / 256;
    return (double)blocks / (rounds * 256.0);
  };
  int s128 = 1, s64 = 1;
  const double o128 = plan(128, &s128), o64 = plan(64, &s64);
  const bool whole = o64 == o128 && s64 == 1 && s128 > 1 && (K <= 3072 || (K <= 4096 && M <= 128));
  double occ;
  if (o128 >= 0.7 || (o128 >= 0 && o64 <= o128 && !whole)) {
    *bn_out = 128;
    *s_out = s128;
    occ = o128;
  } else {
    *bn_out = 64;
    *s_out = o64 >= 0 ? s64 : 1;
    occ = o64;
  }
  // 96-column tiles where they fill the CUs better: the Llama-3-8B QKV projection (N 6144) is
  // 48 x 128-column tiles x 4 K-splits = 192 blocks for 256 CUs, 64 x 96-column tiles x 4 = 256
  // (LK_WS_BN96=0: off)
  static const int bn96 = [] {
    const char* e = getenv("LK_WS_BN96");
    return e ? atoi(e) : 1;
  }();
  if (bn96 && !swiglu) {
    int s96 = 1;
    const double o96 = plan(96, &s96);
    if (o96 > occ + 1e-9) {
      *bn_out = 96;
      *s_out = s96;
    }
  }
}

// per-shape kernel variant of the weight-streaming GEMM: 0 = one LDS ring (wsgemm_kernel),
// 1 = loader waves (wsgemm_lw_kernel); keyed by (row tile MT, N, K, swiglu), set by the decode
// tuner's measurement (ops.tune_decode), default LK_WS_LOADER (0).  Past kWsLoaderRows there is the ring only, whatever was set.
static std::mutex g_ws_var_mu;
static std::map<long, int> g_ws_var;
static long ws_var_key(int MT, int N, int K, int swiglu) {
  return (((long)MT * 1000003L + N) * 1000003L + K) * 2 + (swiglu ? 1 : 0);
}
int lk_wsgemm_variant(int M, int N, int K, int swiglu) {
  if (M > kWsLoaderRows) return 0;
  static const int dflt = [] {
    const char* e = getenv("LK_WS_LOADER");
    return e ? (atoi(e) != 0) : 0;
  }();
  std::lock_guard<std::mutex> lock(g_ws_var_mu);
  auto it = g_ws_var.find(ws_var_key(ws_mt(M), N, K, swiglu));
  return it != g_ws_var.end() ? it->second : dflt;
}
int lk_wsgemm_set_variant(int M, int N, int K, int swiglu, int variant) {
  if (variant < -1 || variant > 1) return -1;
  std::lock_guard<std::mutex> lock(g_ws_var_mu);
  const long key = ws_var_key(ws_mt(M), N, K, swiglu);
  if (variant < 0) g_ws_var.erase(key);
  else g_ws_var[key] = variant;
  return 0;
}

int lk_wsgemm(const bf16_t* x, long ldx, const bf16_t* w, int M, int N, int K, int BN, int S, int swiglu,
              bf16_t* out, long ldo, float* part, hipStream_t st) {
  if (M < 1 || M > 256 || S < 1 || K % (S * 64) || (BN != 64 && BN != 128 && (BN != 96 || swiglu))) return -1;
  const int per = swiglu ? BN / 2 : BN;
  if (swiglu ? (N % 2 || (N / 2) % per) : N % BN) return -1;
  if (S > 1 && part == nullptr) return -1;
  const int I = swiglu ? N / 2 : 0;
  const int n_tiles = (swiglu ? I : N) / per;
  const int MT = ws_mt(M);
  const int ks = K / S;
  float* p = S > 1 ? part : nullptr;
  const int var = lk_wsgemm_variant(M, N, K, swiglu);
  const int rc = swiglu ? dispatch_ws<true>(MT, BN, x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, p, N, st,
                                            1L << 40, var)
                        : dispatch_ws<false>(MT, BN, x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, p, N, st,
                                             1L << 40, var);
  if (rc) return rc;
  if (S > 1) {
    const int n_out = swiglu ? I : N;
    const long work = (long)M * (n_out / 4);
    int grid = (int)((work + 255) / 256);
    if (grid > 2048) grid = 2048;
    if (swiglu)
      splitk_reduce_kernel<true><<<grid, 256, 0, st>>>(part, S, M, N, n_out, I, out, ldo);
    else
      splitk_reduce_kernel<false><<<grid, 256, 0, st>>>(part, S, M, N, n_out, 0, out, ldo);
  }
  LK_CHECK_LAUNCH();
  return 0;
}

void lk_wsgemm_set_rot(int rot_mul) { g_ws_rot_mul = rot_mul < 0 ? -1 : rot_mul; }

// Weight-streaming GEMM with a consumer-side X prologue (WsPro, one LDS ring, M <= 64): kind 1 =
// residual add + RMSNorm of the producer's split-K slabs, kind 2 = flash-decoding merge of a
// paged-decode step's split partials.  x: [M, K] bf16 rows (kind 1: written; kind 2: the
// attention output, merged rows written).  S > 1: partial slabs into part, and with out also the
// reduce (SwiGLU) into out; S == 1: out directly.
int lk_wsgemm_pro(int kind, bf16_t* x, const bf16_t* w, int M, int N, int K, int BN, int S, int swiglu,
                  bf16_t* out, long ldo, float* part, const float* pp, int pS, const bf16_t* res, bf16_t* res_out,
                  long rs, const bf16_t* gamma, float eps, const float* po, const float* pml, const int* ctx, int Hq,
                  int D, int max_splits, int split, hipStream_t st) {
  if (M < 1 || M > 64 || S < 1 || K % (S * 64) || !x || ws_too_far(M, K, K) || (BN != 64 && BN != 128 && (BN != 96 || swiglu))) return -1;
  const int per = swiglu ? BN / 2 : BN;
  if (swiglu ? (N % 2 || (N / 2) % per) : N % BN) return -1;
  if ((S > 1 && !part) || (S == 1 && !out)) return -1;
  WsPro pr;
  pr.kind = kind;
  pr.x = x;
  if (kind == 1) {
    if (K % 8 || K > 8192 || !pp || pS < 1 || !res || !res_out || res == res_out || !gamma || rs % 8) return -1;
    pr.part = pp;
    pr.S = pS;
    pr.slab = (long)M * K;
    pr.res = res;
    pr.res_out = res_out;
    pr.rs = rs;
    pr.gamma = gamma;
    pr.eps = eps;
  } else if (kind == 2) {
    if (!po || !pml || !ctx || D <= 0 || Hq * D != K || max_splits < 1 || split < 1) return -1;
    pr.po = po;
    pr.pml = pml;
    pr.ctx = ctx;
    pr.Hq = Hq;
    pr.D = D;
    pr.max_splits = max_splits;
    pr.split = split;
  } else {
    return -1;
  }
  const int I = swiglu ? N / 2 : 0;
  const int n_tiles = (swiglu ? I : N) / per;
  const int ks = K / S;
  float* p = S > 1 ? part : nullptr;
#define LK_PRO(bn, sw, kd) \
  if (BN == bn && (swiglu != 0) == sw && kind == kd) launch_ws_pro<bn, sw, kd>(x, w, M, K, ks, S, n_tiles, I, out, ldo, p, N, st, pr); else
  LK_PRO(64, false, 1) LK_PRO(96, false, 1) LK_PRO(128, false, 1) LK_PRO(64, true, 1) LK_PRO(128, true, 1)
  LK_PRO(64, false, 2) LK_PRO(96, false, 2) LK_PRO(128, false, 2) return -2;
#undef LK_PRO
  LK_CHECK_LAUNCH();
  if (S > 1 && out) {
    const int n_out = swiglu ? I : N;
    const long work = (long)M * (n_out / 4);
    int grid = (int)((work + 255) / 256);
    if (grid > 2048) grid = 2048;
    if (swiglu)
      splitk_reduce_kernel<true><<<grid, 256, 0, st>>>(part, S, M, N, n_out, I, out, ldo);
    else
      splitk_reduce_kernel<false><<<grid, 256, 0, st>>>(part, S, M, N, n_out, 0, out, ldo);
    LK_CHECK_LAUNCH();
  }
  return 0;
}

int lk_wsgemm_part(const bf16_t* x, long ldx, const bf16_t* w, int M, int N, int K, int BN, int S, float* part,
                   hipStream_t st) {
  if (M < 1 || M > 256 || S < 2 || K % (S * 64) || (BN != 64 && BN != 96 && BN != 128) || N % BN ||
      part == nullptr)
    return -1;
  const int MT = ws_mt(M);
  const int rc = dispatch_ws<false>(MT, BN, x, ldx, w, M, K, K / S, S, N / BN, 0, nullptr, 0, part, N, st,
                                    1L << 40, lk_wsgemm_variant(M, N, K, 0));
  LK_CHECK_LAUNCH();
  return rc;
}

// split-K GEMM whose last split workgroup per head applies RoPE and writes the paged KV (WsTail
// kind 1): the rows lk_splitk_rope_kv would leave, without its launch.  Needs one column tile per
// head (BN == D) and S in {2, 4, 8}; tickets: >= (Hq + 2 Hkv) zeroed int32.
int lk_ws_rope_kv_fused(const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int BN, int S, float* part,
                        int* tickets, bf16_t* qkv, long qs, const int* positions, const float* cos_sin, int Hq,
                        int Hkv, int D, bf16_t* kc, bf16_t* vc, const int* slots, int BS, int neox,
                        int write_k_inplace, hipStream_t st) {
  const int N = (Hq + 2 * Hkv) * D;
  if (M < 1 || M > 256 || !(S == 2 || S == 4 || S == 8) || K % (S * 64) || BN != D || BN != 128 || !part ||
      !tickets || !qkv || qs % 8 || D % 16 || (long)S * M * N * 4 >= 0x7FFFFFF0L)
    return -1;
  WsTail tl;
  tl.kind = 1;
  tl.tickets = tickets;
  tl.out = qkv;
  tl.os = qs;
  tl.positions = positions;
  tl.cos_sin = cos_sin;
  tl.Hq = Hq;
  tl.Hkv = Hkv;
  tl.D = D;
  tl.kc = kc;
  tl.vc = vc;
  tl.slots = slots;
  tl.BS = BS;
  tl.neox = neox;
  tl.write_k_inplace = write_k_inplace;
  const int rc = dispatch_ws<false>(ws_mt(M), BN, x, ldx, w, M, K, K / S, S, N / BN, 0, nullptr, 0, part, N, st,
                                    1L << 40, lk_wsgemm_variant(M, N, K, 0), tl);
  LK_CHECK_LAUNCH();
  return rc;
}

// split-K GEMM + residual add + RMSNorm by the grid's last workgroup (WsTail kind 2), for a few
// rows (M <= 4: one workgroup normalises them all); tickets: >= 1 zeroed int32
int lk_ws_rmsnorm_fused(const bf16_t* x, long ldx, const bf16_t* w, int M, int N, int K, int BN, int S, float* part,
                        int* tickets, bf16_t* out, long os, bf16_t* residual, long rs, const bf16_t* norm_w, float eps,
                        hipStream_t st) {
  if (M < 1 || M > 4 || !(S == 2 || S == 4 || S == 8) || K % (S * 64) || (BN != 64 && BN != 128) || N % BN ||
      !part || !tickets || !out || !residual || os % 8 || rs % 8 || (long)S * M * N * 4 >= 0x7FFFFFF0L)
    return -1;
  WsTail tl;
  tl.kind = 2;
  tl.tickets = tickets;
  tl.out = out;
  tl.os = os;
  tl.residual = residual;
  tl.rs = rs;
  tl.norm_w = norm_w;
  tl.eps = eps;
  const int rc = dispatch_ws<false>(ws_mt(M), BN, x, ldx, w, M, K, K / S, S, N / BN, 0, nullptr, 0, part, N, st,
                                    1L << 40, lk_wsgemm_variant(M, N, K, 0), tl);
  LK_CHECK_LAUNCH();
  return rc;
}

// Scores of a corpus: thousands of tiles with few K stages each, so what counts is that one workgroup's start and end hide behind another's:
// a ring of DEPTH stages leaves room for two or three on a CU, and requests nothing that a short row does not have.  One ring of
// 160 KB / this, us, 485,620 rows, 17 / 40 / 100 queries with their top 5: 128 columns 92.4 / 120.8 / 194.6 -> 67.7 / 100.8 / 174.7 (2 stages), 384 129.5 /
// 159.7 / 243.5 -> 110.5 / 143.6 / 235.8 (3), 768 189.6 / 225.8 / 318.2 -> 174.3 / 212.4 / 314.4 (3); 20,011 rows level.  2 stages of longer rows
// were ahead for a large corpus (17: 172.6) and behind for 1,000 and 20,011 rows (28.4 -> 31.6); past 128 queries there is no room for two.
template <int MT, int DEPTH>
static int launch_scores(const bf16_t* x, long ldx, const bf16_t* w, int M, int K, int tiles, float* out, long ldo, long N, hipStream_t st) {
  constexpr int lds = DEPTH * (16 * MT + 128) * 128;
  LK_SET_MAX_LDS((wsgemm_kernel<MT, 128, false, false, 0, DEPTH>), lds);
  wsgemm_kernel<MT, 128, false, false, 0, DEPTH><<<tiles, 256, lds, st>>>(x, ldx, w, M, K, K, tiles, 0, nullptr, 0, out, ldo, N, 0, WsTail{}, WsPro{});
  return 0;
}

// f32 X W^T for a W of any row count (kNN scores: X = queries, W = corpus rows):
// out[M, N] with row stride ldo; one pass over W, no split-K.
int lk_ws_scores_f32(const bf16_t* x, long ldx, const bf16_t* w, int M, long N, int K, float* out, long ldo,
                     hipStream_t st) {
  if (M < 1 || M > 256 || N < 1 || K % 64 || K < 64) return -1;
  const int BN = 128;
  const long tiles = (N + BN - 1) / BN;
  if (tiles > (1L << 30)) return -1;
  const int MT = ws_mt(M);
  if (ws_too_far(M, ldx, K)) return -1;
  const int deep = K <= 192 ? 2 : MT <= 8 ? 3 : 0;
  int rc = 0;
  switch (MT + 100 * deep) {
    case 204: rc = launch_scores<4, 2>(x, ldx, w, M, K, (int)tiles, out, ldo, N, st); break;
    case 208: rc = launch_scores<8, 2>(x, ldx, w, M, K, (int)tiles, out, ldo, N, st); break;
    case 212: rc = launch_scores<12, 2>(x, ldx, w, M, K, (int)tiles, out, ldo, N, st); break;
    case 216: rc = launch_scores<16, 2>(x, ldx, w, M, K, (int)tiles, out, ldo, N, st); break;
    case 304: rc = launch_scores<4, 3>(x, ldx, w, M, K, (int)tiles, out, ldo, N, st); break;
    case 308: rc = launch_scores<8, 3>(x, ldx, w, M, K, (int)tiles, out, ldo, N, st); break;
    default: rc = dispatch_ws<false>(MT, BN, x, ldx, w, M, K, K, 1, (int)tiles, 0, nullptr, 0, out, ldo, st, N);
  }
  LK_CHECK_LAUNCH();
  return rc;
}

int lk_skinny_splits(int M, int N, int K, int swiglu) {
  (void)M;
  const int BN = 64;
  const int cols = swiglu ? N / 2 : N;
  const int n_tiles = cols / (swiglu ? BN / 2 : BN);
  int S = 1;
  while (n_tiles * S < 256 && S < 8 && K % (2 * S * kSkW * 64) == 0 && K / (2 * S) >= 512) S *= 2;
  return S;
}

// out = X W^T (swiglu=0, out [M,N]) or silu(X Wg^T) * (X Wu^T) (swiglu=1, W = [Wg; Wu]
// of 2I rows, out [M,I]).  part: f32 workspace of S*M*N floats when S > 1.
int lk_skinny_gemm(const bf16_t* x, long ldx, const bf16_t* w, int M, int N, int K, int S, int swiglu,
                   bf16_t* out, long ldo, float* part, hipStream_t st) {
  if (M < 1 || M > 128 || S < 1 || K % (S * kSkW * 64)) return -1;
  const int BN = 64;
  if (swiglu ? (N % 2 || (N / 2) % (BN / 2)) : N % BN) return -1;
  if (S > 1 && part == nullptr) return -1;
  const int I = swiglu ? N / 2 : 0;
  const int n_tiles = swiglu ? I / (BN / 2) : N / BN;
  const int MT = M <= 16 ? 1 : M <= 32 ? 2 : M <= 64 ? 4 : 8;
  const int ks = K / S;
  float* p = S > 1 ? part : nullptr;
  const int rc = swiglu ? dispatch_mt<true>(MT, x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, p, N, st)
                        : dispatch_mt<false>(MT, x, ldx, w, M, K, ks, S, n_tiles, I, out, ldo, p, N, st);
  if (rc) return rc;
  if (S > 1) {
    const int n_out = swiglu ? I : N;
    const long work = (long)M * (n_out / 4);
    int grid = (int)((work + 255) / 256);
    if (grid > 2048) grid = 2048;
    if (swiglu)
      splitk_reduce_kernel<true><<<grid, 256, 0, st>>>(part, S, M, N, n_out, I, out, ldo);
    else
      splitk_reduce_kernel<false><<<grid, 256, 0, st>>>(part, S, M, N, n_out, 0, out, ldo);
  }
  LK_CHECK_LAUNCH();
  return 0;
}
