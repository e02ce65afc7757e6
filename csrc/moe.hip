// Feed-forward of experts chosen per token by a table of token ids (no routing network, equal weights).
//
//   lk_moe_route  (token, choice) pairs p = t * top + k sorted by their expert table[ids[t]][k] (ids null: table[t][k], the
//                 choice a router made for each token of the step): seg[e] .. seg[e + 1] are
//                 expert e's places in `order`.  One workgroup: a histogram and a placement with LDS atomics (the order
//                 inside an expert's segment is arbitrary; every row of the products below is computed on its own).
//   lk_moe_gemm   grouped product over the sorted pairs on MFMA tiles of 16 pairs: a tile's rows belong to one expert,
//                 so its B operand is that expert's weight rows.  The tile list is not materialised: a workgroup finds
//                 its (expert, first pair) by walking seg[], so the launch needs nothing from the host and a step with
//                 experts can be captured in a graph.
//                   act = 1:  mid[place] = silu(W_gate x_t) * (W_up x_t)   (x row of the pair's token; rows of `mid` in
//                             sorted order; W = [gate rows | up rows], F columns each)
//                   act = 0:  out[p]     = W_down mid[place]               (rows of `out` in pair order, so a token's
//                             `top` results are adjacent for the consumer that averages them)
//
// Fragments go straight from global memory / L2 into the MFMA operands (16-byte loads where rows are 16-byte
// aligned, element loads otherwise), f32 accumulation, bf16 (v_mfma_f32_16x16x32_bf16) or f32 (16x16x4) activations.
#include "common.h"
#include "kernels.h"
#include "attn_frag.h"
#include "row_ring.h"

namespace {

constexpr int kRouteThreads = 1024;
constexpr int kMaxExperts = 1024;

// One workgroup; its time is the chain of dependent loads (token id, then table), so a thread requests the ids of all its pairs and then
// all their table entries, kRouteU at a time, and keeps the experts in registers for the second pass where they fit (8,192 pairs).
// 8,192 pairs of 16 experts: one pair after the other, twice, 18.7 us, now 14.6 (the rest are the counters' atomics).  Up to 1,024 pairs
// take the form of one pair per thread (U = 1: eight divisions by top cost a decode step more than its loads:
// 64 tokens x 2 of 16 experts 4.3 -> 2.0 us).
constexpr int kRouteU = 8;

// inclusive sums over the wave's lanes
LK_DEVICE int wave_sums(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr 1, 2, 4, 8: inside 16 lanes
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast 15 to the second and fourth 16
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast 31 to the upper half
  return v;
}

struct RouteTables {
  const int* t[kMaxRouteTables];
};

// one workgroup per table (the layers of a model whose tables are indexed by the token ids know their routing at the step's start)
template <int U>
__global__ __launch_bounds__(kRouteThreads) void moe_route_kernel(const int* __restrict__ ids, const int* __restrict__ live, RouteTables tables,
                                                                  int vocab, int top, int E, int T, int* __restrict__ seg,
                                                                  int* __restrict__ order) {
  const int* __restrict__ table = tables.t[blockIdx.x];
  seg += (long)blockIdx.x * (E + 1);
  order += (long)blockIdx.x * T * top;
  __shared__ int cnt[kMaxExperts];
  __shared__ int nxt[kMaxExperts + 1];   // the last: the pairs of rows that are not live
  const int n = T * top, tid = threadIdx.x;
  for (int e = tid; e < E; e += kRouteThreads) cnt[e] = 0;
  __syncthreads();
  int ex[U], lv[U];
  auto experts = [&](int p0) {   // of pairs p0 + tid + 1024 u (behind the end: the last pair's)
    int id[U], at[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if ((long)p0 + u * kRouteThreads >= n) break;   // (no division for pairs that are not there)
      const int p = (int)min((long)p0 + u * kRouteThreads + tid, (long)n - 1), t = p / top;
      at[u] = p - t * top;
      id[u] = ids ? ids[t] : t;                 // no ids: the table has one row per token of the step
      lv[u] = live ? live[t] : 0;
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if ((long)p0 + u * kRouteThreads >= n) break;
      ex[u] = table[(long)min(max(id[u], 0), vocab - 1) * top + at[u]];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if ((long)p0 + u * kRouteThreads >= n) break;
      ex[u] = lv[u] < 0 ? E : min(max(ex[u], 0), E - 1);
    }
  };
  for (long p0 = 0; p0 < n; p0 += U * kRouteThreads) {
    experts((int)p0);
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (p0 + u * kRouteThreads + tid < n && ex[u] < E) atomicAdd(&cnt[ex[u]], 1);
  }
  __syncthreads();
  if (tid < 64) {   // running sums of the counts, 64 experts at a time
    int acc = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      const int c = e0 + tid < E ? cnt[e0 + tid] : 0;
      const int v = wave_sums(c);
      if (e0 + tid < E) seg[e0 + tid] = nxt[e0 + tid] = acc + v - c;
      acc += __builtin_amdgcn_readlane(v, 63);
    }
    if (tid == 0) seg[E] = nxt[E] = acc;
  }
  __syncthreads();
  for (long p0 = 0; p0 < n; p0 += U * kRouteThreads) {
    if (n > U * kRouteThreads) experts((int)p0);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const long p = p0 + u * kRouteThreads + tid;
      if (p < n) order[atomicAdd(&nxt[ex[u]], 1)] = (int)p;
    }
  }
}

// grid (row tiles of 16 RT pairs: at most pairs / (16 RT) + E, column blocks): 4 waves side by side along the columns, each
// RT row tiles x NB column tiles of 16 x 16 in registers, so a step of the contraction costs RT + NB fragment loads for
// RT x NB MFMAs (RT = 1, NB = 2: decode-sized steps, where the experts' weights are read once and little else
// matters; RT = 4, NB = 4: prompt portions).  The waves of a workgroup read the same x rows (L1 hits).
//   act: a wave's column tiles are NB / 2 gate tiles and the up tiles of the same columns;
//   else: NB neighbouring tiles of output columns.
template <typename T, bool ACT, int RT>
__global__ __launch_bounds__(256) void moe_gemm_kernel(const T* __restrict__ x, long xs, const int* __restrict__ order,
                                                       const int* __restrict__ seg, int E, int top, const T* __restrict__ w, int N,
                                                       int K, T* __restrict__ out, long os, int vec) {
  constexpr int EV = El<T>::V, NB = RT == 1 ? 2 : 4, CW = ACT ? NB / 2 : NB;   // CW: 16-column tiles of output per wave
  constexpr bool EXACT = sizeof(T) == 4;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, n16 = lane & 15, g = lane >> 4;
  // this workgroup's expert and first place: tiles are counted expert by expert
  int e = 0, place0 = 0, end = 0, acc = 0;
  {
    const int tile = blockIdx.x;
    bool found = false;
    for (int i = 0; i < E; ++i) {
      const int a = seg[i], b = seg[i + 1], nt = (b - a + 16 * RT - 1) / (16 * RT);
      if (!found && tile < acc + nt) {
        found = true;
        e = i;
        place0 = a + (tile - acc) * 16 * RT;
        end = b;
      }
      acc += nt;
    }
    if (!found) return;
  }
  const int F = ACT ? N / 2 : N;                       // output columns
  const int c0 = (blockIdx.y * 4 + wv) * CW * 16;
  if (c0 >= F) return;
  const T* xrow[RT];
  bool rvalid[RT];
#pragma unroll
  for (int r = 0; r < RT; ++r) {
    const int place = place0 + 16 * r + n16;
    rvalid[r] = place < end;
    const int pair = rvalid[r] ? order[place] : 0;
    xrow[r] = x + (long)(ACT ? pair / top : (rvalid[r] ? place : 0)) * xs;
  }
  const T* wbase = w + (long)e * N * K;
  // B operand rows: rows of columns past the end read row 0 and are not stored
  const T* wrow[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int oc = c0 + 16 * (c % CW) + n16;                       // output column of this tile
    const int row = ACT && c >= CW ? F + oc : oc;                   // up rows follow the F gate rows
    wrow[c] = wbase + (long)(oc < F ? row : 0) * K;
  }
  floatx4 accv[RT][NB];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < NB; ++c) accv[r][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  // Every lane runs every step (the MFMAs need the whole wave).  With 16-byte aligned rows, groups of U whole steps are
  // plain vector loads issued together before their MFMAs (U x (RT + NB) requests in flight per lane: a decode-sized step
  // is a stream of expert weights, and what it needs is memory-level parallelism); rows behind the end of a tile read a
  // valid row whose results are never stored.  What is left, and unaligned rows, go through frag(), which pads with zeros.
  constexpr int U = RT == 1 ? 4 : 1;
  int kb = 0;
  if (vec) {
    for (; kb + U * 4 * EV <= K; kb += U * 4 * EV) {
      uint4_t a[U][RT], b[U][NB];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int k = kb + (4 * u + g) * EV;
#pragma unroll
        for (int r = 0; r < RT; ++r) a[u][r] = ld16(xrow[r] + k);
#pragma unroll
        for (int c = 0; c < NB; ++c) b[u][c] = ld16(wrow[c] + k);
      }
#pragma unroll
      for (int u = 0; u < U; ++u)
#pragma unroll
        for (int r = 0; r < RT; ++r)
#pragma unroll
          for (int c = 0; c < NB; ++c) accv[r][c] = mma_qk<T>(a[u][r], b[u][c], accv[r][c]);
    }
  }
  for (; kb < K; kb += 4 * EV) {
    const int k = kb + g * EV;
    uint4_t a[RT], b[NB];
#pragma unroll
    for (int r = 0; r < RT; ++r) a[r] = frag<T>(xrow[r], k, K, vec);
#pragma unroll
    for (int c = 0; c < NB; ++c) b[c] = frag<T>(wrow[c], k, K, vec);
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < NB; ++c) accv[r][c] = mma_qk<T>(a[r], b[c], accv[r][c]);
  }
  // accumulator j of this lane: pair row 4 g + j of the row tile, column n16 of the column tile
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int pl = place0 + 16 * r + 4 * g + j;
      if (pl >= end) continue;
      T* orow = out + (long)(ACT ? pl : order[pl]) * os;
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        const int col = c0 + 16 * c + n16;
        if (col >= F) continue;
        if constexpr (ACT) {
          const float gt = accv[r][c][j];
          const float sg = EXACT ? gt / (1.f + expf(-gt)) : gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt));
          El<T>::st(orow + col, sg * accv[r][CW + c][j]);
        } else {
          El<T>::st(orow + col, accv[r][c][j]);
        }
      }
    }
}

// The same product for prompt-sized steps with 16-byte aligned rows: a workgroup owns 32 RT pairs x 128 weight
// rows (act: 64 gate rows and the 64 up rows of the same columns), its 4 waves 16 RT x 64 quarters of it (RT = 4).  Both operands of a
// 64-byte step of the contraction are fetched once per workgroup with coalesced 16-byte loads (the next step's while this
// one is multiplied), staged in LDS (rows padded to 80 bytes against bank conflicts, two buffers, one barrier per step)
// and read from there as MFMA fragments, so global memory sees each operand byte once per workgroup instead of once per wave.
template <typename T, bool ACT, int RT>
__global__ __launch_bounds__(256) void moe_gemm_lds_kernel(const T* __restrict__ x, long xs, const int* __restrict__ order,
                                                           const int* __restrict__ seg, int E, int top, const T* __restrict__ w, int N,
                                                           int K, T* __restrict__ out, long os) {
  constexpr int EV = El<T>::V, KS = 4 * EV, TM = 32 * RT, TN = 128, PA = TM / 64;   // PA: 16-byte pieces of the A tile per thread
  constexpr bool EXACT = sizeof(T) == 4;
  __shared__ uint4_t sA[2][TM][5];
  __shared__ uint4_t sB[2][TN][5];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6, n16 = lane & 15, g = lane >> 4;
  const int F = ACT ? N / 2 : N;
  const int CB = (F + (ACT ? 64 : 128) - 1) / (ACT ? 64 : 128);   // column blocks
  // Work items in the order (expert, column block, row tile of the expert), dealt to the XCDs in contiguous runs: the
  // workgroups an XCD runs together share a few row tiles of x (they stay in its L2 over the column blocks) and each
  // block of weight rows among an expert's row tiles.
  int e = 0, place0 = 0, end = 0, cb = 0, acc = 0;
  {
    const int item = xcd_remap(blockIdx.x, gridDim.x);
    bool found = false;
    for (int i = 0; i < E; ++i) {
      const int a = seg[i], b = seg[i + 1], nt = (b - a + TM - 1) / TM;
      if (!found && item < acc + nt * CB) {
        found = true;
        e = i;
        cb = (item - acc) / nt;
        place0 = a + ((item - acc) % nt) * TM;
        end = b;
      }
      acc += nt * CB;
    }
    if (!found) return;   // the whole workgroup leaves: no barrier is skipped by a part of it
  }
  const int c0 = cb * (ACT ? 64 : 128);
  const T* wbase = w + (long)e * N * K;
  // this thread's two 16-byte pieces of the A tile and of the B tile: piece = tid + 256 i -> row piece / 4, segment piece % 4
  const T* ap[PA];
  const T* bp[2];
  const int pseg = tid & 3, prow = tid >> 2;   // piece tid + 256 i: row prow + 64 i, segment pseg
#pragma unroll
  for (int i = 0; i < PA; ++i) {
    const int place = place0 + prow + 64 * i;
    ap[i] = place < end ? x + (long)(ACT ? order[place] / top : place) * xs : nullptr;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int r = prow + 64 * i;
    const int oc = ACT ? c0 + (r & 63) : c0 + r;
    const int row = ACT && r >= 64 ? F + oc : oc;
    bp[i] = oc < F ? wbase + (long)row * K : nullptr;
  }
  const int wy = wv >> 1, wx = wv & 1;
  int brow[4];   // first B-tile row of the wave's column tiles
#pragma unroll
  for (int c = 0; c < 4; ++c) brow[c] = ACT ? (c < 2 ? wx * 32 + 16 * c : 64 + wx * 32 + 16 * (c - 2)) : wx * 64 + 16 * c;
  floatx4 accv[RT][4];
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int c = 0; c < 4; ++c) accv[r][c] = floatx4{0.f, 0.f, 0.f, 0.f};
  uint4_t ra[PA], rb[2];
  auto fetch = [&](int kb) {
    const int k = kb + pseg * EV;
#pragma unroll
    for (int i = 0; i < PA; ++i) ra[i] = ap[i] && k < K ? ld16(ap[i] + k) : uint4_t{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 2; ++i) rb[i] = bp[i] && k < K ? ld16(bp[i] + k) : uint4_t{0u, 0u, 0u, 0u};
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int i = 0; i < PA; ++i) sA[buf][prow + 64 * i][pseg] = ra[i];
#pragma unroll
    for (int i = 0; i < 2; ++i) sB[buf][prow + 64 * i][pseg] = rb[i];
  };
  fetch(0);
  stage(0);
  __syncthreads();
  int cur = 0;
  for (int kb = 0; kb < K; kb += KS) {
    const bool more = kb + KS < K;
    if (more) fetch(kb + KS);
    uint4_t a[RT], b[4];
#pragma unroll
    for (int r = 0; r < RT; ++r) a[r] = sA[cur][wy * 16 * RT + 16 * r + n16][g];
#pragma unroll
    for (int c = 0; c < 4; ++c) b[c] = sB[cur][brow[c] + n16][g];
#pragma unroll
    for (int r = 0; r < RT; ++r)
#pragma unroll
      for (int c = 0; c < 4; ++c) accv[r][c] = mma_qk<T>(a[r], b[c], accv[r][c]);
    if (more) stage(cur ^ 1);
    __syncthreads();
    cur ^= 1;
  }
  constexpr int CW = ACT ? 2 : 4;
  const int wc0 = c0 + (ACT ? wx * 32 : wx * 64);
#pragma unroll
  for (int r = 0; r < RT; ++r)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int pl = place0 + wy * 16 * RT + 16 * r + 4 * g + j;
      if (pl >= end) continue;
      T* orow = out + (long)(ACT ? pl : order[pl]) * os;
#pragma unroll
      for (int c = 0; c < CW; ++c) {
        const int col = wc0 + 16 * c + n16;
        if (col >= F) continue;
        if constexpr (ACT) {
          const float gt = accv[r][c][j];
          const float sg = EXACT ? gt / (1.f + expf(-gt)) : gt * __builtin_amdgcn_rcpf(1.f + __expf(-gt));
          El<T>::st(orow + col, sg * accv[r][CW + c][j]);
        } else {
          El<T>::st(orow + col, accv[r][c][j]);
        }
      }
    }
}

template <typename T, bool ACT, int RT>
int launch_moe_lds(const void* x, long xs, const int* order, const int* seg, int E, int top, long pairs, const void* w, int N, int K,
                   void* out, long os, hipStream_t st) {
  const int F = ACT ? N / 2 : N, per_wg = ACT ? 64 : 128, TM = 32 * RT;
  const long items = ((pairs + TM - 1) / TM + E) * ((F + per_wg - 1) / per_wg);
  if (items > 2147483647L) return -1;
  const dim3 grid((unsigned)items);
  moe_gemm_lds_kernel<T, ACT, RT><<<grid, 256, 0, st>>>((const T*)x, xs, order, seg, E, top, (const T*)w, N, K, (T*)out, os);
  LK_CHECK_LAUNCH();
  return 0;
}

template <typename T, bool ACT, int RT>
int launch_moe(const void* x, long xs, const int* order, const int* seg, int E, int top, long pairs, const void* w, int N, int K,
               void* out, long os, int vec, hipStream_t st) {
  constexpr int NB = RT == 1 ? 2 : 4, per_wg = 4 * 16 * (ACT ? NB / 2 : NB);
  const int F = ACT ? N / 2 : N;
  const long tiles = (pairs + 16 * RT - 1) / (16 * RT) + E;
  if (tiles > 2147483647L || (F + per_wg - 1) / per_wg > 65535) return -1;
  const dim3 grid((unsigned)tiles, (unsigned)((F + per_wg - 1) / per_wg));
  moe_gemm_kernel<T, ACT, RT><<<grid, 256, 0, st>>>((const T*)x, xs, order, seg, E, top, (const T*)w, N, K, (T*)out, os, vec);
  LK_CHECK_LAUNCH();
  return 0;
}

// A product of the same rows beside the experts' (moe_rows_kernel): y = x w^T [M, N], in the first nb workgroups of the launch.
struct Beside {
  const bf16_t* w = nullptr;
  bf16_t* y = nullptr;
  long ldy = 0;
  int M = 0, N = 0, nb = 0;
};

// The same product for decode-sized steps of bf16 rows: a stream of the experts' weights, each read once.  One workgroup
// takes 16 columns (act: 16 gate and their up columns; else 2 x 16) of ONE expert and all of its pairs, MT x 16 at a
// time (more than that is a second walk over the same weight rows, out of L2); the four waves split K through private
// LDS rings (row_ring.h), so up to 64 KB of weight rows are on their way per CU and no wave waits for another inside the walk.
// 64 tokens x 2 of 16 experts of 2048 x 2816: gate / up 110 us (3.4 TB/s) -> 56 us (6.6 TB/s), down 67 us (2.7 TB/s) -> 30 us.
// BESIDE: the stream's gate is a product of the rows that the experts read, and on its own a launch of 5.7 us for 8 MB (64 x 2,048 x 2,048) before
// theirs, which is bound by the weights' stream; in it the three products take 23.5 -> 20.0 us with one row, 59.5 ->
// 55.9 with 8, 92.3 -> 89.5 with 32, 93.3 -> 91.6 with 64 (spread over the launch instead of in front: 22.5, 70.8 for 73.8, 87.9, 90.9).  Its workgroups take what the experts' take in,
// (MT + 2) 16-row tiles of K, as MT + 1 tiles of rows by 16 columns; the row tiles of a column follow one another on one XCD.
template <bool ACT, int MT, bool BESIDE = false>
__global__ __launch_bounds__(256) void moe_rows_kernel(const bf16_t* __restrict__ x, long xs, const int* __restrict__ order,
                                                       const int* __restrict__ seg, int top, const bf16_t* __restrict__ w, int N, int K,
                                                       bf16_t* __restrict__ out, long os, int blocks, long pairs, int E, Beside p) {
  constexpr int NT = 2, NS = 3;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  int at = blockIdx.x;
  if constexpr (BESIDE) {
    if (at < p.nb) {
      constexpr int BT = MT + 1;
      const int tiles = (p.M + 16 * BT - 1) / (16 * BT), column = (at >> 3) / tiles * 8 + (at & 7), m0 = (at >> 3) % tiles * (16 * BT);
      if (column * 16 >= p.N) return;
      const int all = K / 64, first = wave * all / kRgWaves, nst = (wave + 1) * all / kRgWaves - first, lrow = lane >> 3;
      const long k = (long)first * 64 + rg_lane_col(lane);
      const bf16_t *xp[2 * BT], *wp[2];
#pragma unroll
      for (int i = 0; i < 2 * BT; ++i) xp[i] = x + (long)min(m0 + 8 * i + lrow, p.M - 1) * xs + k;  // rows past M repeat the last one
#pragma unroll
      for (int i = 0; i < 2; ++i) wp[i] = p.w + (long)(column * 16 + 8 * i + lrow) * K + k;
      floatx4 acc[BT][1];
      rg_walk<BT, 1, NS>(xp, wp, nst, smem + wave * NS * rg_stage(BT, 1), acc);
      rg_sums<BT, 1>(smem, acc, [&](int m, const floatx4 (&t)[1]) {
        const int row = m0 + m * 16 + (lane & 15);
        if (row >= p.M) return;
        uint2 pk;
        pk.x = pack_bf2(t[0][0], t[0][1]);
        pk.y = pack_bf2(t[0][2], t[0][3]);
        *reinterpret_cast<uint2*>(p.y + (long)row * p.ldy + column * 16 + 4 * (lane >> 4)) = pk;
      });
      return;
    }
    at -= p.nb;
  }
  const int e = at / blocks, cb = at % blocks;
  if constexpr (!ACT) {   // the pairs of rows that are not live, behind the experts' (lk_moe_route): zeros
    if (e == 0)
      for (long place = seg[E] + (threadIdx.x >> 3); place < pairs; place += 32)
        *reinterpret_cast<uint2*>(out + (long)order[place] * os + cb * 32 + 4 * (threadIdx.x & 7)) = make_uint2(0, 0);
  }
  const int end = seg[e + 1], F = ACT ? N / 2 : N, c0 = cb * (ACT ? 16 : 32);
  const int all = K / 64, first = wave * all / kRgWaves, nst = (wave + 1) * all / kRgWaves - first;
  const int lrow = lane >> 3;
  const long k = (long)first * 64 + rg_lane_col(lane);
  const bf16_t* ws[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i)
    ws[i] = w + ((long)e * N + (ACT ? (long)(i >> 1) * F : (i >> 1) * 16) + c0 + 8 * (i & 1) + lrow) * K + k;
  for (int place0 = seg[e]; place0 < end; place0 += 16 * MT) {
    const bf16_t* xp[2 * MT];
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i) {
      const int place = min(place0 + 8 * i + lrow, end - 1);  // rows past the expert's last pair repeat it
      xp[i] = x + (long)(ACT ? order[place] / top : place) * xs + k;
    }
    floatx4 acc[MT][NT];
    rg_walk<MT, NT, NS>(xp, ws, nst, smem + wave * NS * rg_stage(MT, NT), acc);
    rg_sums<MT, NT>(smem, acc, [&](int m, const floatx4 (&t)[NT]) {
      const int place = place0 + m * 16 + (lane & 15), col = c0 + 4 * (lane >> 4);
      if (place >= end) return;
      bf16_t* dst = out + (long)(ACT ? place : order[place]) * os + col;
#pragma unroll
      for (int n = 0; n < (ACT ? 1 : NT); ++n) {
        float y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) y[j] = ACT ? t[0][j] * __builtin_amdgcn_rcpf(1.f + __expf(-t[0][j])) * t[1][j] : t[n][j];
        uint2 pk;
        pk.x = pack_bf2(y[0], y[1]);
        pk.y = pack_bf2(y[2], y[3]);
        *reinterpret_cast<uint2*>(dst + 16 * n) = pk;
      }
    });
    __syncthreads();  // the sums are read: the rings are free again
  }
}

template <int MT>
int launch_moe_beside(const void* x, long xs, const int* order, const int* seg, int E, int top, const void* w, int N, int K, void* out,
                      long os, Beside p, hipStream_t st) {
  constexpr int lds = rg_lds(MT, 2, 3);
  static_assert(rg_lds(MT + 1, 1, 3) <= lds, "both tiles in one workgroup's LDS");
  LK_SET_MAX_LDS((moe_rows_kernel<true, MT, true>), lds);
  p.nb = (p.N / 16 + 7) / 8 * 8 * ((p.M + 16 * (MT + 1) - 1) / (16 * (MT + 1)));
  moe_rows_kernel<true, MT, true><<<(unsigned)(p.nb + (long)E * (N / 32)), 256, lds, st>>>((const bf16_t*)x, xs, order, seg, top, (const bf16_t*)w, N, K,
                                                                                      (bf16_t*)out, os, N / 32, 0, E, p);
  LK_CHECK_LAUNCH();
  return 0;
}

template <bool ACT, int MT>
int launch_moe_rows(const void* x, long xs, const int* order, const int* seg, int E, int top, long pairs, const void* w, int N, int K, void* out,
                    long os, hipStream_t st) {
  const int blocks = N / 32;  // 16 output columns of two weight rows each, or 32
  constexpr int lds = rg_lds(MT, 2, 3);
  LK_SET_MAX_LDS((moe_rows_kernel<ACT, MT>), lds);
  moe_rows_kernel<ACT, MT><<<(unsigned)((long)E * blocks), 256, lds, st>>>((const bf16_t*)x, xs, order, seg, top, (const bf16_t*)w, N, K,
                                                                          (bf16_t*)out, os, blocks, pairs, E, Beside{});
  LK_CHECK_LAUNCH();
  return 0;
}

template <typename T>
int moe_gemm_t(const void* x, long xs, const int* order, const int* seg, int E, int top, long pairs, const void* w, int N, int K,
               int act, void* out, long os, int vec, hipStream_t st) {
  // wide row tiles once an expert has 64 pairs on average (a choice by sizes the host knows: the same for every replay)
  const bool wide = pairs >= 64L * E;
  if (wide && vec) {   // 128-pair tiles staged in LDS (256-pair tiles, RT = 8, measured slower: 575 us against 365 us)
    return act ? launch_moe_lds<T, true, 4>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, st)
               : launch_moe_lds<T, false, 4>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, st);
  }
  if constexpr (sizeof(T) == 2) {
    // whole 64-column stages and 16-column blocks, 8-byte stores; rows per walk by the pairs an expert has on average (a third
    // more than the mean keeps a second walk rare).  A skewed table's further walks come one after the other, out of caches: both
    // products of 64 tokens, 12 pairs in the fullest of 16 experts / 40 / 64 in each of two: 93 / 109 / 85 us (tiles of 16 pairs over
    // the chip, moe_gemm_kernel: 183 / 195 / 92); of 300 tokens, 46 / 173 / 300: 148 / 179 / 138 us (329 / 324 / 268).
    if (vec && K % 64 == 0 && N % 32 == 0 && os % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 8 == 0 && (long)E * (N / 32) <= 2147483647L) {
      const long avg = pairs / E;
#define LK_MOE_ROWS(MT)                                                                           \
  (act ? launch_moe_rows<true, MT>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, st)        \
       : launch_moe_rows<false, MT>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, st))
      return avg <= 10 ? LK_MOE_ROWS(1) : avg <= 22 ? LK_MOE_ROWS(2) : LK_MOE_ROWS(4);
#undef LK_MOE_ROWS
    }
  }
  if (act) return wide ? launch_moe<T, true, 4>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, vec, st)
                       : launch_moe<T, true, 1>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, vec, st);
  return wide ? launch_moe<T, false, 4>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, vec, st)
              : launch_moe<T, false, 1>(x, xs, order, seg, E, top, pairs, w, N, K, out, os, vec, st);
}

}  // namespace

// Whether both products of T rows run as moe_rows_kernel (aligned operands), which gives zeros for the rows that are not live
int lk_moe_rows_ok(long T, int top, int E, int W, int ff) {
  return T >= 1 && top >= 1 && E >= 1 && T * top < 64L * E && W % 64 == 0 && ff % 64 == 0 && (long)E * (max(2 * ff, W) / 32) <= 2147483647L;
}

// seg [tables][E + 1], order [tables][T * top].  live (or null): the pairs of a row with live < 0 are no expert's and stand behind all others, from
// seg[E] on.  A step captured for 48 rows that has 33 ran its 15 empty ones as token 0, all through the same experts: a second walk over their
// weights (16 experts of 2,048 x 2,816, gate / up 64 us for 57), or experts that nobody else needs.  Four steps of eight such layers, us, with the
// gate beside the experts: 3 sequences 3,291 -> 2,741, 5 3,747 -> 3,144, 17 4,742 -> 4,384, 33 5,525 -> 4,889, 64 5,410 -> 5,068.
int lk_moe_route(const int* ids, const int* live, const int* const* tables, int n, int vocab, int top, int E, int T, int* seg, int* order, hipStream_t st) {
  if (T <= 0) return 0;
  if (E < 1 || E > kMaxExperts || top < 1 || vocab < 1 || n < 1 || n > kMaxRouteTables) return -1;
  RouteTables rt = {};
  for (int i = 0; i < n; ++i) rt.t[i] = tables[i];
  if ((long)T * top <= kRouteThreads) moe_route_kernel<1><<<n, kRouteThreads, 0, st>>>(ids, live, rt, vocab, top, E, T, seg, order);
  else moe_route_kernel<kRouteU><<<n, kRouteThreads, 0, st>>>(ids, live, rt, vocab, top, E, T, seg, order);
  LK_CHECK_LAUNCH();
  return 0;
}

// 16-row tiles of an expert's pairs per walk where the gate runs beside; a workgroup of the gate takes one more of rows
static int beside_tiles(long T, int top, int E) { return T * top / E <= 10 ? 1 : 2; }

// Whether the gate of T rows runs beside the experts' first product: the few-row kernel for both, and the launch that it saves worth more than X
// and W read again out of the L2s, X for every 16 columns and W for every tile of rows.  Those bytes come at 16 MB/us beside the experts' stream;
// on its own the gate takes 2.7 us and its weight at 6.6 MB/us.  Over 456 products (width 512 - 7,168, gates of 256 columns to twice the
// width, 4 - 64 experts of 512 - 14,336, 1 - 96 rows) 0.903 of the time apart, 0.2 % more than the better of both; all of them beside, 0.915.
// Apart / beside, us, 8 / 40 / 80 rows: 2,048 x 2,048 with 16 experts of 2,816 37.9 / 60.5 / 72.1 -> 34.0 / 58.4 / 71.2, 4,096 x 4,096 with 16 of 1,536
// 45.4 / 71.4 / 74.0 -> 43.1 / 74.7 / 81.4, 7,168 x 7,168 with 16 of 2,048 96.7 / 159.7 / 169.0 -> 98.2 / 184.4 / 204.7.
int lk_moe_beside_ok(long T, int top, int E, int N, int K, int N2) {
  if (T < 1 || T > 96 || top < 1 || E < 1 || T * top > 22L * E || K < 1 || K % 64 || N < 1 || N % 32 || N2 < 1 || N2 % 16 || (long)E * (N / 32) > 1 << 30) return 0;
  const int rows = beside_tiles(T, top, E) + 1;   // 16-row tiles of one workgroup
  const double again = (double)(N2 / 16) * ((T + 16 * rows - 1) / (16 * rows)) * (rows + 1) * 16 * K * 2e-6;
  return again / 16 + 0.5 < 2.7 + (double)N2 * K * 2e-6 / 6.6;
}

int lk_moe_gemm_beside(const void* x, long xs, const int* order, const int* seg, int E, int top, long T, const void* w, int N, int K,
                       void* out, long os, const void* w2, int N2, void* y2, long ldy, hipStream_t st) {
  const auto al = [](const void* p, int n) { return reinterpret_cast<uintptr_t>(p) % n == 0; };
  if (!lk_moe_beside_ok(T, top, E, N, K, N2) || xs % 8 || os % 4 || ldy % 4 || !al(x, 16) || !al(w, 16) || !al(w2, 16) || !al(out, 8) || !al(y2, 8)) return -1;
  const Beside p{(const bf16_t*)w2, (bf16_t*)y2, ldy, (int)T, N2, 0};
  return beside_tiles(T, top, E) == 1 ? launch_moe_beside<1>(x, xs, order, seg, E, top, w, N, K, out, os, p, st)
                                      : launch_moe_beside<2>(x, xs, order, seg, E, top, w, N, K, out, os, p, st);
}

int lk_moe_gemm(const void* x, long xs, const int* order, const int* seg, int E, int top, long pairs, const void* w, int N, int K,
                int act, void* out, long os, int esz, hipStream_t st) {
  if (pairs <= 0) return 0;
  if (E < 1 || top < 1 || N < 1 || K < 1 || (act && N % 2)) return -1;
  const int ev = 16 / esz;
  const int vec = K % ev == 0 && xs % ev == 0 && reinterpret_cast<uintptr_t>(x) % 16 == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0;
  return esz == 2 ? moe_gemm_t<bf16_t>(x, xs, order, seg, E, top, pairs, w, N, K, act, out, os, vec, st)
                  : moe_gemm_t<float>(x, xs, order, seg, E, top, pairs, w, N, K, act, out, os, vec, st);
}
