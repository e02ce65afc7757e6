// K6 brute-force cosine kNN with fused top-k over a corpus resident in HBM.
//
// Semantics follow RagIndex.Cosine / QueryAsync (reference
// Minimal_RAG/Helpers/RagIndex.cs:59-67,124-135): score = dot / (|q|*|c| + 1e-9),
// dimension mismatch is rejected on the host, results ordered by descending score
// with ties kept in corpus (insertion) order — i.e. a stable sort.
//
// Pass 1 (lk_knn_partial): workgroup = 256 corpus rows x 32 queries.  Each wave
// computes two 32x32 score tiles with v_mfma_f32_32x32x16_bf16 (A = corpus rows
// read straight from HBM, B = Q^T from a swizzled LDS image).  The MFMA k-order is
// permuted so every lane streams 64 contiguous bytes of its corpus row per group of
// 4 k-steps (the reduction order of a dot product is free).  Scores are staged in
// LDS and each wave extracts the block-local top-k of 8 queries by k rounds of
// wave-wide (score, index) argmax.
// Few queries (lk_knn_scan, <= 16 queries, K <= 8, the serving path): one persistent pass over the corpus that
// keeps its best rows as it goes, and a merge of its workgroups' lists; see knn_scan_kernel.
// Pass 2 (lk_knn_merge): one workgroup per query merges nblocks*k candidates with
// the same tie rule.  Sharded (multi-GPU) search reuses pass 2 on all-gathered
// candidates.
#include "common.h"
#include "kernels.h"
#include "row_ring.h"

namespace {

constexpr int ROWS = 256;  // corpus rows per workgroup
constexpr int QT = 32;     // queries per workgroup

// (score desc, index asc) ordering
LK_DEVICE bool better(float s1, int i1, float s2, int i2) {
  return s1 > s2 || (s1 == s2 && (unsigned)i1 < (unsigned)i2);
}

LK_DEVICE void wave_argmax(float& s, int& i) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const float s2 = __shfl_xor(s, o, 64);
    const int i2 = __shfl_xor(i, o, 64);
    if (better(s2, i2, s, i)) {
      s = s2;
      i = i2;
    }
  }
}

// A hit as one number that orders as (score desc, index asc) does: the score's bits made monotonic, then the index's complement; 0: none.
// (Both zeros are one score.)
typedef unsigned long long hit_t;
LK_DEVICE hit_t hit_of(float s, int i) {
  const unsigned u = __float_as_uint(s + 0.f);
  return s == -INFINITY ? 0 : (hit_t)(u ^ ((unsigned)((int)u >> 31) | 0x80000000u)) << 32 | (unsigned)~i;
}
LK_DEVICE float hit_score(hit_t h) {
  const unsigned u = (unsigned)(h >> 32);
  return h == 0 ? -INFINITY : __uint_as_float(u >> 31 ? u ^ 0x80000000u : ~u);
}
LK_DEVICE int hit_index(hit_t h) { return h == 0 ? -1 : (int)~(unsigned)h; }

// the best of groups of 16 lanes, by row rotations of the vector unit (every lane ends with it)
template <int STEP>
LK_DEVICE hit_t rotate_best(hit_t h) {
  const unsigned lo = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)h, 0x120 + STEP, 0xf, 0xf, true);
  const unsigned hi = (unsigned)__builtin_amdgcn_update_dpp(0, (int)(unsigned)(h >> 32), 0x120 + STEP, 0xf, 0xf, true);
  const hit_t o = (hit_t)hi << 32 | lo;
  return o > h ? o : h;
}
LK_DEVICE hit_t row_best(hit_t h) { return rotate_best<1>(rotate_best<2>(rotate_best<4>(rotate_best<8>(h)))); }
// ... of pairs of them (lanes l and l ^ 16)
LK_DEVICE hit_t rows_best(hit_t h) {
  h = row_best(h);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)h, (unsigned)h, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(h >> 32), (unsigned)(h >> 32), false, false);
  const unsigned l0 = lo[0], l1 = lo[1], h0 = hi[0], h1 = hi[1];
  const hit_t a = (hit_t)h0 << 32 | l0, b = (hit_t)h1 << 32 | l1;
  return a > b ? a : b;
}

template <int D>
__global__ __launch_bounds__(256) void knn_partial_kernel(
    const bf16_t* __restrict__ corpus, const float* __restrict__ cnorm, long N,
    const bf16_t* __restrict__ queries, const float* __restrict__ qnorm, int nq, int K,
    float* __restrict__ part_s, int* __restrict__ part_i, int nblocks) {
  constexpr int CPR = D / 8;  // 16-B chunks per row
  constexpr int NG = D / 64;  // groups of 4 k-steps
  // one LDS buffer: the Q tile during the MFMA phase, then (after a barrier) the score
  // tile for the top-k phase -- max(QT*D*2, QT*(ROWS+1)*4) bytes instead of the sum,
  // so 2-3 workgroups fit per CU
  constexpr int QBYTES = QT * D * 2, SBYTES = QT * (ROWS + 1) * 4;
  __shared__ __attribute__((aligned(16))) unsigned char smem[QBYTES > SBYTES ? QBYTES : SBYTES];
  bf16_t* Qs = reinterpret_cast<bf16_t*>(smem);
  float(*sc)[ROWS + 1] = reinterpret_cast<float(*)[ROWS + 1]>(smem);
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const int r = lane & 31, h = lane >> 5;
  const int qbase = blockIdx.y * QT;
  const long row0 = (long)blockIdx.x * ROWS;

  // stage Q tile (zero-padded) with chunk swizzle c ^ (row & 15)
  for (int c = tid; c < QT * CPR; c += 256) {
    const int qr = c / CPR, ch = c % CPR;
    short8 v = short8{0, 0, 0, 0, 0, 0, 0, 0};
    if (qbase + qr < nq) v = *reinterpret_cast<const short8*>(queries + (long)(qbase + qr) * D + ch * 8);
    *reinterpret_cast<short8*>(Qs + qr * D + (ch ^ (qr & 15)) * 8) = v;
  }
  __syncthreads();

  // k-step (4g+u), element j  <->  d = 64g + 32h + 8u + j
  floatx16 acc2[2];
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    const long doc = row0 + w * 64 + m * 32 + r;
    const long docc = doc < N ? doc : N - 1;
    const bf16_t* cp = corpus + docc * D + 32 * h;
    floatx16 acc;
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[i] = 0.f;
#pragma unroll 2
    for (int g = 0; g < NG; ++g) {
      short8 a[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) a[u] = *reinterpret_cast<const short8*>(cp + 64 * g + 8 * u);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int ch = 8 * g + 4 * h + u;
        const short8 bq = *reinterpret_cast<const short8*>(Qs + r * D + (ch ^ (r & 15)) * 8);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[u], bq, acc, 0, 0, 0);
      }
    }
    acc2[m] = acc;
  }
  __syncthreads();  // every wave done with Qs: the buffer becomes the score tile
  // C[row = doc (i&3)+8(i>>2)+4h][col = query r]
  const float qn = (qbase + r < nq) ? qnorm[qbase + r] : 1.f;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      const int lr = w * 64 + m * 32 + (i & 3) + 8 * (i >> 2) + 4 * h;
      const long d = row0 + lr;
      sc[r][lr] = d < N ? acc2[m][i] / (qn * cnorm[d] + 1e-9f) : -INFINITY;
    }
  }
  __syncthreads();

  // block-local top-k: wave w handles queries w, w+4, ...
  for (int qq = w; qq < QT; qq += 4) {
    if (qbase + qq >= nq) break;
    float v[ROWS / 64];
#pragma unroll
    for (int j = 0; j < ROWS / 64; ++j) v[j] = sc[qq][lane + 64 * j];
    float* ps = part_s + ((long)(qbase + qq) * nblocks + blockIdx.x) * K;
    int* pi = part_i + ((long)(qbase + qq) * nblocks + blockIdx.x) * K;
    for (int kk = 0; kk < K; ++kk) {
      float bs = -INFINITY;
      int bi = 0x7fffffff;
#pragma unroll
      for (int j = 0; j < ROWS / 64; ++j) {
        const int idx = (int)(row0 + lane + 64 * j);
        if (better(v[j], idx, bs, bi)) {
          bs = v[j];
          bi = idx;
        }
      }
      wave_argmax(bs, bi);
      if (lane == 0) {
        ps[kk] = bs;
        pi[kk] = bs == -INFINITY ? -1 : bi;
      }
#pragma unroll
      for (int j = 0; j < ROWS / 64; ++j)
        if ((int)(row0 + lane + 64 * j) == bi) v[j] = -INFINITY;
    }
  }
}

// Top-k over precomputed dot products (scores [nq, ld] from the weight-streaming GEMM,
// csrc/skinny_gemm.hip lk_ws_scores_f32): one workgroup per (chunk of 4096 rows, query)
// normalises dot / (|q| |c| + 1e-9) and extracts the chunk's top-k (score desc, index
// asc) by k rounds of block-wide argmax.
constexpr int SCH = 4096;

__global__ __launch_bounds__(256) void score_topk_kernel(const float* __restrict__ scores, long ld,
                                                         const float* __restrict__ cnorm,
                                                         const float* __restrict__ qnorm, long N, int K,
                                                         float* __restrict__ part_s, int* __restrict__ part_i,
                                                         int nchunks) {
  __shared__ float rs[4];
  __shared__ int ri[4];
  const int q = blockIdx.y, c = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  constexpr int PER = SCH / 256;
  const long base = (long)c * SCH;
  const float qn = qnorm[q];
  float v[PER];
#pragma unroll
  for (int j = 0; j < PER; ++j) {
    const long d = base + j * 256 + tid;
    v[j] = d < N ? scores[(long)q * ld + d] / (qn * cnorm[d] + 1e-9f) : -INFINITY;
  }
  float* ps = part_s + ((long)q * nchunks + c) * K;
  int* pi = part_i + ((long)q * nchunks + c) * K;
  for (int kk = 0; kk < K; ++kk) {
    float bs = -INFINITY;
    int bi = 0x7fffffff;
#pragma unroll
    for (int j = 0; j < PER; ++j) {
      const int idx = (int)(base + j * 256 + tid);
      if (better(v[j], idx, bs, bi)) {
        bs = v[j];
        bi = idx;
      }
    }
    wave_argmax(bs, bi);
    if (lane == 0) {
      rs[w] = bs;
      ri[w] = bi;
    }
    __syncthreads();
    float fs = rs[0];
    int fi = ri[0];
#pragma unroll
    for (int j = 1; j < 4; ++j)
      if (better(rs[j], ri[j], fs, fi)) {
        fs = rs[j];
        fi = ri[j];
      }
    if (tid == 0) {
      ps[kk] = fs;
      pi[kk] = fs == -INFINITY ? -1 : fi;
    }
#pragma unroll
    for (int j = 0; j < PER; ++j)
      if ((int)(base + j * 256 + tid) == fi) v[j] = -INFINITY;
    __syncthreads();
  }
}

// merge: one workgroup per query over `ncand` (score, idx) candidates
__global__ __launch_bounds__(256) void knn_merge_kernel(const float* __restrict__ cs,
                                                        const int* __restrict__ ci, int ncand,
                                                        int K, float* __restrict__ out_s,
                                                        int* __restrict__ out_i) {
  __shared__ float rs[4];
  __shared__ int ri[4];
  __shared__ int last;
  const int q = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
  const float* s = cs + (long)q * ncand;
  const int* ix = ci + (long)q * ncand;
  float prev_s = INFINITY;
  int prev_i = -1;
  for (int kk = 0; kk < K; ++kk) {
    // best candidate strictly "worse" than the previous winner
    float bs = -INFINITY;
    int bi = 0x7fffffff;
    for (int c = tid; c < ncand; c += 256) {
      const float v = s[c];
      const int id = ix[c];
      if (id < 0) continue;
      if (kk > 0 && !better(prev_s, prev_i, v, id)) continue;
      if (better(v, id, bs, bi)) {
        bs = v;
        bi = id;
      }
    }
    wave_argmax(bs, bi);
    if (lane == 0) {
      rs[w] = bs;
      ri[w] = bi;
    }
    __syncthreads();
    if (tid == 0) {
      float fs = rs[0];
      int fi = ri[0];
      for (int j = 1; j < 4; ++j)
        if (better(rs[j], ri[j], fs, fi)) {
          fs = rs[j];
          fi = ri[j];
        }
      out_s[(long)q * K + kk] = fs;
      out_i[(long)q * K + kk] = fi == 0x7fffffff ? -1 : fi;
      rs[0] = fs;
      ri[0] = fi;
    }
    __syncthreads();
    prev_s = rs[0];
    prev_i = ri[0];
    __syncthreads();
  }
  (void)last;
}

// One pass for up to 16 queries and K <= 8.  The corpus is read once (746 MB at 485,620 x 768) and nothing of its size is
// written: the two-pass form wrote and re-read f32 scores of every row (31 MB at 16 queries) and paid two more launches.
// 8 waves per CU, each with the queries' fragments in registers (D / 32 of them) and a private LDS ring of 10 stages of
// 16 rows x 128 bytes (row_ring.h), walk 16-row tiles round robin without a barrier, so 144 KB of corpus are on their way
// per CU.  A lane sees 4 rows of one query per tile and keeps its 8 best in order (rows come in ascending order, so an
// equal score never displaces: the stable order); 32 lists per query meet in LDS at the end.
// What bounds it: the stream of rows at 485,620 x 768 (116 us, 6.4 TB/s, and 4 for the merge; 131 and 6 with a wait per number of stages
// left, row addresses per stage and reductions through the LDS unit); at 20,011 rows the chain of launch, code and first loads: of 10 us the
// rows come between the third and the ninth, the lists and the merge of a workgroup take the rest.  Four waves per CU had a quarter of their
// tiles behind another and met one LDS bank with all lists (13.2 us), and hits in two words compared in three steps (11.2); one question in
// all 29.0 -> 26.5 us, 16 over 485,620 150 -> 145.  The scores' own two-pass form took 158 + 26 + 10 and 11 + 12 + 5.
constexpr int kScanK = 8, kScanQ = 16, kScanStages = 10, kScanWaves = 8, kScanLists = 4 * kScanWaves;

// ls / li descending: s, i enters behind everything that is not smaller
LK_DEVICE void list_insert(float s, int i, float (&ls)[kScanK], int (&li)[kScanK]) {
#pragma unroll
  for (int j = kScanK - 1; j >= 1; --j) {
    const bool here = s > ls[j], above = s > ls[j - 1];
    ls[j] = here ? (above ? ls[j - 1] : s) : ls[j];
    li[j] = here ? (above ? li[j - 1] : i) : li[j];
  }
  if (s > ls[0]) {
    ls[0] = s;
    li[0] = i;
  }
}

// the head leaves (of the padding behind a short list, all heads do: nothing follows it)
LK_DEVICE void list_pop(hit_t (&l)[kScanK]) {
#pragma unroll
  for (int j = 0; j + 1 < kScanK; ++j) l[j] = l[j + 1];
  l[kScanK - 1] = 0;
}

template <int SEG>
__global__ __launch_bounds__(64 * kScanWaves, 1) void knn_scan_kernel(const bf16_t* __restrict__ corpus, const float* __restrict__ cnorm, long N,
                                                          const bf16_t* __restrict__ queries, const float* __restrict__ qnorm, int nq,
                                                          int K, hit_t* __restrict__ part) {
  constexpr int D = SEG * 64, NS = kScanStages;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), r16 = lane & 15, g = lane >> 4;
  // (a workgroup's waves are a grid apart: where there are fewer tiles than waves, every CU has as many)
  const int tiles = (int)((N + 15) / 16), first = w * gridDim.x + blockIdx.x, step = gridDim.x * kScanWaves;
  const int total = first < tiles ? ((tiles - 1 - first) / step + 1) * SEG : 0;  // this wave's stages
  short8 qf[2 * SEG] = {};
  if (total > 0) {   // (a wave without a tile asks for nothing: 16 queries are up to 32 KB that the other waves would wait behind)
    const bf16_t* q = queries + (long)min(r16, nq - 1) * D + 8 * g;
#pragma unroll
    for (int k = 0; k < 2 * SEG; ++k) qf[k] = *reinterpret_cast<const short8*>(q + 32 * k);
  }
  const float qgiven = qnorm ? qnorm[min(r16, nq - 1)] : 0.f;
  unsigned char* const ring = smem + w * NS * 2048;
  const int lrow = lane >> 3, lcol = rg_lane_col(lane);
  const bf16_t* src[2];  // this lane's part of the tile being requested
  int ist = 0, to = 0;   // stages requested; where the next goes
  auto issue = [&](int seg, long tile) {
    if (seg == 0) {
#pragma unroll
      for (int i = 0; i < 2; ++i) src[i] = corpus + min(tile * 16 + 8 * i + lrow, N - 1) * D + lcol;
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) __builtin_amdgcn_global_load_lds((rg_gptr)(src[i] + seg * 64), (rg_lptr)(ring + to + i * 1024), 16, 0, 2);
    ++ist;
    to = to + 2048 == NS * 2048 ? 0 : to + 2048;
  };
#pragma unroll
  for (int p = 0; p < NS - 1; ++p)
    if (p < total) issue(p % SEG, first + (long)(p / SEG) * step);
  // the queries' norms: the diagonal of Q Q^T, in four chains (one chain of D / 32 sums would cost the norm its last bits; against
  // float64 the scores of 640 queries are off by 0.85e-7 (D 128) to 1.8e-7 (1,024) rms, as with eight products at a time in the vector unit)
  float qn = qgiven;
  if (!qnorm) {
    floatx4 n[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) n[c] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int k = 0; k < 2 * SEG; ++k) n[k & 3] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(qf[k], qf[k], n[k & 3], 0, 0, 0);
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 4; ++j)
      if (4 * g + j == r16) ss = (n[0][j] + n[1][j]) + (n[2][j] + n[3][j]);
    ss += __shfl_xor(ss, 16, 64);
    ss += __shfl_xor(ss, 32, 64);
    qn = sqrtf(ss);
  }
  // (the compiler's wait for the queries belongs here: in the loop it would drain the ring at every tile)
#pragma unroll
  for (int k = 0; k < 2 * SEG; ++k) asm volatile("" : "+v"(qf[k]));
  float ls[kScanK];
  int li[kScanK];
#pragma unroll
  for (int j = 0; j < kScanK; ++j) {
    ls[j] = -INFINITY;
    li[j] = 0x7fffffff;
  }
  int st = 0, from = 0;
  for (long t = first; t < tiles; t += step) {
    const long d0 = t * 16 + 4 * g;
    float cn[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) cn[j] = cnorm[min(d0 + j, N - 1)];
    floatx4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int seg = 0; seg < SEG; ++seg, ++st) {
      // Two waits, not one per number of stages left: all of the last NS - 1 are waited for at once, which is 0.3 us of a wave's end, and
      // the code of a stage is a tenth (a short scan runs it once and fetching it is what it waits for)
      if (total - 1 - st >= NS - 2) rg_wait<2 * (NS - 2)>();
      else rg_wait<0>();
      __builtin_amdgcn_sched_barrier(0);
      if (ist < total) issue((seg + NS - 1) % SEG, t + (long)((seg + NS - 1) / SEG) * step);
      __builtin_amdgcn_sched_barrier(0);
      const unsigned char* base = ring + from;
      from = from + 2048 == NS * 2048 ? 0 : from + 2048;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const short8 a = *reinterpret_cast<const short8*>(base + r16 * 128 + (((4 * h + g) ^ (r16 & 7)) << 4));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, qf[2 * seg + h], acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float s = d0 + j < N ? acc[j] / (qn * cn[j] + 1e-9f) : -INFINITY;
      if (s > ls[kScanK - 1]) list_insert(s, (int)(d0 + j), ls, li);
    }
  }
  // [kScanK][kScanLists: 8 waves x 4 lane groups][query], a query's words 17 apart: neither side meets a bank twice, and lanes without a
  // query write nothing (lists of 8 words each behind the other met one bank 16 at a time)
  __syncthreads();
  constexpr int LQ = kScanQ + 1;
  hit_t* ml = reinterpret_cast<hit_t*>(smem);
  if (r16 < nq) {
#pragma unroll
    for (int j = 0; j < kScanK; ++j) ml[(j * kScanLists + w * 4 + g) * LQ + r16] = hit_of(ls[j], li[j]);
  }
  __syncthreads();
  // a wave takes two queries at once, a lane one of their 32 lists: K rounds over the lists' heads
  if (w * 2 < nq) {
    const int q = min(w * 2 + (lane >> 5), nq - 1), l = lane & 31;
    const bool mine = w * 2 + (lane >> 5) < nq;
    hit_t v[kScanK];
#pragma unroll
    for (int j = 0; j < kScanK; ++j) v[j] = ml[(j * kScanLists + l) * LQ + q];
    for (int k = 0; k < K; ++k) {
      const hit_t best = rows_best(v[0]);
      if (l == 0 && mine) part[((long)q * gridDim.x + blockIdx.x) * K + k] = best;
      if (v[0] == best) list_pop(v);
    }
  }
}

// merge of at most 256 lists of K <= 8, each in order: one workgroup per query, a list per thread; every 16 lanes take the
// K best of their lists by the lists' heads, then 16 lanes those of the 16 groups
__global__ __launch_bounds__(256) void knn_merge_lists_kernel(const hit_t* __restrict__ part, int lists, int K, float* __restrict__ out_s,
                                                              int* __restrict__ out_i) {
  __shared__ hit_t rl[16][kScanK];
  const int q = blockIdx.x, tid = threadIdx.x, l16 = tid & 15, grp = tid >> 4;
  hit_t v[kScanK];
#pragma unroll
  for (int j = 0; j < kScanK; ++j) v[j] = tid < lists && j < K ? part[((long)q * lists + tid) * K + j] : 0;
  for (int k = 0; k < K; ++k) {
    const hit_t best = row_best(v[0]);
    if (l16 == 0) rl[grp][k] = best;
    if (v[0] == best) list_pop(v);
  }
  __syncthreads();
  if (grp) return;
#pragma unroll
  for (int j = 0; j < kScanK; ++j) v[j] = j < K ? rl[l16][j] : 0;
  for (int k = 0; k < K; ++k) {
    const hit_t best = row_best(v[0]);
    if (l16 == 0) {  // (each word once, at system scope: in pinned memory the host sees it arrive)
      __hip_atomic_store(out_s + (long)q * K + k, hit_score(best), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
      __hip_atomic_store(out_i + (long)q * K + k, hit_index(best), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    if (v[0] == best) list_pop(v);
  }
}

template <int SEG>
int launch_scan(const bf16_t* corpus, const float* cnorm, long N, const bf16_t* queries, const float* qnorm, int nq, int K, int nb,
                hit_t* part, hipStream_t st) {
  constexpr int lds = kScanWaves * kScanStages * 2048;
  static_assert(lds >= 8 * kScanK * kScanLists * (kScanQ + 1), "the lists at the end");
  LK_SET_MAX_LDS((knn_scan_kernel<SEG>), lds);
  knn_scan_kernel<SEG><<<nb, 64 * kScanWaves, lds, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part);
  LK_CHECK_LAUNCH();
  return 0;
}

}  // namespace

int lk_knn_nblocks(long N) { return (int)((N + ROWS - 1) / ROWS); }

int lk_knn_partial(const bf16_t* corpus, const float* cnorm, long N, int D, const bf16_t* queries,
                   const float* qnorm, int nq, int K, float* part_s, int* part_i,
                   hipStream_t st) {
  if (N <= 0 || nq <= 0) return 0;
  if (K < 1 || K > 64) return -1;
  const int nb = lk_knn_nblocks(N);
  dim3 grid(nb, (nq + QT - 1) / QT);
  switch (D) {
    case 128: knn_partial_kernel<128><<<grid, 256, 0, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part_s, part_i, nb); break;
    case 256: knn_partial_kernel<256><<<grid, 256, 0, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part_s, part_i, nb); break;
    case 512: knn_partial_kernel<512><<<grid, 256, 0, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part_s, part_i, nb); break;
    case 384: knn_partial_kernel<384><<<grid, 256, 0, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part_s, part_i, nb); break;
    case 768: knn_partial_kernel<768><<<grid, 256, 0, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part_s, part_i, nb); break;
    case 1024: knn_partial_kernel<1024><<<grid, 256, 0, st>>>(corpus, cnorm, N, queries, qnorm, nq, K, part_s, part_i, nb); break;
    default: return -2;
  }
  return 0;
}

int lk_knn_score_chunks(long N) { return (int)((N + SCH - 1) / SCH); }

int lk_knn_score_topk(const float* scores, long ld, const float* cnorm, const float* qnorm, long N, int nq, int K,
                      float* part_s, int* part_i, hipStream_t st) {
  if (N <= 0 || nq <= 0) return 0;
  if (K < 1 || K > 64) return -1;
  const int nc = lk_knn_score_chunks(N);
  score_topk_kernel<<<dim3(nc, nq), 256, 0, st>>>(scores, ld, cnorm, qnorm, N, K, part_s, part_i, nc);
  return 0;
}

int lk_knn_merge(const float* cand_s, const int* cand_i, int nq, int ncand, int K, float* out_s,
                 int* out_i, hipStream_t st) {
  if (nq <= 0) return 0;
  knn_merge_kernel<<<nq, 256, 0, st>>>(cand_s, cand_i, ncand, K, out_s, out_i);
  return 0;
}

// workgroups of the one-pass scan (0: it does not take this shape): one per four tiles of 16 rows, up to one per CU (up to 16,384 rows half of
// the waves have no tile)
int lk_knn_scan_blocks(long N, int D, int nq, int K) {
  if (N <= 0 || N >= 0x7fffffffL - 16 || nq < 1 || nq > kScanQ || K < 1 || K > kScanK) return 0;
  if (D != 128 && D != 256 && D != 384 && D != 512 && D != 768 && D != 1024) return 0;
  const long b = ((N + 15) / 16 + 3) / 4;
  return (int)(b < 256 ? b : 256);
}

// out_s / out_i [nq, K]; qnorm null: the queries' norms are taken here; part: [nq, blocks, K] of 8 bytes
int lk_knn_scan(const bf16_t* corpus, const float* cnorm, long N, int D, const bf16_t* queries, const float* qnorm, int nq, int K,
                void* part, float* out_s, int* out_i, hipStream_t st) {
  const int nb = lk_knn_scan_blocks(N, D, nq, K);
  if (!nb) return -1;
  int rc;
  switch (D) {
    case 128: rc = launch_scan<2>(corpus, cnorm, N, queries, qnorm, nq, K, nb, (hit_t*)part, st); break;
    case 256: rc = launch_scan<4>(corpus, cnorm, N, queries, qnorm, nq, K, nb, (hit_t*)part, st); break;
    case 384: rc = launch_scan<6>(corpus, cnorm, N, queries, qnorm, nq, K, nb, (hit_t*)part, st); break;
    case 512: rc = launch_scan<8>(corpus, cnorm, N, queries, qnorm, nq, K, nb, (hit_t*)part, st); break;
    case 768: rc = launch_scan<12>(corpus, cnorm, N, queries, qnorm, nq, K, nb, (hit_t*)part, st); break;
    default: rc = launch_scan<16>(corpus, cnorm, N, queries, qnorm, nq, K, nb, (hit_t*)part, st); break;
  }
  if (rc) return rc;
  knn_merge_lists_kernel<<<nq, 256, 0, st>>>((const hit_t*)part, nb, K, out_s, out_i);
  LK_CHECK_LAUNCH();
  return 0;
}
