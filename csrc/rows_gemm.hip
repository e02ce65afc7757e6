// K2 / K3, few rows: Y[M,N] = act(X[M,K] . W[N,K]^T + bias) for up to some hundred rows in ONE launch, bf16 in,
// f32 sums, one rounding (bias / bias + GELU / bias + ReLU / SwiGLU in the epilogue).
//
// What bounds it: at these sizes neither HBM (a 2048 x 2048 weight is 1.4 us of it) nor the matrix cores
// but the serial chain of a launch: a tiled kernel with a barrier per K stage waits for each of them, and
// a split-K one pays a second launch for its sum.  Here no wave waits for another inside the K walk:
//   * a workgroup of 4 waves owns 16 output columns (wide: 32 or 64; SwiGLU: half of them gate and half the up columns) and up
//     to 64 rows; the waves split K, so each element of X and W reaches the workgroup once;
//   * every wave streams its own K range through a private LDS ring by LDS-DMA (row_ring.h; loads straight into
//     the fragment layout, 16 rows x 64 bytes, ran at a quarter of the rate: 12.0 us against 7.7 at
//     64 x 2048 x 2048, 8.4 against 5.7 at 32 rows);
//   * the waves' sums meet once in LDS, then the epilogue stores 4 columns per lane;
//   * what a CU loads into LDS is then the time: 58 - 68 KB/us, with three stages of the ring in flight or with four.  So the
//     tile is the one with the fewest bytes per CU: 16 columns and few rows where that fills 256 CUs (64 x 2048 x 2048: 64 rows
//     6.9 us, 32 rows 6.0; K 5632: 15.6 -> 12.0; 64 x 768 x 3072: 16 rows 8.5 -> 5.2), 64 columns where N is large (64 x 10496 x
//     2048: 17.9 -> 14.3, SwiGLU 64 x 11264 x 2048: 17.2 -> 14.6; 32 columns need a second round of workgroups).
//     With many rows the re-reading of X out of L2 bounds it and the tiled kernels take over (ops: _rows_rule).
#include "common.h"
#include "kernels.h"
#include "row_ring.h"

namespace {

enum { RG_NONE = 0, RG_SWIGLU = 1, RG_BIAS = 2, RG_GELU = 3, RG_RELU = 4, RG_ADD = 5 };

// Grid (8 XCDs, row tiles, column tiles / 8 rounded up): the row tiles of a column tile follow one another on one XCD, whose L2 then has the
// weight rows.  From z = spread on (rows_spread: the last columns, fewer than 8) they go around over the XCDs instead.
// False: a workgroup without work.
LK_DEVICE bool rg_place(int z, int spread, int columns, int per, int& column, int& item) {
  column = z * 8 + blockIdx.x;
  item = blockIdx.y;
  if (__builtin_expect(z < spread, 1)) return column < columns;
  const int at = blockIdx.y * 8 + blockIdx.x, rest = columns - z * 8;
  column = z * 8 + at % rest;
  item = at / rest;
  return item < per;
}

template <int MT, int NT, int NS, int EPI>
LK_DEVICE void rows_tile(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W, const bf16_t* __restrict__ bias,
                         const bf16_t* __restrict__ R, long ldr, bf16_t* __restrict__ Y, int M, int N, int K, long ldx, long ldy, int cz, int spread) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int all = K / 64, first = wave * all / kRgWaves, nst = (wave + 1) * all / kRgWaves - first;  // stages of this wave
  const int cols = EPI == RG_SWIGLU ? N / 2 : N;
  asm volatile("" ::"s"(X), "s"(W), "s"(Y), "s"(ldx), "s"(ldy));   // (all arguments are loaded before the branch: 0.2 us for a second wait behind it)
  int column, item;
  if (!rg_place(cz, spread, N / (16 * NT), (M + 16 * MT - 1) / (16 * MT), column, item)) return;   // the whole workgroup
  const int n0 = column * (EPI == RG_SWIGLU ? 8 * NT : 16 * NT), m0 = item * (16 * MT);  // first output column and row
  X += (long)m0 * ldx;
  Y += (long)m0 * ldy;
  if constexpr (EPI == RG_ADD) R += (long)m0 * ldr;
  M = min(M - m0, 16 * MT);
  const int lrow = lane >> 3;
  const long k = (long)first * 64 + rg_lane_col(lane);
  const bf16_t* xs[2 * MT];
  const bf16_t* ws[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) xs[i] = X + (long)min(8 * i + lrow, M - 1) * ldx + k;  // rows past M repeat the last one
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) {
    const int t = i >> 1;   // W tile; SwiGLU: the second half are the up rows of the first half's columns
    constexpr int HT = NT > 1 ? NT / 2 : 1;
    const long row = EPI == RG_SWIGLU ? (long)(t / HT) * cols + t % HT * 16 : t * 16;
    ws[i] = W + (row + n0 + 8 * (i & 1) + lrow) * K + k;
  }
  floatx4 acc[MT][NT];
  rg_walk<MT, NT, NS>(xs, ws, nst, smem + wave * NS * rg_stage(MT, NT), acc);
  rg_sums<MT, NT>(smem, acc, [&](int m, const floatx4 (&t)[NT]) {
    const int row = m * 16 + (lane & 15), col = n0 + 4 * (lane >> 4);
    if (row >= M) return;
#pragma unroll
    for (int n = 0; n < (EPI == RG_SWIGLU ? NT / 2 : NT); ++n) {
      float y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (EPI == RG_SWIGLU) {  // rounded as the projection and the activation apart round
          y[j] = bf2f(f2bf(lk_silu(bf2f(f2bf(t[n][j]))))) * bf2f(f2bf(t[n + NT / 2][j]));
        } else {
          y[j] = t[n][j];
          if constexpr (EPI >= RG_BIAS) y[j] += bf2f(bias[col + 16 * n + j]);
          if constexpr (EPI == RG_GELU) y[j] = lk_gelu_erf(y[j]);
          if constexpr (EPI == RG_RELU) y[j] = fmaxf(y[j], 0.f);
          if constexpr (EPI == RG_ADD) y[j] = bf2f(f2bf(y[j])) + bf2f(R[(long)row * ldr + col + 16 * n + j]);  // rounded as the product and the sum apart
        }
      }
      uint2 pk;
      pk.x = pack_bf2(y[0], y[1]);
      pk.y = pack_bf2(y[2], y[3]);
      *reinterpret_cast<uint2*>(Y + (long)row * ldy + col + 16 * n) = pk;
    }
  });
}

template <int MT, int NT, int NS, int EPI>
__global__ __launch_bounds__(64 * kRgWaves, 1) void rows_gemm_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                     const bf16_t* __restrict__ bias, const bf16_t* __restrict__ R,
                                                                     long ldr, bf16_t* __restrict__ Y, int M, int N, int K, long ldx,
                                                                     long ldy, int spread) {
  rows_tile<MT, NT, NS, EPI>(X, W, bias, R, ldr, Y, M, N, K, ldx, ldy, blockIdx.z, spread);
}

// two plain products of the same sizes, the second in the upper half of the grid's z
template <int MT, int NT, int NS>
__global__ __launch_bounds__(64 * kRgWaves, 1) void rows_pair_kernel(const bf16_t* __restrict__ X1, long ldx1, const bf16_t* __restrict__ W1,
                                                                     bf16_t* __restrict__ Y1, const bf16_t* __restrict__ X2, long ldx2,
                                                                     const bf16_t* __restrict__ W2, bf16_t* __restrict__ Y2, int M, int N,
                                                                     int K, int spread) {
  const int half = gridDim.z >> 1, z = blockIdx.z;
  const bool up = z >= half;
  rows_tile<MT, NT, NS, RG_NONE>(up ? X2 : X1, up ? W2 : W1, nullptr, nullptr, 0, up ? Y2 : Y1, M, N, K, up ? ldx2 : ldx1, N, up ? z - half : z,
                                 spread);
}

// The f32 parts of two products with outputs of one shape, K split over workgroups (grid as above, parts for row tiles): part z of
// P [s1 + s2, M, N] is a range of K of the first product (z < s1) or the second.  One row tile.  What bounds a few-row product is the
// bytes that each CU takes in, X's and W's rows of its tile: where N is narrow a whole-K tile for every CU is 16 or 32 columns, and X is most
// of what comes.  Tiles of 64 columns over a part of K take half.  64 rows to 2,048 columns, K 4,096 (2,048) beside 5,632:
// apart 9.5 us each on average -> 11.7 us for both, and the norm that adds the parts takes the 4.8 us it took before.
template <int MT, int NT, int NS>
__global__ __launch_bounds__(64 * kRgWaves, 1) void rows_sums_kernel(const bf16_t* __restrict__ X1, long ldx1, const bf16_t* __restrict__ W1,
                                                                     int K1, const bf16_t* __restrict__ X2, long ldx2,
                                                                     const bf16_t* __restrict__ W2, int K2, float* __restrict__ P, int M,
                                                                     int N, int s1, int spread) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  asm volatile("" ::"s"(X1), "s"(W1), "s"(X2), "s"(W2), "s"(P), "s"(ldx1), "s"(ldx2));   // (as in rows_tile)
  int column, z;
  if (!rg_place(blockIdx.z, spread, N / (16 * NT), gridDim.y, column, z)) return;
  const int n0 = column * (16 * NT);
  const bool second = z >= s1;
  const bf16_t *const X = second ? X2 : X1, *const W = second ? W2 : W1;
  const long ldx = second ? ldx2 : ldx1;
  const int K = second ? K2 : K1, all = K / 64, waves = (second ? (int)gridDim.y - s1 : s1) * kRgWaves;
  const int q = (second ? z - s1 : z) * kRgWaves + wave, first = q * all / waves, nst = (q + 1) * all / waves - first;
  const int lrow = lane >> 3;
  const long k = (long)first * 64 + rg_lane_col(lane);
  const bf16_t* xs[2 * MT];
  const bf16_t* ws[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) xs[i] = X + (long)min(8 * i + lrow, M - 1) * ldx + k;  // rows past M repeat the last one
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) ws[i] = W + (long)(n0 + 8 * i + lrow) * K + k;
  floatx4 acc[MT][NT];
  rg_walk<MT, NT, NS>(xs, ws, nst, smem + wave * NS * rg_stage(MT, NT), acc);
  rg_sums<MT, NT>(smem, acc, [&](int m, const floatx4 (&t)[NT]) {
    const int row = m * 16 + (lane & 15);
    if (row >= M) return;
#pragma unroll
    for (int n = 0; n < NT; ++n) *reinterpret_cast<floatx4*>(P + ((long)z * M + row) * N + n0 + 16 * n + 4 * (lane >> 4)) = t[n];
  });
}

int device_cus() {
  static const int n = [] {
    int dev = 0, v = 0;
    return hipGetDevice(&dev) == hipSuccess && hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0 ? v : 256;
  }();
  return n;
}

// rounds of workgroups, one per CU, where the fullest of the 8 XCDs has `most` of them
int rounds_of(long most) { return (int)((most * 8 + device_cus() - 1) / device_cus()); }

// z from which a launch's last columns (of n products with `per` workgroups a column tile) go around over the XCDs: only where some XCDs would
// have a round more than the others (36 column tiles of 7 row tiles are 35 workgroups on four XCDs of 32 CUs and 28 on four: 400 x 576 x 1152
// 8.4 -> 6.1 us); elsewhere the placement's division is 0.3 us for nothing.
int rows_spread(int cols, int per, int n = 1) {
  const long eights = (cols + 7) / 8, even = (cols / 8 * per + (cols % 8 * per + 7) / 8);
  return rounds_of(eights * per * n) > rounds_of(even * n) ? cols / 8 : 1 << 30;
}

constexpr int ring_stages(int MT, int NT) { return 20 / (MT + NT) > 5 ? 5 : 20 / (MT + NT); }   // as many as 160 KB hold

template <int MT, int NT, int EPI>
int launch(const void* x, const void* w, const void* b, const void* r, long ldr, void* y, int M, int N, int K, long ldx, long ldy, hipStream_t st) {
  constexpr int NS = ring_stages(MT, NT), lds = rg_lds(MT, NT, NS);
  LK_SET_MAX_LDS((rows_gemm_kernel<MT, NT, NS, EPI>), lds);
  const int cols = N / (16 * NT), tiles = (M + 16 * MT - 1) / (16 * MT);
  rows_gemm_kernel<MT, NT, NS, EPI><<<dim3(8, tiles, (cols + 7) / 8), 64 * kRgWaves, lds, st>>>(
      (const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)b, (const bf16_t*)r, ldr, (bf16_t*)y, M, N, K, ldx, ldy, rows_spread(cols, tiles));
  LK_CHECK_LAUNCH();
  return 0;
}

// Row tiles per workgroup: a workgroup's time is its bytes, 16 (MT + NT) rows of K at 58 KB/us, and 1 us more for each one that its CU has had
// before (its first loads and its sums; the rings leave one workgroup per CU).  Where column tiles leave CUs free, fewer rows per workgroup
// read the same weight rows out of L2 again and end sooner.
int row_tiles(int M, int cols, int nt, int K) {
  const int m16 = (M + 15) / 16;
  int best = 4;
  double cost = 1e30;
  for (int mt = m16 < 4 ? m16 : 4; mt >= 1; --mt) {
    const double c = rounds_of(((long)((m16 + mt - 1) / mt) * cols + 7) / 8) * ((mt + nt) * (K / 32) / 58.0 + 1.0);
    if (c < cost) {
      cost = c;
      best = mt;
    }
  }
  return best;
}

template <int NT, int EPI>
int by_rows(const void* x, const void* w, const void* b, const void* r, long ldr, void* y, int M, int N, int K, long ldx, long ldy, hipStream_t st) {
  switch (row_tiles(M, N / (16 * NT), NT, K)) {
    case 1: return launch<1, NT, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
    case 2: return launch<2, NT, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
    case 3: return launch<3, NT, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
    default: return launch<4, NT, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
  }
}

// wide: 0: 16 columns per workgroup (SwiGLU: 16 gate and 16 up), 1: 32 (SwiGLU: as 0), 2: 64 (SwiGLU: 32 and 32), where N divides
template <int EPI>
int by_cols(const void* x, const void* w, const void* b, const void* r, long ldr, void* y, int M, int N, int K, long ldx, long ldy, int wide,
            hipStream_t st) {
  if (wide == 2 && N % 64 == 0) return by_rows<4, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
  if constexpr (EPI == RG_SWIGLU) {
    return by_rows<2, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
  } else {
    if (wide && N % 32 == 0) return by_rows<2, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
    return by_rows<1, EPI>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, st);
  }
}

template <int MT, int NT>
int launch_pair(const void* x1, long ldx1, const void* w1, void* y1, const void* x2, long ldx2, const void* w2, void* y2, int M, int N, int K,
                hipStream_t st) {
  constexpr int NS = ring_stages(MT, NT), lds = rg_lds(MT, NT, NS);
  LK_SET_MAX_LDS((rows_pair_kernel<MT, NT, NS>), lds);
  const int cols = N / (16 * NT), tiles = (M + 16 * MT - 1) / (16 * MT);
  rows_pair_kernel<MT, NT, NS><<<dim3(8, tiles, (cols + 7) / 8 * 2), 64 * kRgWaves, lds, st>>>(
      (const bf16_t*)x1, ldx1, (const bf16_t*)w1, (bf16_t*)y1, (const bf16_t*)x2, ldx2, (const bf16_t*)w2, (bf16_t*)y2, M, N, K, rows_spread(cols, tiles, 2));
  LK_CHECK_LAUNCH();
  return 0;
}

template <int NT>
int pair_by_rows(const void* x1, long ldx1, const void* w1, void* y1, const void* x2, long ldx2, const void* w2, void* y2, int M, int N, int K,
                 hipStream_t st) {
  switch (row_tiles(M, 2 * (N / (16 * NT)), NT, K)) {
    case 1: return launch_pair<1, NT>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
    case 2: return launch_pair<2, NT>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
    case 3: return launch_pair<3, NT>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
    default: return launch_pair<4, NT>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
  }
}

template <int MT>
int launch_sums(const void* x1, long ldx1, const void* w1, int K1, const void* x2, long ldx2, const void* w2, int K2, float* p, int M, int N,
                int s1, int parts, hipStream_t st) {
  constexpr int NT = 4, NS = ring_stages(MT, NT), lds = rg_lds(MT, NT, NS);
  LK_SET_MAX_LDS((rows_sums_kernel<MT, NT, NS>), lds);
  rows_sums_kernel<MT, NT, NS><<<dim3(8, parts, (N / 64 + 7) / 8), 64 * kRgWaves, lds, st>>>(
      (const bf16_t*)x1, ldx1, (const bf16_t*)w1, K1, (const bf16_t*)x2, ldx2, (const bf16_t*)w2, K2, p, M, N, s1, rows_spread(N / 64, parts));
  LK_CHECK_LAUNCH();
  return 0;
}

}  // namespace

// (the epilogue stores 8-byte groups of 4 columns: ldy is a multiple of 4, y 8-byte aligned)
bool lk_rows_gemm_supported(int M, int N, int K, int epi) {
  return M >= 1 && M <= 4096 && K >= 64 && K % 64 == 0 && N >= 16 && N % (epi == RG_SWIGLU ? 32 : 16) == 0;
}

int lk_rows_gemm(const void* x, const void* w, const void* b, const void* r, long ldr, void* y, int M, int N, int K, long ldx, long ldy, int epi,
                 int wide, hipStream_t st) {
  if (!lk_rows_gemm_supported(M, N, K, epi) || ldy % 4) return -1;
  switch (epi) {
    case RG_NONE: return by_cols<RG_NONE>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, wide, st);
    case RG_SWIGLU: return by_cols<RG_SWIGLU>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, wide, st);
    case RG_BIAS: return by_cols<RG_BIAS>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, wide, st);
    case RG_GELU: return by_cols<RG_GELU>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, wide, st);
    case RG_RELU: return by_cols<RG_RELU>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, wide, st);
    case RG_ADD: return by_cols<RG_ADD>(x, w, b, r, ldr, y, M, N, K, ldx, ldy, wide, st);
    default: return -1;
  }
}

// y1 = x1 w1^T and y2 = x2 w2^T of the same sizes in one launch (outputs contiguous).  A product of a few rows is mostly its launch and
// its first loads: 64 x 2048 x 2048 is 6.1 us in a decode step, two of them here 8.7 us, and a launch's gap less.
int lk_rows_pair(const void* x1, long ldx1, const void* w1, void* y1, const void* x2, long ldx2, const void* w2, void* y2, int M, int N, int K,
                 int wide, hipStream_t st) {
  if (!lk_rows_gemm_supported(M, N, K, RG_NONE)) return -1;
  if (wide == 2 && N % 64 == 0) return pair_by_rows<4>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
  if (wide && N % 32 == 0) return pair_by_rows<2>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
  return pair_by_rows<1>(x1, ldx1, w1, y1, x2, ldx2, w2, y2, M, N, K, st);
}

// Parts of x1 w1^T and x2 w2^T (as many as fill the chip's CUs once, split so that the longest K range is shortest): *s1 of the first.
// 0: not taken.  Beyond 64 rows a second row tile would read the weights again; with less than two stages a wave the ring has nothing in
// flight; outputs of less than 1,024 columns would be more than 16 parts to add up (fewer parts leave CUs without work).  Whether the
// launch is worth it where it is taken: ops.sums_pay.  Few rows gain the second launch: four steps of a state-space hybrid (above), 1 / 4 / 16 sequences, 1,579 / 1,807 / 2,178 us
// apart (weight-streaming kernels of up to 16 rows) -> 1,489 / 1,711 / 1,953.
int lk_rows_sums_parts(int M, int N, int K1, int K2, int* s1) {
  if (M < 1 || M > 64 || N < 64 || N > 8192 || N % 64 || K1 % 64 || K2 % 64 || K1 < 64 || K2 < 64) return 0;
  const int parts = device_cus() / (N / 64);
  if (parts < 2 || parts > kMaxSums || (K1 + K2) / 64 < 2 * parts * kRgWaves) return 0;   // (two stages a wave)
  int least = 1 << 30;
  for (int s = 1; s < parts; ++s) {
    const auto longest = [](int K, int n) { return (K / 64 + n * kRgWaves - 1) / (n * kRgWaves); };
    const int t = max(longest(K1, s), longest(K2, parts - s));
    if (t < least) least = t, *s1 = s;
  }
  return parts;
}

int lk_rows_sums(const void* x1, long ldx1, const void* w1, int K1, const void* x2, long ldx2, const void* w2, int K2, float* p, int M, int N,
                 hipStream_t st) {
  int s1 = 0;
  const int parts = lk_rows_sums_parts(M, N, K1, K2, &s1);
  if (!parts) return -1;
  switch ((M + 15) / 16) {
    case 1: return launch_sums<1>(x1, ldx1, w1, K1, x2, ldx2, w2, K2, p, M, N, s1, parts, st);
    case 2: return launch_sums<2>(x1, ldx1, w1, K1, x2, ldx2, w2, K2, p, M, N, s1, parts, st);
    case 3: return launch_sums<3>(x1, ldx1, w1, K1, x2, ldx2, w2, K2, p, M, N, s1, parts, st);
    default: return launch_sums<4>(x1, ldx1, w1, K1, x2, ldx2, w2, K2, p, M, N, s1, parts, st);
  }
}
