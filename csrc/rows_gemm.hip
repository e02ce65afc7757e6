// K2 / K3, few rows: Y[M,N] = act(X[M,K] . W[N,K]^T + bias) for up to some hundred rows in ONE launch, bf16 in,
// f32 sums, one rounding (bias / bias + GELU / bias + ReLU / SwiGLU in the epilogue).
//
// What bounds it: at these sizes neither HBM (a 2048 x 2048 weight is 1.4 us of it) nor the matrix cores
// but the serial chain of a launch: a tiled kernel with a barrier per K stage waits for each of them, and
// a split-K one pays a second launch for its sum.  Here no wave waits for another inside the K walk:
//   * a workgroup of 4 waves owns 16 output columns (wide: 32; SwiGLU: 16 gate and the 16 up columns) and up
//     to 64 rows; the waves split K, so each element of X and W reaches the workgroup once;
//   * every wave streams its own K range through a private LDS ring by LDS-DMA (row_ring.h; loads straight into
//     the fragment layout, 16 rows x 64 bytes, ran at a quarter of the rate: 12.0 us against 7.7 at
//     64 x 2048 x 2048, 8.4 against 5.7 at 32 rows);
//   * the waves' sums meet once in LDS, then the epilogue stores 4 columns per lane;
//   * 16 columns per workgroup give N / 16 workgroups, which is what fills 256 CUs at N 2048-4096; with more
//     rows or columns than that, 32 columns halve the re-reading of X out of L2 (256 x 2048 x 2048: 13.3 -> 8.8 us).
//     That re-reading bounds the large end, where the tiled kernels take over (ops: _rows_rule).
#include "common.h"
#include "kernels.h"
#include "row_ring.h"

namespace {

constexpr int kRgRows = 64;  // rows of a workgroup

enum { RG_NONE = 0, RG_SWIGLU = 1, RG_BIAS = 2, RG_GELU = 3, RG_RELU = 4 };

template <int MT, int NT, int NS, int EPI>
__global__ __launch_bounds__(64 * kRgWaves, 1) void rows_gemm_kernel(const bf16_t* __restrict__ X, const bf16_t* __restrict__ W,
                                                                     const bf16_t* __restrict__ bias, bf16_t* __restrict__ Y, int M,
                                                                     int N, int K, long ldx, long ldy) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int all = K / 64, first = wave * all / kRgWaves, nst = (wave + 1) * all / kRgWaves - first;  // stages of this wave
  const int n0 = blockIdx.x * (EPI == RG_SWIGLU ? 16 : 16 * NT), m0 = blockIdx.y * kRgRows;  // first output column and row
  X += (long)m0 * ldx;
  Y += (long)m0 * ldy;
  M = min(M - m0, kRgRows);
  const int lrow = lane >> 3;
  const long k = (long)first * 64 + rg_lane_col(lane);
  const bf16_t* xs[2 * MT];
  const bf16_t* ws[2 * NT];
#pragma unroll
  for (int i = 0; i < 2 * MT; ++i) xs[i] = X + (long)min(8 * i + lrow, M - 1) * ldx + k;  // rows past M repeat the last one
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) ws[i] = W + ((EPI == RG_SWIGLU ? (long)(i >> 1) * (N >> 1) : (i >> 1) * 16) + n0 + 8 * (i & 1) + lrow) * K + k;
  floatx4 acc[MT][NT];
  rg_walk<MT, NT, NS>(xs, ws, nst, smem + wave * NS * rg_stage(MT, NT), acc);
  rg_sums<MT, NT>(smem, acc, [&](int m, const floatx4 (&t)[NT]) {
    const int row = m * 16 + (lane & 15), col = n0 + 4 * (lane >> 4);
    if (row >= M) return;
#pragma unroll
    for (int n = 0; n < (EPI == RG_SWIGLU ? 1 : NT); ++n) {
      float y[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (EPI == RG_SWIGLU) {  // rounded as the projection and the activation apart round
          y[j] = bf2f(f2bf(lk_silu(bf2f(f2bf(t[0][j]))))) * bf2f(f2bf(t[NT - 1][j]));
        } else {
          y[j] = t[n][j];
          if constexpr (EPI >= RG_BIAS) y[j] += bf2f(bias[col + 16 * n + j]);
          if constexpr (EPI == RG_GELU) y[j] = lk_gelu_erf(y[j]);
          if constexpr (EPI == RG_RELU) y[j] = fmaxf(y[j], 0.f);
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
int launch(const void* x, const void* w, const void* b, void* y, int M, int N, int K, long ldx, long ldy, hipStream_t st) {
  constexpr int lds = rg_lds(MT, NT, NS);
  LK_SET_MAX_LDS((rows_gemm_kernel<MT, NT, NS, EPI>), lds);
  rows_gemm_kernel<MT, NT, NS, EPI><<<dim3(N / (16 * NT), (M + kRgRows - 1) / kRgRows), 64 * kRgWaves, lds, st>>>((const bf16_t*)x, (const bf16_t*)w, (const bf16_t*)b,
                                                                              (bf16_t*)y, M, N, K, ldx, ldy);
  LK_CHECK_LAUNCH();
  return 0;
}

template <int EPI>
int by_rows(const void* x, const void* w, const void* b, void* y, int M, int N, int K, long ldx, long ldy, int wide, hipStream_t st) {
  constexpr int NT = EPI == RG_SWIGLU ? 2 : 1;
  if constexpr (EPI != RG_SWIGLU) {
    if (wide && N % 32 == 0) {
      if (M <= 32) return launch<2, 2, 3, EPI>(x, w, b, y, M, N, K, ldx, ldy, st);
      return launch<4, 2, 3, EPI>(x, w, b, y, M, N, K, ldx, ldy, st);
    }
  }
  if (M <= 16) return launch<1, NT, NT == 1 ? 5 : 4, EPI>(x, w, b, y, M, N, K, ldx, ldy, st);
  if (M <= 32) return launch<2, NT, 4, EPI>(x, w, b, y, M, N, K, ldx, ldy, st);
  if (M <= 48) return launch<3, NT, 4, EPI>(x, w, b, y, M, N, K, ldx, ldy, st);
  return launch<4, NT, NT == 1 ? 4 : 3, EPI>(x, w, b, y, M, N, K, ldx, ldy, st);
}

}  // namespace

// (the epilogue stores 8-byte groups of 4 columns: ldy is a multiple of 4, y 8-byte aligned)
bool lk_rows_gemm_supported(int M, int N, int K, int epi) {
  return M >= 1 && M <= 4096 && K >= 64 && K % 64 == 0 && N >= 16 && N % (epi == RG_SWIGLU ? 32 : 16) == 0;
}

int lk_rows_gemm(const void* x, const void* w, const void* b, void* y, int M, int N, int K, long ldx, long ldy, int epi, int wide,
                 hipStream_t st) {
  if (!lk_rows_gemm_supported(M, N, K, epi) || ldy % 4) return -1;
  switch (epi) {
    case RG_NONE: return by_rows<RG_NONE>(x, w, b, y, M, N, K, ldx, ldy, wide, st);
    case RG_SWIGLU: return by_rows<RG_SWIGLU>(x, w, b, y, M, N, K, ldx, ldy, wide, st);
    case RG_BIAS: return by_rows<RG_BIAS>(x, w, b, y, M, N, K, ldx, ldy, wide, st);
    case RG_GELU: return by_rows<RG_GELU>(x, w, b, y, M, N, K, ldx, ldy, wide, st);
    case RG_RELU: return by_rows<RG_RELU>(x, w, b, y, M, N, K, ldx, ldy, wide, st);
    default: return -1;
  }
}
