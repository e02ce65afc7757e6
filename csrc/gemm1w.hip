// K2, prefill regime, one wave per SIMD: Y[M, N] = epilogue(X[M, K] . W[N, K]^T).
//
// A workgroup of 4 waves, one per SIMD, owns a BM x 256 tile (BM = 256 / 192 / 128; grouped also 288 / 224), a wave (BM / 2) x 128 of it
// as MB x 8 v_mfma_f32_16x16x32_bf16 accumulators (MB = BM / 32), which fill the AGPRs at BM 256 (at 288 the ninth row block's are VGPRs).  K advances by 64 (whole 128-byte lines).
//
// What a K-tile costs at BM 256, in cycles of a CU: 128 MFMAs of 16 per SIMD = 2,048; 32 fragment reads of 1 KB per wave, 128 KB at
// 128 bytes = 1,024 of LDS; 64 KB of LDS-DMA writes = 512.  LDS is busy three quarters of the time, so its work has to be spread over the
// K-tile, and a load takes longer than a K-tile to arrive, so a piece of LDS must be refilled as soon as it has been read.  Hence:
//   * X is resident, W streams.  All X fragments of a K-tile (2 MB of them) sit in registers, those of the next in a second set.  A W
//     fragment serves MB MFMAs in a row and is read WA fragments ahead into a ring of 4; the order is n-major, both halves of K of a
//     column fragment together, so LDS gets one W read per MB MFMAs all along.
//   * A K-tile is two phases, each opened by one barrier that both hands over what has landed and frees what has been read:
//       phase A (W columns 0-63 of a wave's 128 are being read): X's stage is free, its fragments being in registers, and so is the
//         second half of W's stage of the K-tile before: refill W half 2 of t + 1, then X of t + 2;
//       phase B (W columns 64-127): W half 1 of t is free: refill it with t + 2; X fragments of t + 1 are read.
//     Every refill is requested between 1 and 1.5 K-tiles before the barrier that needs it, and the same NP newer requests are in flight
//     at both barriers (s_waitcnt vmcnt(NP)), without draining.
//   * The reads are plain loads, so the compiler counts lgkmcnt per fragment; the order is pinned by scheduling fences.  The LDS-DMA is
//     inline asm (no register results) with M0 written one MFMA before.  The slots within a phase (Tile<BM>) are free parameters within
//     the asserted limits; they were swept (profiles/gemm1w_slots.md).
// One tile per workgroup: the hardware starts the next workgroup on a CU while the finished one's stores drain.  PERSIST, for short K
// where the load ramp is a third of a tile, and an even number of K-tiles (K-tile t lies in stage t & 1 of every tile): one workgroup per
// CU walks the tiles, and the last two K-tiles' refills are the next tile's first ones.
//
// Measured with cold weights: 4096 x 4096 x 4096 on 256-row tiles 91 us (1,500 TFLOP/s; MFMAs alone about 80, with the reads 86 - 89),
// M 2664 on 192-row tiles 69 us, 2664 x 6144 x 4096 on 128-row tiles 107 us; 62500 x 3072 x 768 persistent 257 us.
//
// Layout: two stages of (BM + 256) rows x 128 bytes (X rows | W rows), the 16-byte chunk c of a row at c ^ ((row >> 1) & 7), applied to
// the DMA's SOURCE: the LDS image is lane-linear and the fragment reads meet no bank twice.  The operands are swapped in the MFMA (A <- W
// rows, B <- X rows) and the W rows of every 32-row block permuted so that a lane ends with one output row and 8 consecutive columns per
// fragment pair: 16-byte stores; SwiGLU pairs gate (half 1) and up (half 2) of the same columns.
//
// Row tiles of 192 / 128 fill the 256 CUs where 256-row tiles leave most of a wave idle; the dispatch picks the row tile per M bucket
// from measurements (ops.tune_gemm) or a cost rule; the grouped form takes 128, 192, 224, 256 or 288 rows by the rounds that experts of the
// expected sizes fill (grouped_tile_rows in gemm.hip).  Epilogues (same contracts and rounding as gemm.hip): NONE, SWIGLU, BIAS, BIAS_GELU,
// BIAS_RELU, PARTIAL (split-K fp32 slabs), RESID (r += acc in place + per-row partial sums of squares), QKV (RoPE + paged-KV scatter);
// NONE / SWIGLU / QKV take the folded-RMSNorm row scale (LkEpi::ss_in); rows past M are dropped by the buffer descriptors' range checks.
#include <type_traits>
#include <utility>

#include "common.h"
#include "kernels.h"

namespace {

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));
typedef const __attribute__((address_space(3))) short8* lds_frag_t;
typedef const __attribute__((address_space(3))) unsigned short* lds_half_t;
typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));

constexpr int kBN = 256, kBK = 64;
constexpr int kRowB = kBK * 2;          // 128-B LDS rows
constexpr int kLdsEpi = 8192;           // epilogue scratch above the stages (row scales, RESID sums)

// GELU as a table: it takes a bf16 (the rounded sum with the bias) to a bf16, so the results for |x| in [2^-16, 16) are 2,560 pairs
// (x, -x), 10 KB of LDS, which every workgroup fills from lk_gelu_erf while its first tiles are on their way.  The arithmetic was 19
// instructions and an exponential per element, on SIMDs whose matrix units wait; the look-up is 8 and an LDS read.  The 32 results of a
// lane's row are computed where one of the wave's arguments lies outside.  The results are lk_gelu_erf's, to the bit.  Tiles of 128 rows compute
// them all: a short product waits for the table longer than it saves (949 x 3072 x 768 16.2 us for 14.5).  65,455 x 3072 x 768: 318 -> 288
// us (272 without the activation), 2,048 x 8192 x 2048: 58.7 -> 57.0.  So the time depends on the arguments: with some outside in almost every row
// (a standard deviation of 1e-3 or of 6) 312 -> 365 us, all zeros 287 -> 326, one column of zeros 292; with a standard deviation of 4, 298.
constexpr unsigned kGeluFirst = 111u << 7, kGeluPairs = 20 * 128;   // the bf16 bits of 2^-16; entries
constexpr int kLdsGelu = kGeluPairs * 4;

// A K-tile is NM MFMA slots of a wave; slot i multiplies X fragment m = i % MB with W fragment f = i / MB = 2 n + kk.  Barrier S1 opens
// phase B, S0 phase A of the next K-tile, both 8 MB slots apart and WA fragments ahead of the MFMAs that use what they hand over.
template <int BM>
struct Tile {
  static constexpr int MB = BM / 32, NM = 16 * MB, PX = BM / 32, NP = PX + 8;  // PX / 8: LDS-DMA pieces (1 KB) of X / W per wave
  static constexpr int kOpX = BM * kRowB;                // X rows of one stage
  static constexpr int kStage = kOpX + 256 * kRowB;      // X rows then W rows
  static constexpr int kLdsStages = 2 * kStage;          // 128 / 112 / 96 KB (136 at 288 rows)
  static constexpr int WA = 3;                           // W fragments read ahead
  static constexpr int S1 = (8 - WA) * MB, S0 = (16 - WA) * MB, PH = 8 * MB;
  // slots within a phase: phase A's 4 W pieces, then its PX X pieces; phase B's 4 W pieces and its 2 MB X reads.  (first, step); chosen
  // so that few of them fall on the slots of the W reads (multiples of MB): one wave issues everything, and a slot is four issues long
  static constexpr int AW0 = 1, AWS = BM == 128 ? 2 : BM == 192 ? 3 : 4, AX0 = WA * MB + 1, AXS = 5;
  static constexpr int BW0 = BM == 192 ? 4 : 2, BWS = MB, XR0 = BM == 192 ? 2 : 1, XRS = BM == 192 ? 3 : 2;
  static_assert(WA >= 1 && WA <= 3, "ring of 4");
  static_assert(AW0 >= 1 && AW0 + 3 * AWS < WA * MB && AX0 > WA * MB && AX0 + AXS * (PX - 1) < PH, "phase A");
  static_assert(BW0 >= 1 && BW0 + 3 * BWS < PH && XR0 + XRS * (2 * MB - 1) < PH, "phase B");
};

enum { E_NONE = 0, E_SWIGLU = 1, E_BIAS = 2, E_BIAS_GELU = 3, E_BIAS_RELU = 4, E_PARTIAL = 5, E_RESID = 6,
       E_QKV = 7 };
constexpr bool scalable(int e) { return e == E_NONE || e == E_SWIGLU || e == E_QKV; }

template <class Fn, int... I>
LK_DEVICE void unroll_impl(Fn&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class Fn>
LK_DEVICE void unroll(Fn&& f) {
  unroll_impl(f, std::make_integer_sequence<int, N>{});
}

template <int N>
LK_DEVICE void wait_vm() {  // s_waitcnt vmcnt(N), lgkmcnt / expcnt untouched
  static_assert(N >= 0 && N < 64, "vmcnt");
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
LK_DEVICE void lgkm0() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
LK_DEVICE void barrier_raw() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}
LK_DEVICE void fence() { __builtin_amdgcn_sched_barrier(0); }
LK_DEVICE int swz(int row) { return (row >> 1) & 7; }
LK_DEVICE float rbf(float x) { return bf2f(f2bf(x)); }
LK_DEVICE unsigned rfl(unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); }

// acc (+)= W-frag (16 x 32) . X-frag (32 x 16), acc pinned to AGPRs; volatile keeps issue order
LK_DEVICE void mfma(floatx4& acc, const short8& a, const short8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
LK_DEVICE void mfma0(floatx4& acc, const short8& a, const short8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=a"(acc) : "v"(a), "v"(b));
}
// the same with the accumulator in ordinary registers: the ninth 16-row block of a 288-row tile, for which the 256 AGPRs are taken
LK_DEVICE void mfma_v(floatx4& acc, const short8& a, const short8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+v"(acc) : "v"(a), "v"(b));
}
LK_DEVICE void mfma0_v(floatx4& acc, const short8& a, const short8& b) {
  asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, 0" : "=&v"(acc) : "v"(a), "v"(b));
}
template <int OFF>
LK_DEVICE void set_m0(unsigned base) { asm volatile("s_add_u32 m0, %0, %1" ::"s"(base), "i"(OFF) : "memory", "m0", "scc"); }
LK_DEVICE u32x4_t srd(const void* p, long bytes) {  // buffer descriptor words, wave-uniform
  const unsigned long a = reinterpret_cast<unsigned long>(p);
  return u32x4_t{rfl((unsigned)a), rfl((unsigned)(a >> 32)), (unsigned)min(bytes, 0x7FFFFFF0L), 0x00020000u};
}

// the number of the event at slot u of a phase (n of them from slot `first` on, `step` apart), or -1
constexpr int every(int u, int first, int step, int n) { return u >= first && (u - first) % step == 0 && (u - first) / step < n ? (u - first) / step : -1; }

// vector-memory operations per lane of the plain / bias epilogues (bias loads, then stores): the
// persistent walk's counted wait for the next tile's first K-tile skips them
constexpr bool gelu_table(int epi, int bm) { return epi == E_BIAS_GELU && bm > 128; }
template <int EPI, int BM>
constexpr int epi_lds() { return gelu_table(EPI, BM) ? kLdsGelu : kLdsEpi; }  // (the table lies in front of the stages, the scratch behind)
template <int EPI, int MB>
constexpr int epi_vm_ops() { return (EPI == E_NONE ? 0 : 4) + 4 * MB; }
constexpr bool persistable(int e) { return e == E_NONE || e == E_BIAS || e == E_BIAS_GELU || e == E_BIAS_RELU; }

// SCP: partial-sum planes of the folded-RMSNorm row scale loaded per row (0: no row scale; 16 covers
// a 4096-wide producer, 32 an 8192-wide one).  PERSIST: one workgroup per CU walks the tiles
// blockIdx.x, + gridDim.x, ...; the next tile's first refills are requested during the current
// tile's last two K-tiles, so its load ramp hides behind the current epilogue (short-K shapes: the
// encoder's K = 768 projections, 12 K-tiles per tile)
// GS (grouped form, lk_gemm1w_grouped): rows sorted by expert, sources gathered and results scattered through LkEpi
template <int EPI, int SCP, int BM, bool PERSIST = false, bool GS = false>
__global__ __launch_bounds__(256, 1) void gemm1w_kernel(const bf16_t* __restrict__ X, long ldx,
                                                        const bf16_t* __restrict__ W,
                                                        const bf16_t* __restrict__ bias, int M, int K, int I,
                                                        bf16_t* __restrict__ out, long ldo, int TM, int TN,
                                                        int tn0, int group_m, LkEpi ea) {
  constexpr bool SC = SCP > 0;
  static_assert(!SC || scalable(EPI), "row scale");
  static_assert(BM <= 256 || (!SC && EPI != E_RESID), "one thread per tile row");
  static_assert(!PERSIST || (persistable(EPI) && !SC), "persistent walk: plain / bias epilogues");
  using TL = Tile<BM>;
  constexpr int MB = TL::MB, NM = TL::NM, PX = TL::PX, NP = TL::NP, WM = BM / 2;
  constexpr int kOpX = TL::kOpX, kStage = TL::kStage, kLdsStages = TL::kLdsStages;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = w >> 1, wc = w & 1;
  const int r = lane & 15, g = lane >> 4;
  int tile = blockIdx.x;
  if constexpr (GS) {  // the expert of this tile, its rows and weights
    static_assert(!PERSIST && !SC && (EPI == E_NONE || EPI == E_SWIGLU), "grouped form");
    int e = -1, t0 = 0, r0 = 0, acc_t = 0;
    for (int i = 0; i < ea.experts; ++i) {
      const int a = ea.seg[i], m = ea.seg[i + 1] - a, nt = ((m + BM - 1) / BM) * TN;
      if (e < 0 && (int)blockIdx.x < acc_t + nt) {
        e = i;
        t0 = acc_t;
        r0 = a;
        M = m;
      }
      acc_t += nt;
    }
    if (e < 0) return;  // the whole workgroup: the grid is an upper bound
    tile -= t0;
    TM = (M + BM - 1) / BM;
    W += (long)e * (EPI == E_SWIGLU ? 2 * I : TN * kBN) * K;
    if (ea.gather) ea.gather += r0;
    else X += (long)r0 * ldx;
    if (ea.scatter) ea.scatter += r0;
    else out += (long)r0 * ldo;
  }
  const int nwg = TM * TN;
  const int nkt = K / kBK, kz = blockIdx.y, ks = gridDim.y;
  const int kt0 = kz * nkt / ks, nk = (kz + 1) * nkt / ks - kt0;  // >= 3 (host check)

  auto coords = [&](int tile, int& tm, int& tn) {
    const int L = xcd_remap(tile, nwg);
    const int per_group = group_m * TN;
    const int first = (L / per_group) * group_m;
    const int gm = min(TM - first, group_m);
    tm = first + (L % per_group) % gm;
    tn = tn0 + (L % per_group) / gm;  // (tn0: a column-split launch's first column tile)
  };
  u32x4_t xsrd = srd(X, (long)(GS && ea.gather ? ea.x_rows : M) * ldx * 2);
  u32x4_t wsrd = srd(W, (long)(EPI == E_SWIGLU ? 2 * I : (tn0 + TN) * kBN) * K * 2);
  constexpr int kTable = gelu_table(EPI, BM) ? kLdsGelu : 0;  // in front of the stages: a look-up's address is its index
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>((lds_ptr_t)smem)) + kTable;
  const int wrow = 128 * (w >> 1) + 32 * (w & 1);  // first W row of this wave's pieces of half 1; half 2: + 64
  const unsigned ldsx = rfl(lds0 + (BM / 4) * w * kRowB), ldsw = rfl(lds0 + kOpX + wrow * kRowB);

  // ---- LDS-DMA pieces of a K-tile, 8 rows each: X piece i covers rows BM/4 w + 8 i .., W piece 4 h + j rows wrow + 64 h + 8 j ..;
  // lane l brings the 16-byte chunk of slot l & 7 of row l >> 3.  Byte offsets of this lane's sources at column 0 (32-bit: the host
  // keeps every operand under 2^31 bytes).  A piece's rows are 8 apart, so
  // (row >> 1) & 7 = (lr8 >> 1) ^ 4 (piece & 1); LDS row 8 j + lr8 of a 32-row block of W holds column
  // 8 (lr8 >> 2) + (lr8 & 3) + 16 (j & 1) + 4 (j >> 1) of it.
  const int lr8 = lane >> 3, lc8 = lane & 7;
  unsigned xo[PX], wo[8];
  const unsigned ldxb = (unsigned)ldx * 2, kb = (unsigned)K * 2;
  const unsigned ch0 = (unsigned)((lc8 ^ (lr8 >> 1)) << 4);
  const unsigned chx = PX & w & 1 ? ch0 ^ 64u : ch0;  // (an odd number of pieces per wave: the odd waves' rows begin at an odd piece)
  auto offsets = [&](int tm, int tn, unsigned (&xo)[PX], unsigned (&wo)[8]) {
    const int xr = tm * BM + (BM / 4) * w + lr8;
#pragma unroll
    for (int i = 0; i < PX; ++i) {
      if constexpr (GS) {  // rows past the expert's end point behind the descriptor's range: zeros
        const int tr = xr + 8 * i;
        const int src = tr < M ? (ea.gather ? ea.gather[tr] / ea.top : tr) : -1;
        xo[i] = src >= 0 ? (unsigned)src * ldxb + (chx ^ (unsigned)((i & 1) << 6)) : 0xFFFFFF00u;
      } else {
        xo[i] = (unsigned)(xr + 8 * i) * ldxb + (chx ^ (unsigned)((i & 1) << 6));
      }
    }
    // SwiGLU: half 1 holds the gate rows of 64 output columns per column half, half 2 the up rows of the same
    const unsigned wl = (EPI == E_SWIGLU ? (unsigned)(tn * 128 + (w >> 1) * 64 + 32 * (w & 1)) : (unsigned)(tn * kBN + wrow)) +
                        (unsigned)(8 * (lr8 >> 2) + (lr8 & 3));
    const unsigned half = EPI == E_SWIGLU ? (unsigned)I : 64u;
#pragma unroll
    for (int i = 0; i < 8; ++i)
      wo[i] = (wl + (i >> 2) * half + (unsigned)(16 * (i & 1) + 4 * ((i >> 1) & 1))) * kb + (ch0 ^ (unsigned)((i & 1) << 6));
  };
  // M0 = LDS address of piece i of the K-tile in stage P (one scalar instruction)
  auto m0_x = [&](auto p_t, auto i_t) { set_m0<decltype(p_t)::value * kStage + 8 * decltype(i_t)::value * kRowB>(ldsx); };
  auto m0_w = [&](auto p_t, auto i_t) {
    constexpr int i = decltype(i_t)::value;
    set_m0<decltype(p_t)::value * kStage + (64 * (i >> 2) + 8 * (i & 3)) * kRowB>(ldsw);
  };
  // the piece at column offset so (M0 holds its LDS base)
  auto dma_x = [&](unsigned so, int i) { asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(xo[i]), "s"(xsrd), "s"(so) : "memory"); };
  auto dma_w = [&](unsigned so, int i) { asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" ::"v"(wo[i]), "s"(wsrd), "s"(so) : "memory"); };

  // ---- fragments: lane reads row (16-row base + r) of the stage, 16-byte chunk 4 kk + g
  const int rs = swz(r);
  unsigned bx[2][2], bw[2][2];  // [stage][kk], opaque so that the rest of every address stays the instruction's immediate
#pragma unroll
  for (int kk = 0; kk < 2; ++kk) {
    const unsigned b = lds0 + (((4 * kk + g) ^ rs) << 4) + r * kRowB;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
      bx[p][kk] = b + p * kStage + wr * WM * kRowB;
      bw[p][kk] = b + p * kStage + kOpX + wc * 128 * kRowB;
      asm volatile("" : "+v"(bx[p][kk]), "+v"(bw[p][kk]));
    }
  }
  short8 fx[2][2][MB], fw[4];  // X fragments [stage][kk][m], the ring of W fragments
  auto lds_rd = [](unsigned a, unsigned off) { return *reinterpret_cast<lds_frag_t>(a + off); };
  auto rd_x = [&](int p, int j) { fx[p][j / MB][j % MB] = lds_rd(bx[p][j / MB], (j % MB) * 16 * kRowB); };
  auto rd_w = [&](int p, int f) { fw[f & 3] = lds_rd(bw[p][f & 1], (f >> 1) * 16 * kRowB); };
  floatx4 acc[MB][8];
  using T = std::true_type;
  using F = std::false_type;

  // ---- folded RMSNorm, consumer side: thread tid sums the ss_nt partials of tile row tid.  Requested before everything else and
  // summed behind the K loop, where the compiler's wait for them drains nothing
  float* scl = reinterpret_cast<float*>(smem + kLdsStages);  // [256] row scales
  float ssp[SC ? SCP : 1];

  // K-tile t in stage P = t & 1; its refills are K-tile t + 2's, at column offset so2 of its operands.  FIRST: C = 0, and in a persistent
  // walk's later tiles (later) the epilogue's memory operations lie among the requests.
  auto ktile = [&](auto first_t, auto stage_t, unsigned so2, bool later) {
    constexpr bool FIRST = decltype(first_t)::value;
    constexpr int P = decltype(stage_t)::value, S1 = TL::S1, S0 = TL::S0, WA = TL::WA;
    auto landed = [&]() {  // everything but the newest NP refills
      if constexpr (FIRST && PERSIST) {
        if (later) wait_vm<NP + epi_vm_ops<EPI, MB>()>();
        else wait_vm<NP>();
      } else {
        wait_vm<NP>();
      }
    };
    unroll<NM>([&](auto i_t) {
      constexpr int i = decltype(i_t)::value, f = i / MB, m = i % MB;
      constexpr int ph = i < S1 ? 0 : i < S0 ? 1 : 2;                            // phase A, B, A of t + 1
      constexpr int u = ph == 0 ? i + WA * MB : ph == 1 ? i - S1 : i - S0;       // slot within the phase
      fence();
      if constexpr (i == S1 || i == S0) {
        // S1: W half 2 of t and X of t + 1 have landed, W half 1 of t has been read;
        // S0: W half 1 of t + 1 has landed, W half 2 of t and X of t + 1 have been read
        lgkm0();
        landed();
        barrier_raw();
      }
      if constexpr (m == 0) rd_w(f + WA < 16 ? P : P ^ 1, (f + WA) & 15);
      if constexpr (ph == 1 && every(u, TL::XR0, TL::XRS, 2 * MB) >= 0) rd_x(P ^ 1, every(u, TL::XR0, TL::XRS, 2 * MB));
      // the refill of this slot, then M0 for the next slot's
      constexpr int aw = ph == 2 ? every(u, TL::AW0, TL::AWS, 4) : -1, aw1 = ph == 2 ? every(u + 1, TL::AW0, TL::AWS, 4) : -1;
      constexpr int ax = ph == 0 ? every(u, TL::AX0, TL::AXS, PX) : -1, ax1 = ph == 0 ? every(u + 1, TL::AX0, TL::AXS, PX) : -1;
      constexpr int bw_ = ph == 1 ? every(u, TL::BW0, TL::BWS, 4) : -1, bw1 = ph == 1 ? every(u + 1, TL::BW0, TL::BWS, 4) : -1;
      if constexpr (aw >= 0) dma_w(so2, 4 + aw);
      if constexpr (ax >= 0) dma_x(so2, ax);
      if constexpr (bw_ >= 0) dma_w(so2, bw_);
      if constexpr (aw1 >= 0) m0_w(stage_t, std::integral_constant<int, 4 + aw1>{});
      if constexpr (ax1 >= 0) m0_x(stage_t, std::integral_constant<int, ax1>{});
      if constexpr (bw1 >= 0) m0_w(stage_t, std::integral_constant<int, bw1>{});
      fence();
      if constexpr (FIRST && (f & 1) == 0) {
        if constexpr (m < 8) mfma0(acc[m][f >> 1], fw[f & 3], fx[P][f & 1][m]);
        else mfma0_v(acc[m][f >> 1], fw[f & 3], fx[P][f & 1][m]);
      } else {
        if constexpr (m < 8) mfma(acc[m][f >> 1], fw[f & 3], fx[P][f & 1][m]);
        else mfma_v(acc[m][f >> 1], fw[f & 3], fx[P][f & 1][m]);
      }
    });
  };

  int tm, tn;
  coords(tile, tm, tn);
  offsets(tm, tn, xo, wo);
  if constexpr (SC) {
    const auto ssr = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(ea.ss_in), 0, (int)min((long)ea.ss_nt * ea.ss_ld * 4, 0x7FFFFFF0L), 0x00020000);
#pragma unroll
    for (int p = 0; p < SCP; ++p)  // (planes >= ss_nt lie past the range: 0)
      ssp[p] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(ssr, (unsigned)(tm * BM + tid + p * ea.ss_ld) * 4, 0, 0));
  }
  // prologue: what the refills of the two K-tiles before would have brought, in their order: X 0, W 0 half 1, W 0 half 2, X 1, W 1 half 1
  const unsigned sof = rfl((unsigned)kt0 * kRowB);
  unroll<2 * PX + 12>([&](auto q_t) {
    constexpr int q = decltype(q_t)::value, t = q < PX + 8 ? 0 : 1;
    constexpr bool x = q < PX || (q >= PX + 8 && q < 2 * PX + 8);
    constexpr int i = q < PX ? q : q < PX + 8 ? q - PX : x ? q - PX - 8 : q - 2 * PX - 8;
    constexpr std::integral_constant<int, i> i_t{};
    constexpr std::integral_constant<int, t> t_t{};
    if constexpr (x) m0_x(t_t, i_t);
    else m0_w(t_t, i_t);
    asm volatile("s_nop 0");
    if constexpr (x) dma_x(sof + t * kRowB, i);
    else dma_w(sof + t * kRowB, i);
  });
  if constexpr (kTable > 0) {
    for (unsigned i = tid; i < kGeluPairs; i += 256) {
      const unsigned x = (kGeluFirst + i) << 16;
      reinterpret_cast<unsigned*>(smem)[i] = pack_bf2(lk_gelu_erf(__uint_as_float(x)), lk_gelu_erf(__uint_as_float(x | 0x80000000u)));
    }
  }
  wait_vm<NP>();
  barrier_raw();
  unroll<4>([&](auto j_t) {
    m0_w(std::integral_constant<int, 1>{}, std::integral_constant<int, 4 + decltype(j_t)::value>{});
    asm volatile("s_nop 0");
    dma_w(sof + kRowB, 4 + decltype(j_t)::value);
  });
  for (bool later = false;; later = true) {
    int nxt = 0, tm2 = 0, tn2 = 0;
    bool has_next = false;
    if constexpr (PERSIST) {
      nxt = tile + (int)gridDim.x;
      has_next = nxt < nwg;
      // the last tile of the walk requests its own first K-tiles again (never read)
      coords(has_next ? nxt : tile, tm2, tn2);
    }
    fence();
#pragma unroll
    for (int j = 0; j < 2 * MB; ++j) rd_x(0, j);
#pragma unroll
    for (int f = 0; f < TL::WA; ++f) rd_w(0, f);
    lgkm0();
    barrier_raw();  // X's stage 0 is free
    unsigned so2 = sof + 2 * kRowB;
    // before K-tile t: the refills of the last two K-tiles are the next tile's first ones, or zeros that nobody reads (a descriptor
    // without range), so that every K-tile is the same code
    auto refills = [&](int t) {
      if (t + 2 == nk) {
        if constexpr (PERSIST) {
          offsets(tm2, tn2, xo, wo);
          so2 = sof;
        } else {
          xsrd.z = wsrd.z = 0;
        }
      }
    };
    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    ktile(T{}, even, so2, later);
    for (int t = 1;; t += 2) {
      so2 += kRowB;
      refills(t);
      ktile(F{}, odd, so2, false);
      if (t + 1 >= nk) break;
      so2 += kRowB;
      refills(t + 1);
      ktile(F{}, even, so2, false);
      if (t + 2 >= nk) break;
    }
    // the asm MFMAs are invisible to hipcc's hazard recognizer: wait out MFMA -> accumulator read,
    // and pin every accumulator behind that wait (hipcc otherwise schedules some v_accvgpr_read of
    // the final K-tile's results right after their MFMA is issued, before it has written them)
    asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 3" ::: "memory");
#pragma unroll
    for (int m = 0; m < MB; ++m)
#pragma unroll
      for (int n = 0; n < 8; ++n) {
        if (m < 8) asm volatile("" : "+a"(acc[m][n]));
        else asm volatile("" : "+v"(acc[m][n]));
      }

    if constexpr (!PERSIST) wait_vm<0>();  // the last refills land before the workgroup's LDS is released

    // ================= epilogue of tile (tm, tn)
    // lane holds row tm*256 + wr*128 + 16m + r; fragment pair (2p, 2p+1) the 8 consecutive
    // columns 32p + 8g .. +7 of the wave's 128 (SwiGLU: gate pairs 0, 1 and up pairs 2, 3 of
    // each 64-row half ... the wave's 64 output columns)
    float scm[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) scm[m] = 1.f;
    if constexpr (SC) {
      float ssum = 0.f;
#pragma unroll
      for (int p = 0; p < SCP; ++p) ssum += ssp[p];
      scl[tid] = rsqrtf(ssum * ea.inv_h + ea.eps);
      lgkm0();
      barrier_raw();
#pragma unroll
      for (int m = 0; m < MB; ++m) scm[m] = scl[wr * WM + m * 16 + r];
    }
    // the first byte of an output row's columns at c (grouped: the scattered row, or behind the range)
    const long orows = GS && ea.scatter ? ea.out_rows : M;
    auto row_at = [&](int m, int c) -> unsigned {
      const long row = (long)tm * BM + wr * WM + m * 16 + r;
      if constexpr (GS) {
        if (row >= M) return 0xFFFFFE00u;
        return (unsigned)((ea.scatter ? ea.scatter[row] : row) * ldo + c) * 2;
      } else {
        return (unsigned)(row * ldo + c) * 2;
      }
    };
    auto pk8 = [](const float (&y)[8]) {
      return u32x4_t{pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]), pack_bf2(y[4], y[5]), pack_bf2(y[6], y[7])};
    };
    if constexpr (EPI == E_PARTIAL) {  // fp32 partial sums of split kz: out is float [splits, M, ldo]
      float* part = reinterpret_cast<float*>(out) + (long)kz * M * ldo;
      const auto ps = __builtin_amdgcn_make_buffer_rsrc(part, 0, (int)min((long)M * ldo * 4, 0x7FFFFFF0L), 0x00020000);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const unsigned rb = (unsigned)(((long)tm * BM + wr * WM + m * 16 + r) * ldo + tn * kBN + wc * 128) * 4;
#pragma unroll
        for (int n = 0; n < 8; ++n)
          __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4_t, acc[m][n]), ps,
                                                 rb + (unsigned)((32 * (n >> 1) + 8 * g + 4 * (n & 1)) * 4), 0, 0);
      }
    } else if constexpr (EPI == E_SWIGLU) {
      const auto os = __builtin_amdgcn_make_buffer_rsrc(out, 0, (int)min(orows * ldo * 2, 0x7FFFFFF0L), 0x00020000);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const unsigned rb = row_at(m, tn * 128 + wc * 64 + 8 * g);
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          float y[8];
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v)
              y[4 * h + v] = GS ? lk_silu(acc[m][2 * p + h][v]) * acc[m][4 + 2 * p + h][v]   // f32 up to the result
                                : rbf(lk_silu(rbf(acc[m][2 * p + h][v] * scm[m]))) * rbf(acc[m][4 + 2 * p + h][v] * scm[m]);
          __builtin_amdgcn_raw_buffer_store_b128(pk8(y), os, rb + 64 * p, 0, 0);
        }
      }
    } else if constexpr (EPI == E_RESID) {
      // r = bf16(r + bf16(acc)) in place, then the partial sum of squares of the new r over the
      // tile's 256 columns (lanes g, then the two wc waves through LDS) into ss_out[tn][row]
      const auto rrs = __builtin_amdgcn_make_buffer_rsrc(ea.resid, 0, (int)min((long)M * ea.ldr * 2, 0x7FFFFFF0L), 0x00020000);
      float ssm[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const long row = (long)tm * BM + wr * WM + m * 16 + r;
        const unsigned rb = (unsigned)((row * ea.ldr + (long)tn * kBN + wc * 128 + 8 * g) * 2);
        u32x4_t rv[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) rv[p] = __builtin_amdgcn_raw_buffer_load_b128(rrs, rb + 64 * p, 0, 0);
        float ss = 0.f;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const unsigned rw[4] = {rv[p].x, rv[p].y, rv[p].z, rv[p].w};
          float y[8];
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              const int j = 4 * h + v;
              const float res = bf2f((bf16_t)((rw[j >> 1] >> (16 * (j & 1))) & 0xFFFF));
              y[j] = rbf(rbf(acc[m][2 * p + h][v]) + res);
              ss += y[j] * y[j];
            }
          __builtin_amdgcn_raw_buffer_store_b128(pk8(y), rrs, rb + 64 * p, 0, 0);
        }
        ss += __shfl_xor(ss, 16, 64);
        ss += __shfl_xor(ss, 32, 64);
        ssm[m] = ss;
      }
      float* red = reinterpret_cast<float*>(smem + kLdsStages + 1024);  // [2 wc][BM tile rows]
      if (g == 0) {
#pragma unroll
        for (int m = 0; m < MB; ++m) red[wc * BM + wr * WM + m * 16 + r] = ssm[m];
      }
      lgkm0();
      barrier_raw();
      const int row = tm * BM + tid;
      if (tid < BM && row < M) ea.ss_out[(long)tn * ea.ss_out_ld + row] = red[tid] + red[BM + tid];
    } else if constexpr (EPI == E_QKV) {
      // RoPE (interleaved pairs) on the q / k heads + the paged-KV scatter, on the bf16-rounded
      // (row-scaled) projection: the values "GEMM -> rope_kv_" would leave.  Everything that
      // depends only on the lane's columns is hoisted out of the row loop (no integer division
      // per row), the rows' positions / slots are loaded in one round before any store (a u32
      // store may alias the int metadata, so per-row loads would each wait behind the previous
      // row's stores), and the next row's cos / sin are in flight while this row is rotated.
      const int qcols = ea.hq * ea.hd, kcols = ea.hkv * ea.hd, half = ea.hd >> 1;
      const int cb = tn * kBN + wc * 128;
      int i0[4], coff[4];
      bool rot[4], kv[4], isv[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        const int c = cb + 32 * p + 8 * g;
        rot[p] = c < qcols + kcols;
        kv[p] = c >= qcols;
        isv[p] = c >= qcols + kcols;
        i0[p] = (c % ea.hd) >> 1;  // first rotation pair
        const int cc = c - qcols - (isv[p] ? kcols : 0);
        const int h = cc / ea.hd;
        coff[p] = h * ea.bs * ea.hd + (cc - h * ea.hd);  // head h, dim d within a cache block
      }
      const long blk_stride = (long)ea.hkv * ea.bs * ea.hd;
      int posv[MB], slotv[MB];
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const int row = tm * BM + wr * WM + m * 16 + r;
        const int rc = min(row, M - 1);  // unconditional loads: no branch per row around them
        posv[m] = ea.pos[rc];
        slotv[m] = ea.slots ? ea.slots[rc] : -1;
      }
      floatx4 c4[4], s4[4];
      auto load_cs = [&](int pos, floatx4 (&cv)[4], floatx4 (&sv)[4]) {
        const float* cs = ea.cos_sin + (long)pos * ea.hd;
#pragma unroll
        for (int p = 0; p < 4; ++p) {  // (loaded for v columns too: in range, and branch-free)
          cv[p] = *reinterpret_cast<const floatx4*>(cs + i0[p]);
          sv[p] = *reinterpret_cast<const floatx4*>(cs + half + i0[p]);
        }
      };
      load_cs(posv[0], c4, s4);
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        floatx4 c4n[4], s4n[4];
        if (m + 1 < MB) load_cs(posv[m + 1], c4n, s4n);
        const int row = tm * BM + wr * WM + m * 16 + r;
        if (row < M) {
          const float sc = scm[m];
          const int slot = slotv[m];
          const long kvb = slot >= 0 ? (long)(slot / ea.bs) * blk_stride + (long)(slot % ea.bs) * ea.hd : 0;
          bf16_t* orow = out + (long)row * ldo;
#pragma unroll
          for (int p = 0; p < 4; ++p) {
            float y[8];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int v = 0; v < 4; ++v) y[4 * h + v] = rbf(acc[m][2 * p + h][v] * sc);
            if (rot[p]) {
#pragma unroll
              for (int q = 0; q < 4; ++q) {
                const float a = y[2 * q], b = y[2 * q + 1];
                y[2 * q] = rot_lo(a, b, c4[p][q], s4[p][q]);
                y[2 * q + 1] = rot_hi(a, b, c4[p][q], s4[p][q]);
              }
            }
            const u32x4_t pk = pk8(y);
            *reinterpret_cast<u32x4_t*>(orow + cb + 32 * p + 8 * g) = pk;
            if (kv[p] && slot >= 0 && ea.kc != nullptr)
              *reinterpret_cast<u32x4_t*>((isv[p] ? ea.vc : ea.kc) + kvb + coff[p]) = pk;
          }
        }
        // one row of cos / sin in flight, not all MB (hoisted, they would take MB x 32 VGPRs)
        asm volatile("" ::: "memory");
        if (m + 1 < MB) {
#pragma unroll
          for (int p = 0; p < 4; ++p) c4[p] = c4n[p], s4[p] = s4n[p];
        }
      }
    } else {  // NONE / BIAS / BIAS_GELU / BIAS_RELU
      const auto os = __builtin_amdgcn_make_buffer_rsrc(out, 0, (int)min(orows * ldo * 2, 0x7FFFFFF0L), 0x00020000);
      float bv[8][4];
#pragma unroll
      for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int v = 0; v < 4; ++v) bv[n][v] = 0.f;
      if constexpr (EPI != E_NONE) {
        const auto bs = __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16_t*>(bias), 0, (tn0 + TN) * kBN * 2, 0x00020000);
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          const u32x4_t b = __builtin_amdgcn_raw_buffer_load_b128(bs, (unsigned)((tn * kBN + wc * 128 + 32 * p + 8 * g) * 2), 0, 0);
          const unsigned bw4[4] = {b.x, b.y, b.z, b.w};
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            bv[2 * p + (q >> 1)][2 * (q & 1)] = bf2f((bf16_t)(bw4[q] & 0xFFFF));
            bv[2 * p + (q >> 1)][2 * (q & 1) + 1] = bf2f((bf16_t)(bw4[q] >> 16));
          }
        }
      }
      const unsigned table = lds0 - kTable;
      auto look = [&](unsigned i) -> unsigned { return *reinterpret_cast<lds_half_t>(table + 2 * i); };
      auto act = [&](float e, float b) {  // (GELU: below)
        if constexpr (EPI == E_BIAS || EPI == E_BIAS_RELU) e = rbf(e + b);
        if constexpr (EPI == E_BIAS_GELU) e += b;
        if constexpr (EPI == E_BIAS_RELU) e = fmaxf(e, 0.f);
        return e;
      };
#pragma unroll
      for (int m = 0; m < MB; ++m) {
        const unsigned rb = row_at(m, tn * kBN + wc * 128 + 8 * g);
        u32x4_t pk[4];
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          float y[8];
#pragma unroll
          for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int v = 0; v < 4; ++v) y[4 * h + v] = act(acc[m][2 * p + h][v] * scm[m], bv[2 * p + h][v]);
          pk[p] = pk8(y);
        }
        if constexpr (EPI == E_BIAS_GELU && kTable == 0) {
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const unsigned w = pk[j >> 2][j & 3];
            pk[j >> 2][j & 3] = pack_bf2(lk_gelu_erf(__uint_as_float(w << 16)), lk_gelu_erf(__uint_as_float(w & 0xffff0000u)));
          }
        }
        if constexpr (kTable > 0) {
          // a table index is the magnitude's bits, then the sign (every half word rotated left by one), from the first entry's on
          ushort2_t at[16], far = {0, 0};
#pragma unroll
          for (int j = 0; j < 16; ++j) {
            const ushort2_t e = __builtin_bit_cast(ushort2_t, (unsigned)pk[j >> 2][j & 3]);
            at[j] = (ushort2_t)((e << 1) | (e >> 15)) - (unsigned short)(2 * kGeluFirst);
            far = __builtin_elementwise_max(far, at[j]);
          }
          if (__any(max(far.x, far.y) >= 2 * kGeluPairs)) {
            u32x4_t q = pk[0];
#pragma unroll 1
            for (int p = 0; p < 4; ++p) {  // (the four groups go round: one copy of the arithmetic)
#pragma unroll
              for (int j = 0; j < 4; ++j)
                q[j] = pack_bf2(lk_gelu_erf(__uint_as_float(q[j] << 16)), lk_gelu_erf(__uint_as_float(q[j] & 0xffff0000u)));
              pk[0] = pk[1];
              pk[1] = pk[2];
              pk[2] = pk[3];
              pk[3] = q;
              q = pk[0];
            }
          } else {
#pragma unroll
            for (int j = 0; j < 16; ++j) pk[j >> 2][j & 3] = look(at[j].x) | look(at[j].y) << 16;
          }
        }
#pragma unroll
        for (int p = 0; p < 4; ++p) __builtin_amdgcn_raw_buffer_store_b128(pk[p], os, rb + 64 * p, 0, 0);
      }
    }
    if constexpr (!PERSIST) {
      break;
    } else {
      if (!has_next) {
        wait_vm<0>();  // the walk's last (unread) DMAs land before the workgroup's LDS is released
        break;
      }
      tile = nxt;
      tm = tm2;
      tn = tn2;
    }
  }
}

// split-K reduction: out[r, c..c+3] = epi(sum_z part[z, r, c..c+3] (+ bias)), rounded like the
// fused epilogues; one thread per 4 columns.  All ranges' loads are in flight at once (kS of them, the
// count a constant): in a loop over a count from the host each waited for the one before it.  0.3 - 0.7 us
// of a split product, 0.7 - 1.2 us with the residual, whose sum also was one workgroup to a row and 256 columns.
template <int kS>
__device__ __forceinline__ floatx4 sum_parts(const float* p, long MN) {
  floatx4 t[kS];
#pragma unroll
  for (int z = 0; z < kS; ++z) t[z] = *reinterpret_cast<const floatx4*>(p + z * MN);
#pragma unroll
  for (int z = 1; z < kS; ++z) t[0] += t[z];
  return t[0];
}

template <int EPI, int kS>
__global__ __launch_bounds__(256) void reduce1w_kernel(const float* __restrict__ part, int M, int N,
                                                       const bf16_t* __restrict__ bias, bf16_t* __restrict__ out,
                                                       long ldo) {
  const unsigned i = blockIdx.x * 256u + threadIdx.x, nq = N / 4;  // (M * N * 4 bytes are below 2^31)
  if (i >= M * nq) return;
  const unsigned row = i / nq, col = i % nq * 4;
  const floatx4 a = sum_parts<kS>(part + (long)i * 4, (long)M * N);
  float y[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    float e = a[v];
    if constexpr (EPI != E_NONE) e = rbf(e + bf2f(bias[col + v]));
    if constexpr (EPI == E_BIAS_GELU) e = lk_gelu_erf(e);
    if constexpr (EPI == E_BIAS_RELU) e = fmaxf(e, 0.f);
    y[v] = e;
  }
  *reinterpret_cast<uint2*>(out + (long)row * ldo + col) = make_uint2(pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]));
}

// split-K reduction for RESID (same planes as the unsplit epilogue: partial sums per 256 columns), one wave per row and
// plane, four rows to a workgroup
template <int kS>
__global__ __launch_bounds__(256) void reduce1w_resid_kernel(const float* __restrict__ part, int M, int N, LkEpi ea) {
  const int tn = blockIdx.x, row = blockIdx.y * 4 + threadIdx.x / 64, lane = threadIdx.x % 64, col = tn * 256 + 4 * lane;
  if (row >= M) return;
  bf16_t* rp = ea.resid + (long)row * ea.ldr + col;
  const uint2 rv = *reinterpret_cast<const uint2*>(rp);
  const floatx4 a = sum_parts<kS>(part + (long)row * N + col, (long)M * N);
  const unsigned rw[2] = {rv.x, rv.y};
  float y[4], ss = 0.f;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    y[v] = rbf(rbf(a[v]) + bf2f((bf16_t)((rw[v >> 1] >> (16 * (v & 1))) & 0xFFFF)));
    ss += y[v] * y[v];
  }
  *reinterpret_cast<uint2*>(rp) = make_uint2(pack_bf2(y[0], y[1]), pack_bf2(y[2], y[3]));
  ss = wave_sum(ss);
  if (lane == 0) ea.ss_out[(long)tn * ea.ss_out_ld + row] = ss;
}

template <int kS>
int launch_reduce1w(const float* ws, int M, int N, int epi, const bf16_t* bias, bf16_t* out, long ldo, hipStream_t st, const LkEpi& ea) {
  const int blocks = (int)(((long)M * (N / 4) + 255) / 256);
  switch (epi) {
    case E_RESID: reduce1w_resid_kernel<kS><<<dim3(N / 256, (M + 3) / 4), 256, 0, st>>>(ws, M, N, ea); break;
    case E_NONE: reduce1w_kernel<E_NONE, kS><<<blocks, 256, 0, st>>>(ws, M, N, bias, out, ldo); break;
    case E_BIAS: reduce1w_kernel<E_BIAS, kS><<<blocks, 256, 0, st>>>(ws, M, N, bias, out, ldo); break;
    case E_BIAS_GELU: reduce1w_kernel<E_BIAS_GELU, kS><<<blocks, 256, 0, st>>>(ws, M, N, bias, out, ldo); break;
    case E_BIAS_RELU: reduce1w_kernel<E_BIAS_RELU, kS><<<blocks, 256, 0, st>>>(ws, M, N, bias, out, ldo); break;
    default: return -1;
  }
  return 0;
}

int group1w() {  // row tiles per XCD group of the tile order (LK_GEMM_GROUP_M, default 4)
  static const int g = [] {
    const char* e = getenv("LK_GEMM_GROUP_M");
    const int v = e ? atoi(e) : 4;
    return v >= 1 ? v : 4;
  }();
  return g;
}

int cu_count() {
  static const int n = [] {
    int dev = 0, v = 0;
    (void)hipGetDevice(&dev);
    return hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess && v > 0 ? v : 256;
  }();
  return n;
}

// persistent walk for short K (LK_GEMM1W_PERSIST_KT: the most K-tiles of 64 it is used for; 0: off)
int persist_kt() {
  static const int v = [] {
    const char* e = getenv("LK_GEMM1W_PERSIST_KT");
    return e ? atoi(e) : 16;
  }();
  return v;
}

template <int EPI, int SCP, int BM, bool PERSIST = false>
void launch1w_p(const bf16_t* x, long ldx, const bf16_t* w, const bf16_t* bias, int M, int K, int I, bf16_t* out,
                long ldo, int TN, int tn0, int ks, int group_m, hipStream_t st, const LkEpi& ea) {
  constexpr int lds = Tile<BM>::kLdsStages + epi_lds<EPI, BM>();
  LK_SET_MAX_LDS((gemm1w_kernel<EPI, SCP, BM, PERSIST>), lds);
  const int TM = (M + BM - 1) / BM;
  const int grid = PERSIST ? min(TM * TN, cu_count()) : TM * TN;
  gemm1w_kernel<EPI, SCP, BM, PERSIST><<<dim3(grid, ks), 256, lds, st>>>(x, ldx, w, bias, M, K, I, out, ldo, TM, TN,
                                                                       tn0, group_m > 0 ? group_m : group1w(), ea);
}
template <int EPI, int SCP, int BM>
void launch1w(const bf16_t* x, long ldx, const bf16_t* w, const bf16_t* bias, int M, int K, int I, bf16_t* out,
              long ldo, int TN, int tn0, int ks, int group_m, hipStream_t st, const LkEpi& ea) {
  if constexpr (persistable(EPI) && SCP == 0 && BM == 256) {
    const int tiles = ((M + BM - 1) / BM) * TN;
    if (ks == 1 && K / kBK <= persist_kt() && K / kBK % 2 == 0 && tiles > 2 * cu_count()) {
      launch1w_p<EPI, SCP, BM, true>(x, ldx, w, bias, M, K, I, out, ldo, TN, tn0, ks, group_m, st, ea);
      return;
    }
  }
  launch1w_p<EPI, SCP, BM, false>(x, ldx, w, bias, M, K, I, out, ldo, TN, tn0, ks, group_m, st, ea);
}
template <int EPI, int SCP>
void launch1w_bm(int bm, const bf16_t* x, long ldx, const bf16_t* w, const bf16_t* bias, int M, int K, int I,
                 bf16_t* out, long ldo, int TN, int tn0, int ks, int group_m, hipStream_t st, const LkEpi& ea) {
  if (bm == 192) launch1w<EPI, SCP, 192>(x, ldx, w, bias, M, K, I, out, ldo, TN, tn0, ks, group_m, st, ea);
  else if (bm == 128) launch1w<EPI, SCP, 128>(x, ldx, w, bias, M, K, I, out, ldo, TN, tn0, ks, group_m, st, ea);
  else launch1w<EPI, SCP, 256>(x, ldx, w, bias, M, K, I, out, ldo, TN, tn0, ks, group_m, st, ea);
}
template <int EPI, int SCP>
void launch1w_tiles(int bm, const bf16_t* x, long ldx, const bf16_t* w, const bf16_t* bias, int M, int K, int I,
                    bf16_t* out, long ldo, int TN, int ks, int group_m, hipStream_t st, const LkEpi& ea) {
  if (bm == LK_GEMM1W_SPLIT128 || bm == LK_GEMM1W_SPLIT192) {
    // column split: the column tiles that fill whole waves of the CUs with 256-row tiles, then
    // the rest -- less than one wave of 256-row tiles -- on smaller row tiles that fill one.
    // The QKV projection at M 4096 (16 x 24 tiles = 1.5 waves of 256 CUs) runs 16 x 16 256-row
    // tiles, then 32 x 8 128-row tiles: 1 + ~0.6 tile times instead of 2.
    const int ca = lk_gemm1w_split_cols(M, TN, cu_count());
    if (ca > 0 && ca < TN) {
      launch1w_bm<EPI, SCP>(256, x, ldx, w, bias, M, K, I, out, ldo, ca, 0, ks, group_m, st, ea);
      launch1w_bm<EPI, SCP>(bm == LK_GEMM1W_SPLIT128 ? 128 : 192, x, ldx, w, bias, M, K, I, out, ldo, TN - ca, ca, ks,
                            group_m, st, ea);
      return;
    }
    bm = 256;
  }
  launch1w_bm<EPI, SCP>(bm, x, ldx, w, bias, M, K, I, out, ldo, TN, 0, ks, group_m, st, ea);
}
template <int EPI>
void launch1w_sc(int bm, const bf16_t* x, long ldx, const bf16_t* w, const bf16_t* bias, int M, int K, int I,
                 bf16_t* out, long ldo, int TN, int ks, int group_m, hipStream_t st, const LkEpi& ea) {
  if constexpr (scalable(EPI)) {
    if (ea.ss_in != nullptr) {
      if (ea.ss_nt <= 16) launch1w_tiles<EPI, 16>(bm, x, ldx, w, bias, M, K, I, out, ldo, TN, ks, group_m, st, ea);
      else launch1w_tiles<EPI, 32>(bm, x, ldx, w, bias, M, K, I, out, ldo, TN, ks, group_m, st, ea);
      return;
    }
  }
  launch1w_tiles<EPI, 0>(bm, x, ldx, w, bias, M, K, I, out, ldo, TN, ks, group_m, st, ea);
}

template <int EPI, int BM>
int launch1w_grouped(const bf16_t* x, long ldx, const bf16_t* w, long rows, int K, int I, bf16_t* out, long ldo, int TN, hipStream_t st,
                     const LkEpi& ea) {
  constexpr int lds = Tile<BM>::kLdsStages + epi_lds<EPI, BM>();
  LK_SET_MAX_LDS((gemm1w_kernel<EPI, 0, BM, false, true>), lds);
  const long grid = ((rows + BM - 1) / BM + ea.experts) * TN;
  if (grid > 2147483647L) return -1;
  gemm1w_kernel<EPI, 0, BM, false, true><<<dim3((unsigned)grid, 1), 256, lds, st>>>(x, ldx, w, nullptr, 0, K, I, out, ldo, 0, TN, 0,
                                                                                    group1w(), ea);
  LK_CHECK_LAUNCH();
  return 0;
}

}  // namespace

int lk_gemm1w_grouped_supported(long rows, long ldx, long x_rows, int N, int K, int swiglu, long ldo) {
  if (K % kBK || K / kBK < 3 || (swiglu ? N % 2 || (N / 2) % 128 : N % kBN)) return 0;
  return (long)N * K * 2 < 0x7FFFFFF0L && max(rows, x_rows) * ldx * 2 < 0x7FFFFFF0L && rows * ldo * 2 < 0x7FFFFFF0L;
}

int lk_gemm1w_grouped(const bf16_t* x, long ldx, const bf16_t* w, const int* seg, int E, long rows, int N, int K, int swiglu, bf16_t* out,
                      long ldo, hipStream_t st, const int* gather, long x_rows, const int* scatter, int top, int bm) {
  if (!lk_gemm1w_grouped_supported(rows, ldx, gather ? x_rows : rows, N, K, swiglu, ldo)) return -1;
  LkEpi ea{};
  ea.seg = seg;
  ea.experts = E;
  ea.gather = gather;
  ea.top = top;
  ea.scatter = scatter;
  ea.x_rows = x_rows;
  ea.out_rows = rows;
#define LK_G1W(BM)                                                                                                  \
  case BM:                                                                                                          \
    return swiglu ? launch1w_grouped<E_SWIGLU, BM>(x, ldx, w, rows, K, N / 2, out, ldo, N / kBN, st, ea)            \
                  : launch1w_grouped<E_NONE, BM>(x, ldx, w, rows, K, 0, out, ldo, N / kBN, st, ea)
  switch (bm) {
    LK_G1W(128);
    LK_G1W(192);
    LK_G1W(224);
    LK_G1W(256);
    LK_G1W(288);
    default: return -1;
  }
#undef LK_G1W
}

int lk_gemm1w_split_cols(int M, int TN, int cus) {
  const int tm = (M + 255) / 256;
  const int waves = tm * TN / cus;  // whole waves of 256-row tiles
  return min(TN, waves * cus / tm);
}

int lk_gemm1w_supported(int M, int N, int K, int epi, int ks, int bm) {
  if (bm != 256 && bm != 192 && bm != 128 && bm != LK_GEMM1W_SPLIT128 && bm != LK_GEMM1W_SPLIT192) return 0;
  if (M < 1 || K % kBK || ks < 1 || ks > 8 || K / kBK < 3 * ks) return 0;  // >= 3 K-tiles per split
  if (ks > 1 && (epi == E_SWIGLU || epi == E_QKV || N % 256)) return 0;
  if (epi == E_SWIGLU) return N % 2 == 0 && (N / 2) % 128 == 0;
  if (epi == E_RESID || epi == E_QKV) return N % kBN == 0;
  return epi >= E_NONE && epi <= E_BIAS_RELU && N % kBN == 0;
}

// out = epi(X W^T (+ bias)): the contract of lk_gemm with a bm x 256 tile, bm = 256 / 192 / 128
// (ea: the fused chain arguments, see kernels.h).  group_m <= 0: LK_GEMM_GROUP_M / 4.
int lk_gemm1w(const bf16_t* x, long ldx, const bf16_t* w, const bf16_t* bias, int M, int N, int K, int epi,
              bf16_t* out, long ldo, hipStream_t st, int ks, float* ws, const LkEpi* ea_, int group_m, int bm) {
  LkEpi ea = ea_ ? *ea_ : LkEpi{};
  if (ea.ss_in && (ea.ss_nt < 1 || ea.ss_nt > 32 || ea.ss_ld < M || ea.inv_h <= 0.f || ks > 1)) return -1;
  if (epi == E_RESID && (!ea.resid || !ea.ss_out || ea.ldr % 8 || ea.ss_out_ld < M)) return -1;
  if (epi == E_QKV && (!ea.pos || !ea.cos_sin || ea.hd % 16 || ea.hd <= 0 || N != (ea.hq + 2 * ea.hkv) * ea.hd ||
                       ((ea.kc || ea.vc) && (!ea.slots || ea.bs < 1))))
    return -1;
  if (!lk_gemm1w_supported(M, N, K, epi, ks, bm) || ldx % 8 || ldo % 8 || reinterpret_cast<uintptr_t>(out) % 16 ||
      (bias != nullptr && reinterpret_cast<uintptr_t>(bias) % 16))
    return -1;
  if (epi >= E_BIAS && epi <= E_BIAS_RELU && bias == nullptr) return -1;
  if ((long)N * K * 2 >= 0x7FFFFFF0L) return -1;
  // 32-bit buffer offsets: X, the output (fp32 partials for split-K) and the residual in row chunks
  const int bmx = bm < 128 ? 256 : bm;  // (a column split's largest row tile)
  const int TMall = (M + bmx - 1) / bmx;
  const long rows_pad = (long)TMall * bmx;
  const long xb = rows_pad * ldx * 2, ob = rows_pad * ldo * (ks > 1 ? 4 * ks : 2), rb = epi == E_RESID ? rows_pad * ea.ldr * 2 : 0;
  if (xb >= 0x7FFFFFF0L || ob >= 0x7FFFFFF0L || rb >= 0x7FFFFFF0L) {
    if (ea_ || ks > 1) return -1;  // (the fused chain indexes whole-M side buffers)
    const long per = max(ldx, ldo) * 2;
    const long max_rows = (0x7FFFFFF0L / per) / bmx * bmx - bmx;
    if (max_rows < bmx) return -1;
    for (long m0 = 0; m0 < M; m0 += max_rows) {
      const int mc = (int)min((long)M - m0, max_rows);
      const int rc = lk_gemm1w(x + m0 * ldx, ldx, w, bias, mc, N, K, epi, out + m0 * ldo, ldo, st, 1, nullptr, nullptr,
                               group_m, bm);
      if (rc) return rc;
    }
    return 0;
  }
  if (ks > 1) {  // fp32 partials of ks K-ranges into ws [ks, M, N], then the reduce applies the epilogue
    if (ws == nullptr) return -1;
    launch1w_sc<E_PARTIAL>(bm, x, ldx, w, nullptr, M, K, 0, reinterpret_cast<bf16_t*>(ws), N, N / kBN, ks, group_m, st,
                           ea);
    int rc = -1;
    switch (ks) {
#define LK_R1W(S) case S: rc = launch_reduce1w<S>(ws, M, N, epi, bias, out, ldo, st, ea); break;
      LK_R1W(2) LK_R1W(3) LK_R1W(4) LK_R1W(5) LK_R1W(6) LK_R1W(7) LK_R1W(8)
#undef LK_R1W
    }
    if (rc) return rc;
    LK_CHECK_LAUNCH();
    return 0;
  }
  switch (epi) {
    case E_NONE: launch1w_sc<E_NONE>(bm, x, ldx, w, bias, M, K, 0, out, ldo, N / kBN, 1, group_m, st, ea); break;
    case E_SWIGLU: launch1w_sc<E_SWIGLU>(bm, x, ldx, w, bias, M, K, N / 2, out, ldo, N / 256, 1, group_m, st, ea); break;
    case E_BIAS: launch1w_tiles<E_BIAS, 0>(bm, x, ldx, w, bias, M, K, 0, out, ldo, N / kBN, 1, group_m, st, ea); break;
    case E_BIAS_GELU: launch1w_tiles<E_BIAS_GELU, 0>(bm, x, ldx, w, bias, M, K, 0, out, ldo, N / kBN, 1, group_m, st, ea); break;
    case E_BIAS_RELU: launch1w_tiles<E_BIAS_RELU, 0>(bm, x, ldx, w, bias, M, K, 0, out, ldo, N / kBN, 1, group_m, st, ea); break;
    case E_RESID: launch1w_tiles<E_RESID, 0>(bm, x, ldx, w, nullptr, M, K, 0, out, ldo, N / kBN, 1, group_m, st, ea); break;
    case E_QKV: launch1w_sc<E_QKV>(bm, x, ldx, w, nullptr, M, K, 0, out, ldo, N / kBN, 1, group_m, st, ea); break;
    default: return -1;
  }
  LK_CHECK_LAUNCH();
  return 0;
}

// probes (benchmarks/gemm1w_probe.py): plain / SwiGLU / bias epilogues through ctypes
extern "C" int lk_gemm1w_c(const void* x, long ldx, const void* w, const void* bias, int M, int N, int K, int epi,
                           void* out, long ldo, void* stream, int group_m, int bm) {
  return lk_gemm1w((const bf16_t*)x, ldx, (const bf16_t*)w, (const bf16_t*)bias, M, N, K, epi, (bf16_t*)out, ldo,
                   (hipStream_t)stream, 1, nullptr, nullptr, group_m, bm);
}
