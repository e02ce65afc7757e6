// Prompt rows of bf16 over a paged K/V cache ([blocks, G, BS, dim] and key-contiguous [blocks, G, vdim, BS]), the keys and values of a
// step staged in LDS once for the four waves of a workgroup: 16 consecutive queries of a head per wave, the waves side by side
// over wh heads of one kv group and 4 / wh runs of queries, so a staged tile of 32 keys serves 64 (query, head) columns.
//
// Straight from the cache into the fragments of one wave (16 queries, four waves over the keys), each of a K/V line's many readers
// waits for it on its own; that walk was bound by those waits.  Here one LDS-DMA instruction moves 1 KB of whole key rows, or the 16-key
// pieces of 32 value rows, in the order of their addresses (as fragments, 16 rows x 64 bytes, the loads were a third of the loop);
// the 16-byte chunks are placed so that the fragment reads meet no bank twice.  The two tiles behind the present one are on their
// way, with one barrier per tile.  The block table is read by scalar loads, so that the waits count fragments alone.
//
// A wave's step is a chain (LDS, products, exponentials, products), so what counts is how many waves hide each other's: 16 queries and three
// buffers leave three per SIMD.  32 queries per wave (two waves per SIMD, half the LDS traffic) took 72 instead of 48 us, four buffers
// (two waves) likewise.
//
// What a wave's 16 queries meet is what they met alone: tiles between their own first and last visible key, and in the last of
// them nothing of the key runs of 8 behind it (an infinity or NaN there, times a weight of zero, would reach them).
#pragma once
#include "common.h"
#include "attn_frag.h"

namespace {

constexpr int kStageMaxPad = 128;   // head sizes up to here: beyond, accumulators leave too few waves

struct StageCache {
  const bf16_t* kc;
  const bf16_t* vc;
  const int* bt;   // of the sequence
  int G, kvh, dim, vdim, BS, bs_shift;   // bs_shift: log2(BS), -1 when BS is no power of two
};

// What the columns past a head that does not fill PAD hold: they meet zeros of q, and an infinity or NaN there (a piece of the key again)
// times zero would reach the scores.
__device__ __attribute__((aligned(16))) const bf16_t stage_zeros[8] = {};

constexpr int kStageBufs = 3;
constexpr int stage_frags(int PAD) { return 2 * (PAD / 32) + PAD / 16; }   // a multiple of 4: every wave fetches as many
constexpr int stage_lds(int PAD) { return kStageBufs * stage_frags(PAD) * 1024; }

template <int L, int AHEAD>
LK_DEVICE void stage_wait(int ahead) {  // all but the newest `ahead` tiles of L fragments have arrived
  if (ahead >= AHEAD) {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(L * AHEAD) : "memory");
    return;
  }
  if constexpr (AHEAD > 0) stage_wait<L, AHEAD - 1>(ahead);
}
// Whether a step's prompt rows take the staged kernel (PAD: the padded head size; window: the keys that a query sees, 0 for all; the
// pooled or kept keys behind a window are few).  Staged, a wave walks all keys of its 16 queries, so it needs (tile, head) pairs for
// every CU, or short walks; else the kernel whose four waves split a tile's keys is faster.  The key counts are on the device: the line
// is drawn by pairs alone.  Split / staged in us, sigmoid and causal softmax:
//   16 heads of 128 over 4:  16 rows behind 8,000 keys 193 / 252 and 183 / 286, 512 rows (512 pairs) behind 2,000 66 / 80 and 65 / 94,
//     1,024 rows 135 / 95 and 129 / 112, 2,048 rows 304 / 130 and 354 / 149;
//   16 heads of 64:  1,024 rows (1,024 pairs) behind 2,000 keys 68 / 92 and 60 / 119, 2,048 rows 153 / 154 and 237 / 182;
//   12 heads of 96:  1,536 pairs 0.6 - 1.0 and 0.7 - 1.4 of the time, 2,048 pairs 0.5 - 0.85 and 0.6 - 1.1.
// At 1,024 pairs of 128 one causal prompt from its first token is slower still (16 heads, 1,024 rows 40 / 45; 8 heads, 2,048 rows 62 / 82),
// several prompts or a longer past are faster (16 x 64 rows 17 / 10).  Windows of 512: 16 rows 44 / 26, 2,048 rows 68 / 31.
// (65,535 tiles: the grid)
inline bool stage_pays(long ntiles, int H, int PAD, int window) {
  if (PAD > kStageMaxPad || ntiles > 65535) return false;
  return (window > 0 && window <= 512) || ntiles * H >= (PAD > 96 ? 1024 : 2048);
}
inline int stage_heads(int rep) { return rep % 4 == 0 ? 4 : rep % 2 == 0 ? 2 : 1; }   // wh: the most that divide the heads of a kv group

// The place of chunk c among the CPR of key row `row` (dir 1), or the chunk at place c (dir -1): turned by the row, so that the 16 rows
// of a fragment (bits 0, 1, 3, 4 of the row) put the same chunk into different banks.
template <int CPR>
LK_DEVICE int stage_chunk(int c, int row, int dir) {
  const int n = (row & 3) | ((row >> 3) << 2);
  if constexpr ((CPR & (CPR - 1)) == 0) return c ^ (n & (CPR - 1));
  const int t = c + dir * ((n >> 1) & 3);   // 12: four more rows apart by their odd bit's 64 bytes
  return t < 0 ? t + CPR : t >= CPR ? t - CPR : t;
}

// q fragments of one row (zeros past dim)
template <int PAD>
LK_DEVICE void stage_q(const bf16_t* qrow, int dim, uint4_t (&qf)[PAD / 32]) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int s = 0; s < PAD / 32; ++s) {
    const int d0 = 32 * s + 8 * g;
    qf[s] = d0 < dim ? ld16(qrow + d0) : uint4_t{0u, 0u, 0u, 0u};
  }
}

// Keys [k0, k1) of the workgroup (k0 a multiple of 32); this wave takes part in tiles of [g0, g1) (g0 a multiple of 32; g1 <= g0: none).
// weights(kb, s0, s1) gives the 8 weights of keys kb + 8 g .. + 7 for column lane & 15 from the raw scores (in
// that order) as bf16.  Every wave of the workgroup calls this with the same k0 and k1.  FULL: dim is PAD (the test per request for others
// took 5 % of a prompt's softmax).
template <int PAD, bool FULL, typename F>
LK_DEVICE void stage_walk(const StageCache& p, bf16_t* lds, uint4_t (&qf)[PAD / 32], int k0, int k1, int g0, int g1, floatx4 (&o)[PAD / 16],
                          F weights) {
  constexpr int KS = PAD / 32, VT = PAD / 16, NK = 2 * KS, FR = NK + VT, CPR = PAD / 8;   // CPR: 16-byte chunks of a key row
  static_assert(FR % 4 == 0 && FR == stage_frags(PAD), "fragments per wave");
  // (q has arrived: else the loop would wait for it, and with it for every fragment)
#pragma unroll
  for (int i = 0; i < KS; ++i) asm volatile("" : "+v"(qf[i]));
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n16 = lane & 15, g = lane >> 4;
  const int krow = 8 * (n16 >> 2) + (n16 & 3);   // K row of a fragment's row n16: lane group g then has the weights of keys 8 g .. 8 g + 7
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((lds_void_ptr)lds);
  // (keys behind the last are never read: places are clamped to the last one, which weighs zero; BS is a multiple of 16, so each half
  // of a tile lies in one block)
  int pg[2], at[2];   // the blocks of the halves of the next tile to be requested, and their first keys
  auto pages = [&](int kb) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int key = min(kb + 16 * h, k1 - 1), page = __builtin_amdgcn_readfirstlane(p.bs_shift >= 0 ? key >> p.bs_shift : key / p.BS);
      pg[h] = ((const __attribute__((address_space(4))) int*)p.bt)[page];
      at[h] = page * p.BS;
    }
  };
  auto issue = [&](int kb, int buf) {
#pragma unroll
    for (int i = 0; i < FR / 4; ++i) {
      const int f = 4 * i + w;
      const unsigned off = lds0 + (unsigned)(buf * FR + f) * 1024u;
      if (f < NK) {
        const int q = 64 * f + lane, row = q / CPR, ch = stage_chunk<CPR>(q % CPR, row, -1), h = row >> 4;
        const bf16_t* kr = p.kc + (((long)(h ? pg[1] : pg[0]) * p.G + p.kvh) * p.BS - (h ? at[1] : at[0]) + min(kb + row, k1 - 1)) * p.dim;
        dma16(off, FULL || 8 * ch < p.dim ? kr + 8 * ch : stage_zeros);
      } else {
        const int h = (f - NK) / (VT / 2), vd = (f - NK) % (VT / 2) * 32 + (lane >> 1), c = (lane ^ (vd >> 2)) & 1;
        const bf16_t* vr = p.vc + ((long)(h ? pg[1] : pg[0]) * p.G + p.kvh) * p.vdim * p.BS + min(kb + 16 * h + 8 * c, (k1 - 1) & ~7) - (h ? at[1] : at[0]);
        dma16(off, vr + (long)min(vd, p.vdim - 1) * p.BS);   // (values past vdim are not stored)
      }
    }
  };
  // this lane's places in a tile: chunk 4 s + g of K rows krow + 4 t, and the run 8 g of V row 16 vt + n16
  int kat[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) kat[s] = (krow * CPR + stage_chunk<CPR>(4 * s + g, krow, 1)) * 8;
  const int vat = NK * 512 + (g >> 1) * (VT / 2) * 512 + n16 * 16 + (((g & 1) ^ (n16 >> 2)) & 1) * 8;
  if (k0 >= k1) return;
  __syncthreads();   // (a walk before this one has read its last tiles)
  pages(k0);
  for (int t = 0; t < kStageBufs - 1; ++t)
    if (k0 + 32 * t < k1) {
      issue(k0 + 32 * t, t);
      pages(k0 + 32 * (t + 1));
    }
  int buf = 0;
  for (int kb = k0; kb < k1; kb += 32, buf = buf + 1 < kStageBufs ? buf + 1 : 0) {
    stage_wait<FR / 4, kStageBufs - 2>((k1 - 1 - kb) >> 5);   // this wave's part of the tile has arrived
    __syncthreads();                                          // all of it has, and the tile before has been consumed
    const int kn = kb + 32 * (kStageBufs - 1);
    if (kn < k1) {
      issue(kn, buf ? buf - 1 : kStageBufs - 1);   // where the tile before lay
      pages(kn + 32);
    }
    if (kb < g0 || kb >= g1) continue;
    const bf16_t* fr = lds + buf * FR * 512;
    // all K fragments are requested before the first product and all V fragments before the weights (left alone, the compiler waits
    // for LDS pair by pair)
    floatx4 c[2];
    uint4_t kf[2][KS], vf[VT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[t][s] = ld16(fr + kat[s] + t * (4 * CPR * 8));   // (rows krow and krow + 4 are placed alike)
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) c[t] = mma_qk<bf16_t>(kf[t][s], qf[s], s == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : c[t]);
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) vf[vt] = ld16(fr + vat + vt * 256);
    __builtin_amdgcn_sched_barrier(0);
    const short8 pb = weights(kb, c[0], c[1]);
    if (kb + 32 > g1) {   // (wave-uniform)
      const bool seen = kb + 8 * g < g1;   // this lane group's run of 8 keys
#pragma unroll
      for (int vt = 0; vt < VT; ++vt)
#pragma unroll
        for (int e = 0; e < 4; ++e) vf[vt][e] = seen ? vf[vt][e] : 0u;
    }
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(short8, vf[vt]), pb, o[vt], 0, 0, 0);
  }
}

// Decode: one wave alone with keys first, first + 128, .. (32 at a time) below k1, read once and therefore non-temporally, through its own
// 1 / 4 of the workgroup's LDS without a barrier.  A step's fragments go to registers together, so that the next step's 16 KB (heads of 128)
// are requested before this step's arithmetic.  As fragments straight from the cache, 16 rows x 64 bytes, a CU took 17 KB/us.
constexpr int stage_wave_lds(int PAD) { return 4 * stage_frags(PAD) * 1024; }

template <int PAD, bool FULL, typename F>
LK_DEVICE void stage_wave(const StageCache& p, bf16_t* lds, uint4_t (&qf)[PAD / 32], int first, int k1, floatx4 (&o)[PAD / 16], F weights) {
  constexpr int KS = PAD / 32, VT = PAD / 16, NK = 2 * KS, FR = NK + VT, CPR = PAD / 8;
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n16 = lane & 15, g = lane >> 4;
  const int krow = 8 * (n16 >> 2) + (n16 & 3);
  bf16_t* fr = lds + w * FR * 512;
  const unsigned lds0 = (unsigned)reinterpret_cast<uintptr_t>((lds_void_ptr)fr);
  auto issue = [&](int kb) {
    int pg[2], at[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int key = min(kb + 16 * h, k1 - 1), page = __builtin_amdgcn_readfirstlane(p.bs_shift >= 0 ? key >> p.bs_shift : key / p.BS);
      pg[h] = ((const __attribute__((address_space(4))) int*)p.bt)[page];
      at[h] = page * p.BS;
    }
#pragma unroll
    for (int f = 0; f < FR; ++f) {
      const unsigned off = lds0 + (unsigned)f * 1024u;
      if (f < NK) {
        const int q = 64 * f + lane, row = q / CPR, ch = stage_chunk<CPR>(q % CPR, row, -1), h = row >> 4;
        const bf16_t* kr = p.kc + (((long)(h ? pg[1] : pg[0]) * p.G + p.kvh) * p.BS - (h ? at[1] : at[0]) + min(kb + row, k1 - 1)) * p.dim;
        dma16<true>(off, FULL || 8 * ch < p.dim ? kr + 8 * ch : stage_zeros);
      } else {
        const int h = (f - NK) / (VT / 2), vd = (f - NK) % (VT / 2) * 32 + (lane >> 1), c = (lane ^ (vd >> 2)) & 1;
        const bf16_t* vr = p.vc + ((long)pg[h] * p.G + p.kvh) * p.vdim * p.BS + min(kb + 16 * h + 8 * c, (k1 - 1) & ~7) - at[h];
        dma16<true>(off, vr + (long)min(vd, p.vdim - 1) * p.BS);
      }
    }
  };
  int kat[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) kat[s] = (krow * CPR + stage_chunk<CPR>(4 * s + g, krow, 1)) * 8;
  const int vat = NK * 512 + (g >> 1) * (VT / 2) * 512 + n16 * 16 + (((g & 1) ^ (n16 >> 2)) & 1) * 8;
  // (a walk before this one has its last fragments in registers)
  if (first < k1) issue(first);
#pragma unroll
  for (int i = 0; i < KS; ++i) asm volatile("" : "+v"(qf[i]));   // (q has arrived: the waits in the loop are for fragments alone)
  for (int kb = first; kb < k1; kb += 128) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    uint4_t kf[2][KS], vf[VT];
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int s = 0; s < KS; ++s) kf[t][s] = ld16(fr + kat[s] + t * (4 * CPR * 8));
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) vf[vt] = ld16(fr + vat + vt * 256);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the fragments are read before a load may write there
    __builtin_amdgcn_sched_barrier(0);
    if (kb + 128 < k1) issue(kb + 128);
    __builtin_amdgcn_sched_barrier(0);
    floatx4 c[2];
#pragma unroll
    for (int s = 0; s < KS; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) c[t] = mma_qk<bf16_t>(kf[t][s], qf[s], s == 0 ? floatx4{0.f, 0.f, 0.f, 0.f} : c[t]);
    const short8 pb = weights(kb, c[0], c[1]);
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) o[vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(short8, vf[vt]), pb, o[vt], 0, 0, 0);
  }
}

}  // namespace
