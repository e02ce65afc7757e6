// The K walk of the few-row products: a wave multiplies MT x 16 rows of X by NT x 16 rows of W over its own range of K,
// both streamed through a private LDS ring by 16-byte LDS-DMA (8 rows x one whole 128-byte line per instruction), counted
// vmcnt, no barrier.  The four waves of a workgroup split K; rg_sums() joins them.
#pragma once
#include "common.h"

constexpr int kRgWaves = 4;

typedef __attribute__((address_space(3))) void* rg_lptr;
typedef const __attribute__((address_space(1))) void* rg_gptr;

template <int N>
LK_DEVICE void rg_wait() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
}
LK_DEVICE void rg_wait_lds() { __builtin_amdgcn_s_waitcnt(0xF | (0x3 << 14) | (0x7 << 4)); }  // lgkmcnt(0) alone
template <int L, int AHEAD>
LK_DEVICE void rg_wait_ahead(int ahead) {  // all but the newest `ahead` stages of L loads have landed
  if constexpr (AHEAD > 0) {
    if (ahead >= AHEAD) {
      rg_wait<L * AHEAD>();
      return;
    }
    rg_wait_ahead<L, AHEAD - 1>(ahead);
  } else {
    rg_wait<0>();
  }
}

// 64 K columns of (MT + NT) 16-row tiles: one stage of a wave's ring
constexpr int rg_stage(int MT, int NT) { return (MT + NT) * 2048; }
constexpr int rg_lds(int MT, int NT, int NS) {
  const int ring = kRgWaves * NS * rg_stage(MT, NT), sums = kRgWaves * MT * NT * 1024;
  return ring > sums ? ring : sums;
}

// the part of an operand's pointer that lane and wave decide: LDS row `row` holds the eight 16-byte chunks of its 128 bytes
// in the order chunk ^ (row & 7), so that the fragment reads meet no bank twice
LK_DEVICE int rg_lane_col(int lane) { return ((lane & 7) ^ (lane >> 3)) * 8; }

// acc[m][n], lane l: row l & 15 of X tile m, rows 4 (l >> 4) .. + 3 of W tile n.  xs / ws: this lane's source (row lane >> 3 of
// the i-th 8 rows, rg_lane_col), at the wave's first column; nst: its stages of 64 columns.
template <int MT, int NT, int NS>
LK_DEVICE void rg_walk(const bf16_t* const (&xs)[2 * MT], const bf16_t* const (&ws)[2 * NT], int nst, unsigned char* ring,
                       floatx4 (&acc)[MT][NT]) {
  constexpr int SB = rg_stage(MT, NT), L = (MT + NT) * 2;
  const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
  auto issue = [&](int st) {
    unsigned char* base = ring + (st % NS) * SB;
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i)
      __builtin_amdgcn_global_load_lds((rg_gptr)(ws[i] + st * 64), (rg_lptr)(base + (2 * MT + i) * 1024), 16, 0, 2);
#pragma unroll
    for (int i = 0; i < 2 * MT; ++i)
      __builtin_amdgcn_global_load_lds((rg_gptr)(xs[i] + st * 64), (rg_lptr)(base + i * 1024), 16, 0, 0);
  };
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) acc[m][n] = (floatx4){0.f, 0.f, 0.f, 0.f};
  // Three stages or more: the next is requested into the slot of the stage before, whose fragments its products have consumed.  Two: a
  // stage's fragments go to registers together and its own slot is requested again before the products, which keeps both on their way
  // (the wait for LDS in between costs 0.2 us of a walk of 8 stages, and a deeper ring gains nothing from it).
  constexpr bool SELF = NS < 3;
  constexpr int AHEAD = SELF ? NS : NS - 1;
#pragma unroll
  for (int p = 0; p < AHEAD; ++p)
    if (p < nst) issue(p);
  for (int st = 0; st < nst; ++st) {
    rg_wait_ahead<L, AHEAD - 1>(min(AHEAD - 1, nst - 1 - st));
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (!SELF) {
      if (st + AHEAD < nst) issue(st + AHEAD);
      __builtin_amdgcn_sched_barrier(0);
    }
    const unsigned char* base = ring + (st % NS) * SB;
    short8 a[2][MT], b[2][NT];
    auto read = [&](int h) {
      const int at = r16 * 128 + (((4 * h + g) ^ (r16 & 7)) << 4);
#pragma unroll
      for (int n = 0; n < NT; ++n) b[h][n] = *reinterpret_cast<const short8*>(base + (MT + n) * 2048 + at);
#pragma unroll
      for (int m = 0; m < MT; ++m) a[h][m] = *reinterpret_cast<const short8*>(base + m * 2048 + at);
    };
    read(0);
    if constexpr (SELF) {
      read(1);
      if (st + AHEAD < nst) {
        __builtin_amdgcn_sched_barrier(0);
        rg_wait_lds();   // the reads are done before a load may write there
        __builtin_amdgcn_sched_barrier(0);
        issue(st + AHEAD);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      if (!SELF && h == 1) read(1);
      // W as the A operand: the lane ends with one output row and 4 consecutive columns
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[m][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[h][n], a[h][m], acc[m][n], 0, 0, 0);
    }
  }
}

// The four waves' partial tiles through LDS (the rings' memory, read by everyone before): wave m, m + 4, .. gets tile row m
// from total(m, t) with t[n] = the sum of tile n.
template <int MT, int NT, typename F>
LK_DEVICE void rg_sums(unsigned char* smem, const floatx4 (&acc)[MT][NT], F total) {
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __syncthreads();
  floatx4* part = reinterpret_cast<floatx4*>(smem);
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int n = 0; n < NT; ++n) part[(wave * MT * NT + m * NT + n) * 64 + lane] = acc[m][n];
  __syncthreads();
#pragma unroll
  for (int m = wave; m < MT; m += kRgWaves) {
    floatx4 t[NT];
#pragma unroll
    for (int n = 0; n < NT; ++n) {
      t[n] = part[(m * NT + n) * 64 + lane];
#pragma unroll
      for (int w = 1; w < kRgWaves; ++w) t[n] += part[((w * MT + m) * NT + n) * 64 + lane];
    }
    total(m, t);
  }
}
