// Rows of a step's projections on their way to the paged caches (bf16), the parts that the kernels which norm or
// rotate them share.  A workgroup takes R adjacent rows and a part of their heads: R = 16 for prompts, where the
// values of 16 tokens are turned round in LDS so that a store instruction writes the runs of 16 tokens that a
// key-contiguous block [vdim][BS] holds side by side (4 x 32 bytes instead of 64 two-byte pieces in 64 sectors),
// R = 1 for steps of few rows, where the heads' parts give every row several workgroups instead of one.  A head is
// LPH lanes of 8 elements (16-byte accesses); rotated pairs and a head's sum of squares stay inside its lanes.
#pragma once
#include "common.h"

constexpr int kFileRows = 16;      // rows of a prompt tile
constexpr int kFileFewRows = 512;  // steps of fewer rows take one row per workgroup (a tile of 16 leaves CUs without work)

template <int R, int LPH>
struct KvTile {
  static constexpr int HEADS = R == 1 ? 256 / LPH : 4;  // q / k heads of a part
  static constexpr int VCOLS = R == 1 ? 2048 : 512;     // value columns of a part
};

// lanes of a head of up to 256 elements
inline int kv_lanes(int dim) { return dim <= 64 ? 8 : dim <= 128 ? 16 : 32; }

// Columns [c0, c1) of the G heads' values (column = head * VD + d, multiples of 8) of `tl` rows from row t0:
// val(row, head, d, f) gives 8 of them.  sv: R > 1 only, [R][VCOLS + 2].
template <int R, int VCOLS, typename F>
LK_DEVICE void kv_file_values(const int* __restrict__ slots, long t0, int tl, int c0, int c1, int G, int VD, int BS, bf16_t* __restrict__ vc,
                              bf16_t (*sv)[VCOLS + 2], F val) {
  if constexpr (R == 1) {
    const int slot = slots[t0];
    if (slot < 0) return;
    const long blk = slot / BS;
    const int off = slot % BS;
    for (int c = c0 + threadIdx.x * 8; c < c1; c += 2048) {
      float f[8];
      val(t0, c / VD, c % VD, f);
      bf16_t* dst = vc + (blk * G * VD + c) * (long)BS + off;
#pragma unroll
      for (int e = 0; e < 8; ++e) dst[(long)e * BS] = f2bf(f[e]);
    }
  } else {
    const int nc = c1 - c0, per = nc / 8;
    for (int i = threadIdx.x; i < tl * per; i += 256) {
      const int r = i / per, c = c0 + (i % per) * 8;
      float f[8];
      val(t0 + r, c / VD, c % VD, f);
#pragma unroll
      for (int e = 0; e < 8; e += 2) *reinterpret_cast<unsigned*>(&sv[r][c - c0 + e]) = pack_bf2(f[e], f[e + 1]);
    }
    __syncthreads();
    const int r = threadIdx.x & (R - 1);  // lanes run over the rows first
    const int slot = r < tl ? slots[t0 + r] : -1;
    if (slot < 0) return;
    bf16_t* dst = vc + ((long)(slot / BS) * G * VD + c0) * BS + slot % BS;
    for (int c = threadIdx.x / R; c < nc; c += 256 / R) dst[(long)c * BS] = sv[r][c];
  }
}
