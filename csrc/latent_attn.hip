// Softmax attention over a cached latent that all query heads share.  A token's cache row is [latent c (RP columns) | rotated key
// part (RDP columns)], KD = RP + RDP; the queries have been brought to it, so
//
//   s(i, j) = scale * <qa_(i, h), row_j>                 for first(i) <= j <= i      (sliding window; 0: causal)
//   p(i, j) = exp(s(i, j)) / (exp(sink_h) + sum_j' exp(s(i, j')))                    (the sink is optional, not scaled)
//   lat_(i, h) = sum_j p(i, j) c_j                       the average goes through the head's value projection afterwards
//
// One row serves scores and values of every head: a tile of 32 rows is staged in LDS once and multiplied with many (query, head)
// columns.  Wave layout: 16 columns against 32 keys,
//   S^T (keys x columns) = rows . qa^T  on v_mfma_f32_16x16x32_bf16 (rows as 16-byte LDS fragments, queries in registers),
//   O^T (latent x columns) += c^T . P^T with c^T by transposed LDS reads (ds_read_b64_tr_b16) and P^T straight from the S^T
//   accumulators (both sides use the key order 4g + j, 16 + 4g + j).
// LDS rows are unpadded multiples of 128 bytes; the 16-byte pieces of a row are XOR-swizzled inside groups of 8 so that both kinds
// of reads spread over the banks.
//
// Prompt portions: a workgroup owns 128 columns = the heads of a block x consecutive queries of one sequence (32
// columns per wave), tiles double-buffered.  Decode rows: a workgroup (4 waves) owns a sequence and a block of at most 16 heads, each wave walks its own
// tiles (LDS-DMA into a wave-private region), merged through LDS; key splits over workgroups are merged by a second kernel.
// f32 rows (and latents wider than the instances) run on a plain kernel, one workgroup per (row, head).
//
// Masks are taken from absolute positions: a prompt cut anywhere, a decode row and a whole prompt are the same sums.
//
// lk_latent_prep prepares the operands (norms, rotation, the cache row) in f32; the queries come from head_linear.hip.
#include <type_traits>

#include "common.h"
#include "kernels.h"
#include "attn_frag.h"

namespace {

typedef const __attribute__((address_space(1))) void* gbl_void_ptr;

constexpr float kNegBig = -1e30f;
constexpr float kLog2e = 1.4426950408889634f;

struct LatParams {
  const void* q;       // [rows, H, KD]
  long qs;             // elements between rows
  const void* cache;   // [blocks, BS, KD]
  const int* bt;
  int bt_stride;
  int BS, H, HC, KD, RP;   // HC: heads per block
  int window;          // 0: causal
  float scale;
  const float* sink;   // [H] or null
  void* out;           // [rows, H, OH]: the averages, or with OH = 2 RP their bf16 value and, RP columns on, the bf16 of the rest
  long os;
  int OH;
  const void* gate;    // rows aligned with q's: the averages of head h times sigmoid(column h); null: none
  long gs;
};

template <typename T>
LK_DEVICE float lat_gate(const LatParams& p, long row, int head) {
  if (!p.gate) return 1.f;
  const float g = El<T>::ld(reinterpret_cast<const T*>(p.gate) + row * p.gs + head);
  return sizeof(T) == 4 ? 1.f / (1.f + expf(-g)) : __builtin_amdgcn_rcpf(1.f + __expf(-g));
}

// four averages of a row whose parts start at o: one rounding to bf16, or two parts that keep 16 bits
LK_DEVICE void store_avg(const LatParams& p, bf16_t* o, const float (&v)[4]) {
  short4_t hi, lo;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const bf16_t h = f2bf(v[j]);
    hi[j] = (short)h;
    lo[j] = (short)f2bf(v[j] - bf2f(h));
  }
  *reinterpret_cast<short4_t*>(o) = hi;
  if (p.OH > p.RP) *reinterpret_cast<short4_t*>(o + p.RP) = lo;
}

LK_DEVICE int first_key(int qpos, int window) { return window > 0 ? max(0, qpos - window + 1) : 0; }

LK_DEVICE int swz(int row) { return (row & 6) | ((row >> 3) & 1); }

// A column's weights are 2^(s - m) with m = its largest score in the first tile it sees, not a running maximum: bf16 and f32 keep
// their relative precision at any scale, so sums and accumulators may grow with later, larger scores and are never rescaled
// (a rescale of accumulators that fill the registers costs a copy of all of them).  Only if a score passes m by more than this
// (base 2), the pass over the keys is repeated with m = the largest score of all.
constexpr float kMaxGrowth = 96.f;

// 32 staged rows (keys kb .. kb + 31) against CG groups of 16 columns: a row fragment read from LDS serves all groups.  m: the
// column's reference (kNegBig: no key seen yet), top: its largest score so far (both base 2, equal in the four lane groups of a
// column), l: this lane group's share of the sum, o: O^T accumulators.  qpos < 0: column without a query.
// LDS reads as assembly with explicit waits: the fragments of a tile stream through a ring of registers several places ahead of the
// MFMAs that use them (left to itself the compiler reads, waits and multiplies one fragment at a time when the accumulators fill
// the registers).  LDS reads return in order, so "at most N outstanding" names the oldest ones.
template <int OFF>
LK_DEVICE void lds_read16(uint4_t& v, unsigned addr) {
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
}
template <int OFF>
LK_DEVICE void lds_read_tr(short4_t& v, unsigned addr) {
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
}
template <int N, typename V>
LK_DEVICE void lds_wait(V& a, V& b) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(a), "+v"(b) : "n"(N));
}
template <int N, int I = 0, typename F>
LK_DEVICE void static_for(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<N, I + 1>(f);
  }
}

template <int RP, int RDP, int CG, bool THIN>
LK_DEVICE void lat_tile(const bf16_t* tile, const uint4_t (&qf)[CG][(RP + RDP) / 32], int kb, const int (&qpos)[CG], const int (&klo)[CG], float s2,
                        float (&m)[CG], float (&top)[CG], float (&l)[CG], floatx4 (&o)[CG][RP / 16]) {
  constexpr int KD = RP + RDP, NKS = KD / 32, VT = RP / 16;
  constexpr int QA = RP > 256 && CG == 1 && THIN ? 3 : 4, VA = 4;   // fragments requested ahead of their products (QA pairs, VA c^T fragments)
  const int lane = threadIdx.x & 63, n16 = lane & 15, g = lane >> 4;
  const unsigned base = (unsigned)reinterpret_cast<uintptr_t>((lds_void_ptr)tile);
  floatx4 c[CG][2];
#pragma unroll
  for (int x = 0; x < CG; ++x) c[x][0] = c[x][1] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int sw = swz(n16);   // (rows n16 and 16 + n16 have the same swizzle)
  const unsigned k0 = base + n16 * KD * 2 + (g ^ sw) * 16, k1 = base + n16 * KD * 2 + ((4 + g) ^ sw) * 16;
  uint4_t kf[QA][2];
  static_for<QA>([&](auto sc_) {
    constexpr int s = decltype(sc_)::value;
    lds_read16<128 * (s / 2)>(kf[s][0], (s & 1) ? k1 : k0);
    lds_read16<128 * (s / 2) + 16 * KD * 2>(kf[s][1], (s & 1) ? k1 : k0);
  });
  static_for<NKS>([&](auto sc_) {
    constexpr int s = decltype(sc_)::value, ahead = (s + QA < NKS ? QA : NKS - s) - 1;
    lds_wait<2 * ahead>(kf[s % QA][0], kf[s % QA][1]);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int x = 0; x < CG; ++x) c[x][t] = mma_qk<bf16_t>(kf[s % QA][t], qf[x][s], c[x][t]);
    if constexpr (s + QA < NKS) {
      lds_read16<128 * ((s + QA) / 2)>(kf[s % QA][0], ((s + QA) & 1) ? k1 : k0);
      lds_read16<128 * ((s + QA) / 2) + 16 * KD * 2>(kf[s % QA][1], ((s + QA) & 1) ? k1 : k0);
    }
  });
  // the first c^T fragments travel under the softmax arithmetic
  const int qq = n16 >> 2, pp = n16 & 3, swv = swz(4 * g + qq);   // rows 4g + qq and 16 + 4g + qq have the same swizzle
  const unsigned vr = base + (4 * g + qq) * KD * 2 + 8 * (pp & 1);
  unsigned va[4];
#pragma unroll
  for (int x = 0; x < 4; ++x) va[x] = vr + ((2 * x + (pp >> 1)) ^ swv) * 16;
  short4_t vlo[VA], vhi[VA];
  static_for<VA>([&](auto vc_) {
    constexpr int vt = decltype(vc_)::value;
    lds_read_tr<128 * (vt / 4)>(vlo[vt], va[vt % 4]);
    lds_read_tr<128 * (vt / 4) + 16 * KD * 2>(vhi[vt], va[vt % 4]);
  });
  short8 pb[CG];
#pragma unroll
  for (int x = 0; x < CG; ++x) {
    float sc[2][4];
    bool ok[2][4];
    float mx = kNegBig;
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int key = kb + 16 * t + 4 * g + j;
        ok[t][j] = key <= qpos[x] && key >= klo[x];
        sc[t][j] = c[x][t][j] * s2;
        if (ok[t][j]) mx = fmaxf(mx, sc[t][j]);
      }
    mx = max_groups(mx);
    if (m[x] == kNegBig) m[x] = mx;
    top[x] = fmaxf(top[x], mx);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float p = ok[t][j] ? __builtin_amdgcn_exp2f(sc[t][j] - m[x]) : 0.f;
        l[x] += p;
        pb[x][4 * t + j] = (short)f2bf(p);
      }
  }
  static_for<VT>([&](auto vc_) {
    constexpr int vt = decltype(vc_)::value, ahead = (vt + VA < VT ? VA : VT - vt) - 1;
    lds_wait<2 * ahead>(vlo[vt % VA], vhi[vt % VA]);
    const short8 a = __builtin_shufflevector(vlo[vt % VA], vhi[vt % VA], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
    for (int x = 0; x < CG; ++x) o[x][vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[x], o[x][vt], 0, 0, 0);
    if constexpr (vt + VA < VT) {
      lds_read_tr<128 * ((vt + VA) / 4)>(vlo[vt % VA], va[(vt + VA) % 4]);
      lds_read_tr<128 * ((vt + VA) / 4) + 16 * KD * 2>(vhi[vt % VA], va[(vt + VA) % 4]);
    }
  });
}

template <int RP, int RDP>
LK_DEVICE void load_q(const bf16_t* qrow, bool valid, uint4_t (&qf)[(RP + RDP) / 32]) {
  const int g = (threadIdx.x & 63) >> 4;
#pragma unroll
  for (int s = 0; s < (RP + RDP) / 32; ++s) qf[s] = valid ? ld16(qrow + 32 * s + 8 * g) : uint4_t{0u, 0u, 0u, 0u};
}

// a page's number and place: shifts where pages hold a power of two of rows (a division of scalars is 40 instructions)
struct Paging {
  int BS, shift;
  LK_DEVICE explicit Paging(int bs) : BS(bs), shift((bs & (bs - 1)) == 0 ? __builtin_ctz(bs) : -1) {}
  LK_DEVICE int page(int key) const { return shift >= 0 ? key >> shift : key / BS; }
  LK_DEVICE int row(int key) const { return shift >= 0 ? key & (BS - 1) : key % BS; }
};
// the page of the 16-key group kg (a multiple of 16, clamped to the sequence's last group): pages hold a multiple of 16 rows, so
// a group lies in one page
LK_DEVICE int group_page(const int* bt, const Paging& pg, int kg, int last) { return bt[pg.page(min(kg, last))]; }

// 64 pieces of 16 bytes (one per lane) to 1,024 consecutive bytes of LDS at `dst` (wave-uniform), without registers.  Written as
// assembly: the builtin makes the compiler wait for it before every transposed LDS read, also of the other buffer.  The caller
// waits (vmcnt) before the piece is read.
LK_DEVICE void request_piece(const void* base, unsigned at, unsigned dst) {   // (base, dst: wave-uniform; at: this lane's bytes behind base)
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(dst), "v"(at), "s"(base) : "memory", "m0");
}

constexpr int kPreCols = 128;
// column groups per wave: two where the accumulators of both fit the registers
template <int RP>
constexpr int pre_groups() { return 2; }
template <int RP>
constexpr int pre_waves() { return kPreCols / (16 * pre_groups<RP>()); }

// the tile of a prompt workgroup, found by walking the sequences (at most ceil(qlen / NQ) tiles each, a sequence's last queries first: they
// see the most keys); false: none
LK_DEVICE bool find_tile(const int* cu_q, int nseq, int NQ, int& b, int& q0) {
  const int tile = blockIdx.x;
  int acc = 0;
  for (int i = 0; i < nseq; ++i) {
    const int nt = (cu_q[i + 1] - cu_q[i] + NQ - 1) / NQ;
    if (tile < acc + nt) {
      b = i;
      q0 = (nt - 1 - (tile - acc)) * NQ;
      return true;
    }
    acc += nt;
  }
  return false;
}

// 32 cache rows from key kb on (pages page0, page1) to LDS at dst without registers (LDS-DMA) by W waves: 64 pieces of 16 bytes per wave
// instruction, in the order of their places in LDS; the source piece of a place is the one the swizzle puts there
template <int KD, int W>
struct TileRequest {
  static constexpr int CPR = KD / 8, NCH = 32 * CPR, NL = (NCH / 64 + W - 1) / W, STEP = 64 * W;   // NL: instructions of a wave, STEP: pieces per round of the waves
  static_assert(16 * CPR % 64 == 0, "an instruction's pieces belong to one 16-key group");
  const bf16_t* group[2];
  unsigned dst;
  int w, r, pos;   // row and place of this lane's piece, stepped from instruction to instruction (made anew per tile: registers are scarce)
  LK_DEVICE TileRequest(const bf16_t* cache, const Paging& pg, int kb, int last, int page0, int page1, unsigned char* to) {
    w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    group[0] = cache + ((long)__builtin_amdgcn_readfirstlane(page0) * pg.BS + pg.row(min(kb, last))) * KD;
    group[1] = cache + ((long)__builtin_amdgcn_readfirstlane(page1) * pg.BS + pg.row(min(kb + 16, last)) - 16) * KD;
    dst = __builtin_amdgcn_readfirstlane((unsigned)reinterpret_cast<uintptr_t>((lds_void_ptr)to));
    const int piece0 = 64 * w + (int)(threadIdx.x & 63);
    r = piece0 / CPR;
    pos = piece0 % CPR;
    asm volatile("" : "+v"(r), "+v"(pos));
  }
  LK_DEVICE void issue(int i) {   // the i-th, in order
    const int blk = W * i + w;    // wave-uniform
    if (NCH / 64 % W == 0 || blk < NCH / 64)
      request_piece(group[blk >= 16 * CPR / 64], (unsigned)(r * (KD * 2) + ((pos & ~7) | ((pos & 7) ^ swz(r))) * 16), dst + blk * 1024);
    r += STEP / CPR;
    pos += STEP % CPR;
    if (pos >= CPR) {
      pos -= CPR;
      ++r;
    }
  }
  LK_DEVICE void all() {
#pragma unroll
    for (int i = 0; i < NL; ++i) issue(i);
  }
};

// grid (query tiles, head blocks)
template <int RP, int RDP>
__global__ __launch_bounds__(pre_waves<RP>() * 64, RP >= 256 ? 1 : 2) void lat_prefill_kernel(LatParams p, const int* __restrict__ cu_q, const int* __restrict__ ctx_lens,
                                                                     int nseq) {
  constexpr int KD = RP + RDP, VT = RP / 16, CG = pre_groups<RP>();
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // two tiles of 32 rows
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), n16 = lane & 15, g = lane >> 4;
  const int NQ = kPreCols / p.HC;
  int b = 0, q0 = 0;
  if (!find_tile(cu_q, nseq, NQ, b, q0)) return;   // the whole workgroup leaves
  const int qbeg = cu_q[b], qlen = cu_q[b + 1] - qbeg, ctx = ctx_lens[b], past = ctx - qlen;
  uint4_t qf[CG][KD / 32];
  floatx4 o[CG][VT];
  float m[CG], top[CG], l[CG];
  int qpos[CG], klo[CG];
#pragma unroll
  for (int x = 0; x < CG; ++x) {
    const int c = 16 * (CG * w + x) + n16, qi = q0 + c / p.HC, head = blockIdx.y * p.HC + c % p.HC;
    const bool valid = c / p.HC < NQ && qi < qlen && head < p.H;
    qpos[x] = valid ? past + qi : -1;
    klo[x] = first_key(qpos[x], p.window);
    load_q<RP, RDP>(reinterpret_cast<const bf16_t*>(p.q) + (long)(qbeg + min(qi, qlen - 1)) * p.qs + (long)min(head, p.H - 1) * KD, valid, qf[x]);
    m[x] = kNegBig;
  }
  const float s2 = p.scale * kLog2e;
  const int k1 = min(ctx, past + q0 + NQ), k0 = first_key(past + q0, p.window) & ~31, last = (k1 - 1) & ~15;
  const int* bt = p.bt + (long)b * p.bt_stride;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(p.cache);
  const Paging pg(p.BS);
  auto request = [&](int kb, int page0, int page1, int which) { TileRequest<KD, pre_waves<RP>()>(cache, pg, kb, last, page0, page1, smem + which * 64 * KD).all(); };
  for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
    for (int x = 0; x < CG; ++x) {
      top[x] = kNegBig;
      l[x] = 0.f;
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) o[x][vt] = floatx4{0.f, 0.f, 0.f, 0.f};
    }
    request(k0, group_page(bt, pg, k0, last), group_page(bt, pg, k0 + 16, last), 0);
    int n0 = group_page(bt, pg, k0 + 32, last), n1 = group_page(bt, pg, k0 + 48, last);   // the pages of the tile to request next
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int cur = 0;
    for (int kb = k0; kb < k1; kb += 32) {
      if (kb + 32 < k1) {
        request(kb + 32, n0, n1, cur ^ 1);
        n0 = group_page(bt, pg, kb + 64, last);   // (raw: used, and waited for, in the next round)
        n1 = group_page(bt, pg, kb + 80, last);
      }
      lat_tile<RP, RDP, CG, true>(reinterpret_cast<const bf16_t*>(smem + cur * 64 * KD), qf, kb, qpos, klo, s2, m, top, l, o);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next tile has arrived (this wave's part of it)
      __syncthreads();
      cur ^= 1;
    }
    int again = 0;
#pragma unroll
    for (int x = 0; x < CG; ++x) {
      again |= top[x] > m[x] + kMaxGrowth;
      m[x] = pass == 0 && top[x] > m[x] + kMaxGrowth ? top[x] : m[x];
    }
    if (!__syncthreads_or(again)) break;
  }
#pragma unroll
  for (int x = 0; x < CG; ++x) {
    l[x] += __shfl_xor(l[x], 16, 64);
    l[x] += __shfl_xor(l[x], 32, 64);
    const int c = 16 * (CG * w + x) + n16, qi = q0 + c / p.HC, head = blockIdx.y * p.HC + c % p.HC;
    if (qpos[x] >= 0) {
      if (p.sink) l[x] += __builtin_amdgcn_exp2f(p.sink[head] * kLog2e - m[x]);   // one more term without a value
      const float f = l[x] > 0.f ? lat_gate<bf16_t>(p, qbeg + qi, head) / l[x] : 0.f;
      bf16_t* orow = reinterpret_cast<bf16_t*>(p.out) + (long)(qbeg + qi) * p.os + (long)head * p.OH + 4 * g;
#pragma unroll
      for (int vt = 0; vt < VT; ++vt) store_avg(p, orow + 16 * vt, {o[x][vt][0] * f, o[x][vt][1] * f, o[x][vt][2] * f, o[x][vt][3] * f});
    }
  }
}

// The same for latents of 512 + 64 columns, by two pairs of waves.  Four waves of 32 columns each fill a SIMD's registers alone, so nothing
// hides what a tile's steps wait for: 10,200 cycles a tile for 2,200 of MFMAs, 2,200 of other instructions and 1,700 of LDS.  A pair has 32
// columns: a wave takes half of the scores' dimensions and half of the latent for all of them and the softmax of its own 16.  Per tile
// the waves exchange partial scores (f32) and weights (bf16) of 16 columns through LDS, 6 KB a wave for the 34 KB of the tile that it no
// longer reads.  The registers halve, and two workgroups share a CU, each with its two tiles in half of the LDS to the byte, so one
// multiplies while the other waits at a barrier (one workgroup of four pairs: 133 us for the first line).  The next tile is requested an
// instruction per step of the scores: in one go that took 1,300 cycles in which the wave did nothing else.
// 4,095 rows of 4 prompts, 16 heads, window 512: 144 -> 129 us; 32 heads, window 2,048: 322 -> 282; 300 rows behind 700: 68 -> 44.  Many portions of
// little to read are where twice the workgroups, each of which walks the sequences for its tile, cost more: 200 of 16 rows behind 100, 93 -> 101.
constexpr int kPairWaves = 4, kPairCols = 16 * kPairWaves;
constexpr int pair_lds(int KD) { return 2 * 64 * KD + kPairWaves * 2048; }
template <int RP, int RDP>
constexpr bool in_pairs() { return RP > 256 && 2 * pair_lds(RP + RDP) <= 160 * 1024; }   // (512 + 128 columns: one workgroup a CU, 112 us for 87 by four single waves)
template <int RP, int RDP>
__global__ __launch_bounds__(64 * kPairWaves, 2) void lat_prefill_pair_kernel(LatParams p, const int* __restrict__ cu_q, const int* __restrict__ ctx_lens,
                                                                             int nseq) {
  constexpr int KD = RP + RDP, VT = RP / 16, HV = VT / 2, HS = KD / 64;   // HV, HS: c^T tiles and steps of 32 dimensions of a wave
  static_assert(TileRequest<RP + RDP, kPairWaves>::NL <= HS, "an instruction per step");
  constexpr int QA = 2, VA = 4;                                            // fragments requested ahead of their products
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];    // two tiles of 32 rows, the exchange
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), pr = w >> 1, hf = w & 1;
  int lane, n16, g;
  auto fresh = [&]() {   // addresses are made anew from these per tile: kept over the loop they would be spilled
    lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));
    n16 = lane & 15;
    g = lane >> 4;
  };
  fresh();
  const int NQ = kPairCols / p.HC;
  int b = 0, q0 = 0;
  if (!find_tile(cu_q, nseq, NQ, b, q0)) return;   // the whole workgroup leaves
  const int qbeg = cu_q[b], qlen = cu_q[b + 1] - qbeg, ctx = ctx_lens[b], past = ctx - qlen;
  floatx4* const xs = reinterpret_cast<floatx4*>(smem + 128 * KD) + 128 * w;                  // this wave's partial scores for its partner [2][64]
  const floatx4* const ys = reinterpret_cast<const floatx4*>(smem + 128 * KD) + 128 * (w ^ 1);   // the partner's for this wave, then this wave's weights
  // columns: y = 0 this wave's 16, y = 1 the partner's
  uint4_t qf[2][HS];
  int qpos = -1;
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int c = 16 * (2 * pr + (hf ^ y)) + n16, qi = q0 + c / p.HC, head = blockIdx.y * p.HC + c % p.HC;
    const bool valid = c / p.HC < NQ && qi < qlen && head < p.H;
    if (y == 0) qpos = valid ? past + qi : -1;
    const bf16_t* qrow = reinterpret_cast<const bf16_t*>(p.q) + (long)(qbeg + min(qi, qlen - 1)) * p.qs + (long)min(head, p.H - 1) * KD;
#pragma unroll
    for (int s = 0; s < HS; ++s) qf[y][s] = valid ? ld16(qrow + 32 * (hf * HS + s) + 8 * g) : uint4_t{0u, 0u, 0u, 0u};
  }
  const int klo = first_key(qpos, p.window);
  float m = kNegBig, top, l;
  floatx4 o[2][HV];
  const float s2 = p.scale * kLog2e;
  const int k1 = min(ctx, past + q0 + NQ), k0 = first_key(past + q0, p.window) & ~31, last = (k1 - 1) & ~15;
  const int* bt = p.bt + (long)b * p.bt_stride;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(p.cache);
  const Paging pg(p.BS);
  using Request = TileRequest<KD, kPairWaves>;
  auto handed = [&]() {   // LDS written and read as far as asked; the next tile stays on its way
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  for (int pass = 0; pass < 2; ++pass) {
    top = kNegBig;
    l = 0.f;
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int vt = 0; vt < HV; ++vt) o[y][vt] = floatx4{0.f, 0.f, 0.f, 0.f};
    Request(cache, pg, k0, last, group_page(bt, pg, k0, last), group_page(bt, pg, k0 + 16, last), smem).all();
    int n0 = group_page(bt, pg, k0 + 32, last), n1 = group_page(bt, pg, k0 + 48, last);   // the pages of the tile to request next
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    int cur = 0;
    for (int kb = k0; kb < k1; kb += 32) {
      fresh();
      const bool more = kb + 32 < k1;
      Request next(cache, pg, kb + 32, last, n0, n1, smem + (cur ^ 1) * 64 * KD);   // (requested between the scores' products: issuing takes its time)
      if (more) {
        n0 = group_page(bt, pg, kb + 64, last);   // (raw: used, and waited for, in the next round)
        n1 = group_page(bt, pg, kb + 80, last);
      }
      const unsigned base = (unsigned)reinterpret_cast<uintptr_t>((lds_void_ptr)(smem + cur * 64 * KD));
      // ---- this half's scores of both column groups: steps hf HS + s; the two 16-byte chunks of a 64-column piece alternate from step to step
      floatx4 c[2][2];
#pragma unroll
      for (int y = 0; y < 2; ++y) c[y][0] = c[y][1] = floatx4{0.f, 0.f, 0.f, 0.f};
      const int sw = swz(n16), S0 = hf * HS;   // (rows n16 and 16 + n16 have the same swizzle)
      const unsigned kc0 = base + n16 * KD * 2 + (g ^ sw) * 16, kc1 = base + n16 * KD * 2 + ((4 + g) ^ sw) * 16;
      const unsigned ke = ((S0 & 1) ? kc1 : kc0) + 128 * (S0 / 2), ko = ((S0 & 1) ? kc0 : kc1) + 128 * ((S0 + 1) / 2);
      uint4_t kf[QA][2];
      static_for<QA>([&](auto sc_) {
        constexpr int s = decltype(sc_)::value;
        lds_read16<128 * (s / 2)>(kf[s][0], (s & 1) ? ko : ke);
        lds_read16<128 * (s / 2) + 16 * KD * 2>(kf[s][1], (s & 1) ? ko : ke);
      });
      static_for<HS>([&](auto sc_) {
        constexpr int s = decltype(sc_)::value, ahead = (s + QA < HS ? QA : HS - s) - 1;
        lds_wait<2 * ahead>(kf[s % QA][0], kf[s % QA][1]);
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
          for (int y = 0; y < 2; ++y) c[y][t] = mma_qk<bf16_t>(kf[s % QA][t], qf[y][s], c[y][t]);
        if constexpr (s + QA < HS) {
          lds_read16<128 * ((s + QA) / 2)>(kf[s % QA][0], ((s + QA) & 1) ? ko : ke);
          lds_read16<128 * ((s + QA) / 2) + 16 * KD * 2>(kf[s % QA][1], ((s + QA) & 1) ? ko : ke);
        }
        if constexpr (s < Request::NL) {
          if (more) next.issue(s);
        }
      });
#pragma unroll
      for (int t = 0; t < 2; ++t) xs[t * 64 + lane] = c[1][t];
      handed();
      // ---- the softmax of this wave's columns (the c^T fragments are requested behind it: before the second hand-over they would have to be waited for)
      const int qq = n16 >> 2, pp = n16 & 3, swv = swz(4 * g + qq);   // rows 4g + qq and 16 + 4g + qq have the same swizzle
      const unsigned vr = base + (4 * g + qq) * KD * 2 + 8 * (pp & 1) + hf * (RP / 2) * 2;
      unsigned va[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) va[x] = vr + ((2 * x + (pp >> 1)) ^ swv) * 16;
      const floatx4 d0 = ys[lane], d1 = ys[64 + lane];
      float sc[2][4];
      bool ok[2][4];
      float mx = kNegBig;
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int key = kb + 16 * t + 4 * g + j;
          ok[t][j] = key <= qpos && key >= klo;
          sc[t][j] = (c[0][t][j] + (t ? d1[j] : d0[j])) * s2;
          if (ok[t][j]) mx = fmaxf(mx, sc[t][j]);
        }
      mx = max_groups(mx);
      if (m == kNegBig) m = mx;
      top = fmaxf(top, mx);
      short8 pb[2];
#pragma unroll
      for (int t = 0; t < 2; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float e = ok[t][j] ? __builtin_amdgcn_exp2f(sc[t][j] - m) : 0.f;
          l += e;
          pb[0][4 * t + j] = (short)f2bf(e);
        }
      const_cast<floatx4*>(ys)[lane] = __builtin_bit_cast(floatx4, pb[0]);   // (only this wave reads there before)
      handed();
      pb[1] = __builtin_bit_cast(short8, xs[lane]);
      // ---- this half of the latent for both column groups
      short4_t vlo[VA], vhi[VA];
      static_for<VA>([&](auto vc_) {
        constexpr int vt = decltype(vc_)::value;
        lds_read_tr<128 * (vt / 4)>(vlo[vt], va[vt % 4]);
        lds_read_tr<128 * (vt / 4) + 16 * KD * 2>(vhi[vt], va[vt % 4]);
      });
      static_for<HV>([&](auto vc_) {
        constexpr int vt = decltype(vc_)::value, ahead = (vt + VA < HV ? VA : HV - vt) - 1;
        lds_wait<2 * ahead>(vlo[vt % VA], vhi[vt % VA]);
        const short8 a = __builtin_shufflevector(vlo[vt % VA], vhi[vt % VA], 0, 1, 2, 3, 4, 5, 6, 7);
#pragma unroll
        for (int y = 0; y < 2; ++y) o[y][vt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pb[y], o[y][vt], 0, 0, 0);
        if constexpr (vt + VA < HV) {
          lds_read_tr<128 * ((vt + VA) / 4)>(vlo[vt % VA], va[(vt + VA) % 4]);
          lds_read_tr<128 * ((vt + VA) / 4) + 16 * KD * 2>(vhi[vt % VA], va[(vt + VA) % 4]);
        }
      });
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the next tile has arrived (this wave's part of it)
      __syncthreads();
      cur ^= 1;
    }
    // (a vote through the exchange's words: the library's takes LDS of its own, and then no second workgroup fits a CU)
    const bool grew = top > m + kMaxGrowth;
    m = pass == 0 && grew ? top : m;
    const int any = __any(grew);
    if (lane == 0) *reinterpret_cast<int*>(xs) = any;
    handed();
    int again = 0;
#pragma unroll
    for (int i = 0; i < kPairWaves; ++i) again |= *reinterpret_cast<const int*>(smem + 128 * KD + 2048 * i);
    handed();
    if (!again) break;
  }
  // ---- both groups' factors, then this half of the averages
  fresh();
  l += __shfl_xor(l, 16, 64);
  l += __shfl_xor(l, 32, 64);
  float f[2];
  const int c0 = 16 * (2 * pr + hf) + n16, head0 = blockIdx.y * p.HC + c0 % p.HC;
  if (p.sink && qpos >= 0) l += __builtin_amdgcn_exp2f(p.sink[head0] * kLog2e - m);   // one more term without a value
  f[0] = qpos >= 0 && l > 0.f ? lat_gate<bf16_t>(p, qbeg + q0 + c0 / p.HC, head0) / l : 0.f;
  reinterpret_cast<float*>(xs)[lane] = f[0];
  handed();
  f[1] = reinterpret_cast<const float*>(ys)[lane];
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int c = 16 * (2 * pr + (hf ^ y)) + n16, qi = q0 + c / p.HC, head = blockIdx.y * p.HC + c % p.HC;
    if (c / p.HC < NQ && qi < qlen && head < p.H) {
      bf16_t* orow = reinterpret_cast<bf16_t*>(p.out) + (long)(qbeg + qi) * p.os + (long)head * p.OH + hf * (RP / 2) + 4 * g;
#pragma unroll
      for (int vt = 0; vt < HV; ++vt) store_avg(p, orow + 16 * vt, {o[y][vt][0] * f[y], o[y][vt][1] * f[y], o[y][vt][2] * f[y], o[y][vt][3] * f[y]});
    }
  }
}

// grid (sequences, head blocks, key splits).  part: [B, H, Z, RP + 2] f32 = O^T relative to m (base 2), then m, l
template <int RP, int RDP>
__global__ __launch_bounds__(256) void lat_decode_kernel(LatParams p, const int* __restrict__ ctx_lens, int Z, float* __restrict__ part) {
  constexpr int KD = RP + RDP, CPR = KD / 8, VT = RP / 16, NCH = 32 * CPR;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];   // 4 wave-private regions of 32 rows
  const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, n16 = lane & 15, g = lane >> 4;
  const int b = blockIdx.x, z = blockIdx.z, ctx = ctx_lens[b];
  const int head = blockIdx.y * p.HC + n16;
  const bool valid = n16 < p.HC && head < p.H && ctx > 0;
  unsigned char* region = smem + w * 64 * KD;
  const int qpos[1] = {valid ? ctx - 1 : -1}, klo[1] = {first_key(ctx - 1, p.window)}, k0 = klo[0];
  const bf16_t* qrow = reinterpret_cast<const bf16_t*>(p.q) + (long)b * p.qs + (long)min(head, p.H - 1) * KD;
  uint4_t qf[1][KD / 32];
  load_q<RP, RDP>(qrow, valid, qf[0]);
  floatx4 o[1][VT];
  float m[1] = {kNegBig}, top[1], l[1];
  const float s2 = p.scale * kLog2e;
  const int nsteps = ctx > 0 ? (ctx - k0 + 31) / 32 : 0, spz = (nsteps + Z - 1) / Z, e1 = min(nsteps, (z + 1) * spz);
  const int* bt = p.bt + (long)b * p.bt_stride;
  const bf16_t* cache = reinterpret_cast<const bf16_t*>(p.cache);
  for (int pass = 0; pass < 2; ++pass) {
    top[0] = kNegBig;
    l[0] = 0.f;
#pragma unroll
    for (int vt = 0; vt < VT; ++vt) o[0][vt] = floatx4{0.f, 0.f, 0.f, 0.f};
    for (int step = z * spz + w; step < e1; step += 4) {
      const int kb = k0 + 32 * step;
      // tiles start at the first visible key (a window of 32 n keys is n tiles): lane x looks up the cache row of key kb + x % 32
      const int key = min(kb + (lane & 31), ctx - 1), mine = bt[key / p.BS] * p.BS + key % p.BS;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // the previous tile's LDS reads are done
  #pragma unroll
      for (int i = 0; i < NCH / 64; ++i) {
        // LDS piece x = 64 i + lane of the region is position x % CPR of row x / CPR: it holds the source piece swizzled back
        const int x = 64 * i + lane, r = x / CPR, pos = x % CPR, cc = (pos & ~7) | ((pos & 7) ^ swz(r));
        __builtin_amdgcn_global_load_lds((gbl_void_ptr)(cache + (long)__shfl(mine, r, 64) * KD + cc * 8), (lds_void_ptr)(region + i * 1024), 16, 0, 0);
      }
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lat_tile<RP, RDP, 1, false>(reinterpret_cast<const bf16_t*>(region), qf, kb, qpos, klo, s2, m, top, l, o);
    }
    if (!__any(top[0] > m[0] + kMaxGrowth)) break;
    m[0] = top[0] > m[0] + kMaxGrowth ? top[0] : m[0];
  }
  // ---- merge the 4 waves: (m, l) behind every region's O block, then O relative to the common maximum
  l[0] += __shfl_xor(l[0], 16, 64);
  l[0] += __shfl_xor(l[0], 32, 64);
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  float* ml = reinterpret_cast<float*>(region + 64 * RP);   // RP * 16 f32 of O come first; KD > RP leaves room behind them
  if (g == 0) {
    ml[n16] = m[0];
    ml[16 + n16] = l[0];
  }
  __syncthreads();
  // (the sink is one more term without a value, counted by the first split)
  const float sk = p.sink && z == 0 ? p.sink[min(head, p.H - 1)] * kLog2e : kNegBig;
  float M = sk, L = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) M = fmaxf(M, reinterpret_cast<const float*>(smem + i * 64 * KD + 64 * RP)[n16]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const float* q = reinterpret_cast<const float*>(smem + i * 64 * KD + 64 * RP);
    L += q[16 + n16] * __builtin_amdgcn_exp2f(q[n16] - M);
  }
  if (p.sink && z == 0) L += __builtin_amdgcn_exp2f(sk - M);
  const float f = __builtin_amdgcn_exp2f(m[0] - M);
  floatx4* ob = reinterpret_cast<floatx4*>(region);
#pragma unroll
  for (int vt = 0; vt < VT; ++vt) ob[vt * 64 + lane] = floatx4{o[0][vt][0] * f, o[0][vt][1] * f, o[0][vt][2] * f, o[0][vt][3] * f};
  __syncthreads();
  const float inv = L > 0.f ? lat_gate<bf16_t>(p, b, min(head, p.H - 1)) / L : 0.f;
#pragma unroll
  for (int i = 0; i < VT / 4; ++i) {
    const int vt = 4 * i + w;
    floatx4 s = reinterpret_cast<const floatx4*>(smem)[vt * 64 + lane];
#pragma unroll
    for (int x = 1; x < 4; ++x) {
      const floatx4 t = reinterpret_cast<const floatx4*>(smem + x * 64 * KD)[vt * 64 + lane];
#pragma unroll
      for (int j = 0; j < 4; ++j) s[j] += t[j];
    }
    if (n16 < p.HC && head < p.H) {
      if (Z == 1) {
        store_avg(p, reinterpret_cast<bf16_t*>(p.out) + (long)b * p.os + (long)head * p.OH + 16 * vt + 4 * g,
                  {s[0] * inv, s[1] * inv, s[2] * inv, s[3] * inv});
      } else {
        float* pp = part + (((long)b * p.H + head) * Z + z) * (RP + 2) + 16 * vt + 4 * g;
#pragma unroll
        for (int j = 0; j < 4; ++j) pp[j] = s[j];
      }
    }
  }
  if (Z > 1 && w == 0 && g == 0 && n16 < p.HC && head < p.H) {
    float* pp = part + (((long)b * p.H + head) * Z + z) * (RP + 2) + RP;
    pp[0] = M;
    pp[1] = L;
  }
}

// One workgroup per (sequence, head), four columns per thread.  A chain of three waits (maxima, sums, averages): the splits' maxima and
// sums are read by the lanes side by side and the averages four splits at a time; one split after the other it took 6.5 us at 64 x 16
// rows of 512 columns in 4 splits, 4.7 side by side.  Up to four splits every thread takes them all, requested together: the lanes' sums
// cost a step of few splits more than they save (whole decode attention, 64 x 32 rows of 256 columns in 2 splits of 512 keys: 13.8 -> 12.9).
constexpr int kLatFew = 4;

__global__ __launch_bounds__(256) void lat_reduce_kernel(LatParams p, const float* __restrict__ part, int Z) {
  const int b = blockIdx.x, head = blockIdx.y, RP = p.RP, lane = threadIdx.x & 63;
  const float* pp = part + ((long)b * p.H + head) * Z * (RP + 2);
  const float gate = lat_gate<bf16_t>(p, b, head);
  bf16_t* const orow = reinterpret_cast<bf16_t*>(p.out) + (long)b * p.os + (long)head * p.OH;
  float M = kNegBig, L = 0.f;
  if (Z <= kLatFew) {
    float e[kLatFew], l[kLatFew];
#pragma unroll
    for (int z = 0; z < kLatFew; ++z) {
      e[z] = z < Z ? pp[(long)z * (RP + 2) + RP] : kNegBig;
      l[z] = z < Z ? pp[(long)z * (RP + 2) + RP + 1] : 0.f;
    }
#pragma unroll
    for (int z = 0; z < kLatFew; ++z) M = fmaxf(M, e[z]);
#pragma unroll
    for (int z = 0; z < kLatFew; ++z) {
      e[z] = __builtin_amdgcn_exp2f(e[z] - M);
      if (z < Z) L += l[z] * e[z];
    }
    const float inv = L > 0.f ? gate / L : 0.f;
    for (int d = 4 * threadIdx.x; d < RP; d += 1024) {
      float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int z = 0; z < kLatFew; ++z) {
        if (z >= Z) break;
        const float* q = pp + (long)z * (RP + 2) + d;   // (a row is RP + 2 long: 8-byte loads)
        const float2 v = *reinterpret_cast<const float2*>(q), w = *reinterpret_cast<const float2*>(q + 2);
        s[0] += v.x * e[z];
        s[1] += v.y * e[z];
        s[2] += w.x * e[z];
        s[3] += w.y * e[z];
      }
      store_avg(p, orow + d, {s[0] * inv, s[1] * inv, s[2] * inv, s[3] * inv});
    }
    return;
  }
  for (int z = lane; z < Z; z += 64) M = fmaxf(M, pp[(long)z * (RP + 2) + RP]);
  M = wave_max(M);
  for (int z = lane; z < Z; z += 64) L += pp[(long)z * (RP + 2) + RP + 1] * __builtin_amdgcn_exp2f(pp[(long)z * (RP + 2) + RP] - M);
  L = wave_sum(L);
  const float inv = L > 0.f ? gate / L : 0.f;
  for (int d = 4 * threadIdx.x; d < RP; d += 1024) {
    float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int z = 0; z < Z; ++z) {
      const float* q = pp + (long)z * (RP + 2);
      const float2 v = *reinterpret_cast<const float2*>(q + d), w = *reinterpret_cast<const float2*>(q + d + 2);
      const float e = __builtin_amdgcn_exp2f(q[RP] - M);
      s[0] += v.x * e;
      s[1] += v.y * e;
      s[2] += w.x * e;
      s[3] += w.y * e;
    }
    store_avg(p, orow + d, {s[0] * inv, s[1] * inv, s[2] * inv, s[3] * inv});
  }
}

// ---- plain form: one workgroup per (row, head), keys in rounds of 256 (one per thread for the scores, all threads over the
// latent's columns for the average).  cu_q null: decode rows.
constexpr int kPlainDims = 8;   // latent columns per thread: RP <= 2048

template <typename T>
__global__ __launch_bounds__(256) void lat_plain_kernel(LatParams p, const int* __restrict__ cu_q, const int* __restrict__ ctx_lens, int nseq) {
  constexpr bool EXACT = sizeof(T) == 4;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  float* q = reinterpret_cast<float*>(smem);          // [KD]
  float* pw = q + p.KD;                                // [256]
  long* rows = reinterpret_cast<long*>(pw + 256);      // [256] element offsets of the cache rows
  __shared__ float red[4];
  const int row = blockIdx.x, head = blockIdx.y, tid = threadIdx.x;
  int b = row, qpos;
  if (cu_q) {
    for (b = 0; b < nseq - 1 && row >= cu_q[b + 1]; ++b) {}
    qpos = ctx_lens[b] - (cu_q[b + 1] - row);
  } else {
    qpos = ctx_lens[b] - 1;
  }
  T* orow = reinterpret_cast<T*>(p.out) + (long)row * p.os + (long)head * p.OH;
  if (qpos < 0) {
    for (int d = tid; d < p.OH; d += 256) El<T>::st(orow + d, 0.f);
    return;
  }
  const T* qrow = reinterpret_cast<const T*>(p.q) + (long)row * p.qs + (long)head * p.KD;
  for (int d = tid; d < p.KD; d += 256) q[d] = El<T>::ld(qrow + d) * p.scale;
  const int* bt = p.bt + (long)b * p.bt_stride;
  const T* cache = reinterpret_cast<const T*>(p.cache);
  float m = p.sink ? p.sink[head] : kNegBig, l = p.sink ? 1.f : 0.f;
  float acc[kPlainDims];
#pragma unroll
  for (int i = 0; i < kPlainDims; ++i) acc[i] = 0.f;
  for (int k0 = first_key(qpos, p.window); k0 <= qpos; k0 += 256) {
    const int n = min(256, qpos + 1 - k0);
    __syncthreads();   // q is there; the previous round's weights have been read
    float s = kNegBig;
    if (tid < n) {
      const int key = k0 + tid;
      const long off = ((long)bt[key / p.BS] * p.BS + key % p.BS) * p.KD;
      rows[tid] = off;
      const T* kr = cache + off;
      float a[4] = {0.f, 0.f, 0.f, 0.f};
      for (int d = 0; d < p.KD; d += 4)
#pragma unroll
        for (int e = 0; e < 4; ++e) a[e] += q[d + e] * El<T>::ld(kr + d + e);
      s = (a[0] + a[1]) + (a[2] + a[3]);
    }
    float mx = wave_max(s);
    if ((tid & 63) == 0) red[tid >> 6] = mx;
    __syncthreads();
    mx = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float mn = fmaxf(m, mx);
    const float alpha = EXACT ? expf(m - mn) : __expf(m - mn);
    const float w = tid < n ? (EXACT ? expf(s - mn) : __expf(s - mn)) : 0.f;
    pw[tid] = w;
    m = mn;
    l = l * alpha + block_sum<4>(w, red);   // (its barriers also publish pw and rows)
#pragma unroll
    for (int i = 0; i < kPlainDims; ++i) {
      const int d = tid + 256 * i;
      if (d < p.RP) {
        float v = acc[i] * alpha;
        for (int k = 0; k < n; ++k) v += pw[k] * El<T>::ld(cache + rows[k] + d);
        acc[i] = v;
      }
    }
  }
  const float inv = l > 0.f ? lat_gate<T>(p, row, head) / l : 0.f;
#pragma unroll
  for (int i = 0; i < kPlainDims; ++i) {
    const int d = tid + 256 * i;
    if (d < p.RP) {
      const float v = acc[i] * inv;
      El<T>::st(orow + d, v);
      if (p.OH > p.RP) El<T>::st(orow + p.RP + d, v - El<T>::ld(orow + d));   // (this thread's own store)
    }
  }
}

// ---- operands ------------------------------------------------------------------------------------------------------
struct PrepParams {
  const void* u;
  long us;
  int dq, qr;
  const float* wq;
  int dkv, R;
  const float* wkv;    // null: no cache row
  int rd;
  const float* freq;
  const int* positions;
  float eps;
  void* cache;
  const int* slots;
  int RP, KD;
  void* cq;
  long cqs;
  int adj;             // pairs (2 i, 2 i + 1) instead of (i, i + rd / 2)
  float mag;           // times cos and sin
};

// One workgroup per token: both root mean squares in one pass over the row, the normed query latent, the cache row.
template <typename T>
__global__ __launch_bounds__(256) void latent_prep_kernel(PrepParams p) {
  __shared__ float red[2][4];
  const long t = blockIdx.x;
  const int tid = threadIdx.x;
  const T* uq = reinterpret_cast<const T*>(p.u) + t * p.us + p.dq;
  const T* ukv = reinterpret_cast<const T*>(p.u) + t * p.us + p.dkv;
  float sq = 0.f, sk = 0.f;
  for (int c = tid; c < p.qr; c += 256) {
    const float v = El<T>::ld(uq + c);
    sq += v * v;
  }
  const int slot = p.wkv ? p.slots[t] : -1;
  if (p.wkv)
    for (int c = tid; c < p.R; c += 256) {
      const float v = El<T>::ld(ukv + c);
      sk += v * v;
    }
  sq = block_sum<4>(sq, red[0]);
  T* cq = reinterpret_cast<T*>(p.cq) + t * p.cqs;
  const float iq = 1.f / sqrtf(sq / (float)p.qr + p.eps);
  for (int c = tid; c < p.qr; c += 256) El<T>::st(cq + c, El<T>::ld(uq + c) * iq * p.wq[c]);
  if (slot < 0) return;   // the same for the whole workgroup
  sk = block_sum<4>(sk, red[1]);
  const float ik = 1.f / sqrtf(sk / (float)p.R + p.eps);
  T* row = reinterpret_cast<T*>(p.cache) + (long)slot * p.KD;   // pages are contiguous: slot = block * BS + offset
  for (int c = tid; c < p.RP; c += 256) El<T>::st(row + c, c < p.R ? El<T>::ld(ukv + c) * ik * p.wkv[c] : 0.f);
  const int half = p.rd / 2;
  const float pos = (float)p.positions[t];
  for (int i = tid; i < half; i += 256) {
    float sn, cs;
    sincosf(pos * p.freq[i], &sn, &cs);
    cs *= p.mag;
    sn *= p.mag;
    const int ia = p.adj ? 2 * i : i, ib = p.adj ? 2 * i + 1 : half + i;
    const float a = El<T>::ld(ukv + p.R + ia), b = El<T>::ld(ukv + p.R + ib);
    El<T>::st(row + p.RP + ia, a * cs - b * sn);
    El<T>::st(row + p.RP + ib, b * cs + a * sn);
  }
  for (int c = p.RP + p.rd + tid; c < p.KD; c += 256) El<T>::st(row + c, 0.f);
}

bool mfma_shape(int RP, int KD) {
  const int rdp = KD - RP;
  return (RP == 128 || RP == 256 || RP == 512) && (rdp == 64 || rdp == 128);
}

#define LK_LAT_DISPATCH(FN, ...)                                  \
  switch (p.RP * 1000 + p.KD - p.RP) {                            \
    case 128064: return FN<128, 64>(__VA_ARGS__);                 \
    case 128128: return FN<128, 128>(__VA_ARGS__);                \
    case 256064: return FN<256, 64>(__VA_ARGS__);                 \
    case 256128: return FN<256, 128>(__VA_ARGS__);                \
    case 512064: return FN<512, 64>(__VA_ARGS__);                 \
    case 512128: return FN<512, 128>(__VA_ARGS__);                \
    default: return -1;                                           \
  }

template <int RP, int RDP>
int launch_prefill(const LatParams& p, const int* cu_q, const int* ctx, int nseq, long rows, hipStream_t st) {
  constexpr size_t lds = 2 * 64 * (RP + RDP);
  const int NQ = (in_pairs<RP, RDP>() ? kPairCols : kPreCols) / p.HC;
  const long tiles = (rows + NQ - 1) / NQ + nseq;   // every sequence ends with at most one partial tile
  const dim3 grid((unsigned)tiles, (unsigned)((p.H + p.HC - 1) / p.HC));
  if constexpr (in_pairs<RP, RDP>()) {
    LK_SET_MAX_LDS((lat_prefill_pair_kernel<RP, RDP>), pair_lds(RP + RDP));
    lat_prefill_pair_kernel<RP, RDP><<<grid, 64 * kPairWaves, pair_lds(RP + RDP), st>>>(p, cu_q, ctx, nseq);
  } else {
    LK_SET_MAX_LDS((lat_prefill_kernel<RP, RDP>), lds);
    lat_prefill_kernel<RP, RDP><<<grid, pre_waves<RP>() * 64, lds, st>>>(p, cu_q, ctx, nseq);
  }
  LK_CHECK_LAUNCH();
  return 0;
}

template <int RP, int RDP>
int launch_decode(const LatParams& p, const int* ctx, int B, int Z, float* part, hipStream_t st) {
  constexpr size_t lds = 4 * 64 * (RP + RDP);
  LK_SET_MAX_LDS((lat_decode_kernel<RP, RDP>), lds);
  lat_decode_kernel<RP, RDP><<<dim3((unsigned)B, (unsigned)((p.H + p.HC - 1) / p.HC), (unsigned)Z), 256, lds, st>>>(p, ctx, Z, part);
  LK_CHECK_LAUNCH();
  if (Z > 1) {
    lat_reduce_kernel<<<dim3((unsigned)B, (unsigned)p.H), 256, 0, st>>>(p, part, Z);
    LK_CHECK_LAUNCH();
  }
  return 0;
}

int run_prefill(const LatParams& p, const int* cu_q, const int* ctx, int nseq, long rows, hipStream_t st) {
  LK_LAT_DISPATCH(launch_prefill, p, cu_q, ctx, nseq, rows, st)
}

int run_decode(const LatParams& p, const int* ctx, int B, int Z, float* part, hipStream_t st) {
  LK_LAT_DISPATCH(launch_decode, p, ctx, B, Z, part, st)
}

template <typename T>
int run_plain(const LatParams& p, const int* cu_q, const int* ctx, int nseq, long rows, hipStream_t st) {
  const size_t lds = sizeof(float) * (p.KD + 256) + sizeof(long) * 256;
  if (p.RP > 256 * kPlainDims || lds > 64 * 1024 || rows > 2147483647L) return -1;
  lat_plain_kernel<T><<<dim3((unsigned)rows, (unsigned)p.H), 256, lds, st>>>(p, cu_q, ctx, nseq);
  LK_CHECK_LAUNCH();
  return 0;
}

bool make_params(LatParams& p, const void* q, long qs, const void* cache, const int* bt, int bt_stride, int BS, int H, int KD, int RP, int window,
                 float scale, const float* sink, const void* gate, long gs, void* out, long os, int OH, int esz) {
  p.gate = gate; p.gs = gs; p.OH = OH;
  p.q = q; p.qs = qs; p.cache = cache; p.bt = bt; p.bt_stride = bt_stride; p.BS = BS; p.H = H; p.KD = KD; p.RP = RP; p.window = window;
  p.scale = scale; p.sink = sink; p.out = out; p.os = os;
  const int blocks = (H + 15) / 16;
  p.HC = blocks > 0 ? (H + blocks - 1) / blocks : 1;
  const auto a16 = [](const void* x) { return reinterpret_cast<uintptr_t>(x) % 16 == 0; };
  return H >= 1 && H <= 65535 && BS >= 16 && BS % 16 == 0 && RP >= 16 && KD > RP && KD % 64 == 0 && RP % 64 == 0 && window >= 0 && (OH == RP || OH == 2 * RP) && a16(q) &&
         a16(cache) && a16(out) && qs % (16 / esz) == 0 && os % (16 / esz) == 0;
}

}  // namespace

int lk_latent_attn_prefill(const void* q, long qs, const void* cache, const int* bt, int bt_stride, const int* cu_q, const int* ctx_lens, int nseq,
                           long rows, int BS, int H, int KD, int RP, int window, float scale, const float* sink, const void* gate, long gs,
                           void* out, long os, int OH, int esz, hipStream_t st) {
  if (rows <= 0 || nseq <= 0) return 0;
  LatParams p;
  if (!make_params(p, q, qs, cache, bt, bt_stride, BS, H, KD, RP, window, scale, sink, gate, gs, out, os, OH, esz)) return -1;
  if (esz == 2 && mfma_shape(RP, KD)) return run_prefill(p, cu_q, ctx_lens, nseq, rows, st);
  return esz == 2 ? run_plain<bf16_t>(p, cu_q, ctx_lens, nseq, rows, st) : run_plain<float>(p, cu_q, ctx_lens, nseq, rows, st);
}

int lk_latent_attn_decode(const void* q, long qs, const void* cache, const int* bt, int bt_stride, const int* ctx_lens, int B, int Z, int BS, int H,
                          int KD, int RP, int window, float scale, const float* sink, const void* gate, long gs, void* out, long os,
                          int OH, float* part, int esz, hipStream_t st) {
  if (B <= 0) return 0;
  LatParams p;
  if (!make_params(p, q, qs, cache, bt, bt_stride, BS, H, KD, RP, window, scale, sink, gate, gs, out, os, OH, esz)) return -1;
  if (esz == 2 && mfma_shape(RP, KD)) {
    if (Z < 1 || Z > 65535 || (Z > 1 && !part)) return -1;
    return run_decode(p, ctx_lens, B, Z, part, st);
  }
  return esz == 2 ? run_plain<bf16_t>(p, nullptr, ctx_lens, B, B, st) : run_plain<float>(p, nullptr, ctx_lens, B, B, st);
}

int lk_latent_prep(const void* u, long us, int dq, int qr, const float* wq, int dkv, int R, const float* wkv, int rd, const float* freq,
                   const int* positions, float eps, void* cache, const int* slots, int RP, int KD, void* cq, long cqs, long rows, int adj, float mag,
                   int esz, hipStream_t st) {
  if (rows <= 0) return 0;
  if (qr < 1 || !wq || (wkv && (R < 1 || R > RP || rd < 0 || rd % 2 || RP + rd > KD || !cache || !slots || (rd > 0 && !freq)))) return -1;
  PrepParams p;
  p.u = u; p.us = us; p.dq = dq; p.qr = qr; p.wq = wq; p.dkv = dkv; p.R = R; p.wkv = wkv; p.rd = rd; p.freq = freq; p.positions = positions;
  p.eps = eps; p.cache = cache; p.slots = slots; p.RP = RP; p.KD = KD; p.cq = cq; p.cqs = cqs; p.adj = adj; p.mag = mag;
  if (esz == 2) latent_prep_kernel<bf16_t><<<(unsigned)rows, 256, 0, st>>>(p);
  else latent_prep_kernel<float><<<(unsigned)rows, 256, 0, st>>>(p);
  LK_CHECK_LAUNCH();
  return 0;
}
