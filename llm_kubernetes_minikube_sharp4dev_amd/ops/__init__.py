"""Kernel entry points.  GPU tensors -> hand-written gfx950 HIP kernels (``_C``);
CPU tensors -> fp32 torch references (``reference``).  See ``_ext`` for the policy.

Layouts are documented in :mod:`.reference`.
"""
from __future__ import annotations

import logging
import math
import os
from typing import Optional, Sequence

import numpy as np
import torch

from . import reference as ref
from ._ext import available, force_reference, lib, use_hip  # noqa: F401
from .mixers import (conv_silu, embed_norm, embed_pos, gated_group_rmsnorm, linear_swiglu_any, sig_decode_splits,  # noqa: F401
                     sig_prefill_tiles, sigattn_supported, sigmoid_attention_decode, sigmoid_attention_prefill,
                     softcap, ssm_scan, stream_rmsnorm, unitnorm_kv_write, embed_stream, stream_layernorm, gelu_tanh_mul,
                     dual_rmsnorm_mean, normrope_kv_write, sink_attention_prefill, sink_attention_decode, mask_first_key,
                     pooled_blocks_seen, stream_sandwich_layernorm, MASK_CAUSAL, MASK_CHUNK, MASK_WINDOW, SIG_TILE_ROWS)
from .window import moe_route, moe_routes, moe_skips_rows, pool_kv_write, rms_cols, rot_kv_write, linear_table_experts, run_experts, stream_gated_norm, stream_gated_norm_conv, table_experts  # noqa: F401
from .routed import clamped_glu, routed_experts, router_topk, sigmoid_mul_, silu_, stream_parallel_norm  # noqa: F401
from .hyper import (GROUP_MAX, GROUP_TOP2, MAX_STREAMS, SCORE_SIGMOID, SCORE_SOFTMAX, gate_proj, relu_sq_, router_choice,  # noqa: F401
                    stream_hyper_norm)
from .latent import (head_linear, latent_attention_decode, latent_attention_prefill, latent_decode_splits, latent_prep,  # noqa: F401
                     latent_query, latent_query_rot, latent_row)
from .diff import (diff_attention_decode, diff_attention_prefill, diff_attention_supported, diff_prefill_rows, qkv_file, row_tiles,  # noqa: F401
                   tile_attention_prefill, tile_attention_rows, tile_attention_supported)
from .head_delta import head_delta, head_delta_supported  # noqa: F401
from .mlstm import mlstm_scan, mlstm_state, mlstm_supported  # noqa: F401
from .delta import (delta_scan, delta_scan_supported, gated_delta_prep, general_delta_prep, head_norm_gate, tanh_,  # noqa: F401
                    GATE_SIGMOID, GATE_SILU)

__all__ = [
    "rmsnorm", "layernorm", "embed_layernorm", "silu_mul", "gelu_", "relu_", "rope_kv_",
    "kv_write", "paged_decode", "flash_prefill", "prefill_tiles", "knn_topk", "knn_merge",
    "pool_normalize", "row_norms", "select_tokens", "repeat_penalty_", "sample", "linear", "linear_swiglu",
    "decode_splits", "rope_cos_sin", "argmax_key", "key_to_id", "tune_gemm", "tune_decode", "gemm", "linear_add_rmsnorm", "linear_rope_kv",
    "prefill_chain_ok", "linear_resid", "linear_qkv_fused", "linear_swiglu_scaled", "embed_rows", "scatter_ids",
    "gather_rows",
]

rope_cos_sin = ref.rope_cos_sin
DECODE_MAX_SPLIT = 2048  # csrc/attn_decode.hip kMaxSplit


def rmsnorm(x, w, eps: float, residual: Optional[torch.Tensor] = None, out=None):
    """out = RMSNorm(x [+ residual]) * w; if ``residual`` is given it is updated in
    place to ``x + residual`` (fused add+norm of the pre-norm decoder block)."""
    if use_hip(x):
        return lib().rmsnorm(x, w, eps, residual, out)
    y = ref.rmsnorm(x, w, eps, residual)
    if out is not None:
        out.copy_(y)
        return out
    return y


def layernorm(x, w, b, eps: float, residual=None, write_residual: bool = False):
    if use_hip(x):
        return lib().layernorm(x, w, b, eps, residual, write_residual)
    return ref.layernorm(x, w, b, eps, residual, write_residual)


def embed_layernorm(ids, pos_ids, type_ids, tok, pos, typ, w, b, eps: float):
    if use_hip(tok):
        return lib().embed_layernorm(ids, pos_ids, type_ids, tok, pos, typ, w, b, eps)
    return ref.embed_layernorm(ids, pos_ids, type_ids, tok, pos, typ, w, b, eps)


def silu_mul(x, out=None):
    if use_hip(x):
        return lib().silu_mul(x, out)
    y = ref.silu_mul(x)
    if out is not None:
        out.copy_(y)
        return out
    return y


def gelu_(x, bias=None, approximate: str = "none"):
    kind = 1 if approximate == "tanh" else 0
    if use_hip(x):
        lib().activation_(x, bias, kind)
        return x
    return ref.activation_(x, bias, kind)


def relu_(x, bias=None):
    if use_hip(x):
        lib().activation_(x, bias, 2)
        return x
    return ref.activation_(x, bias, 2)


def rope_kv_(qkv, positions, cos_sin, Hq: int, Hkv: int, D: int, k_cache=None, v_cache=None,
             slots=None, neox: bool = True, write_k_inplace: bool = False):
    if use_hip(qkv):
        lib().rope_kv_(qkv, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots, neox,
                       write_k_inplace)
        return qkv
    return ref.rope_kv_(qkv, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots, neox,
                        write_k_inplace)


def kv_write(k, v, k_cache, v_cache, slots):
    if use_hip(k):
        return lib().kv_write(k, v, k_cache, v_cache, slots)
    return ref.kv_write(k, v, k_cache, v_cache, slots)


# keys per decode workgroup once the batch alone fills the CUs (B * Hkv >= 512); LK_DECODE_SPLIT
# overrides it (A/B knob: three 256-thread workgroups per CU make 768 slots, so ~1.1-1.5 rounds
# of unsplit workgroups at the serving batch leave part of the last round idle).  2048: the RAG
# bench's ~1k-key rows stay in one split, so no step launches the split-merge kernel (same box,
# interleaved: mixed-step GPU time 9.21 / 9.18 vs 9.25 / 9.25 s, 108.2 / 108.3 vs 108.2 / 107.8 q/s)
DECODE_SPLIT_LARGE = int(os.environ.get("LK_DECODE_SPLIT", "2048"))
# keys per decode workgroup below 32 (sequence, kv head) pairs (batch 1: 8 kv heads)
DECODE_SPLIT_SMALL = int(os.environ.get("LK_DECODE_SPLIT_SMALL", "128"))


def decode_split_size(B: int, Hkv: int) -> int:
    """Keys per decode workgroup (mirrors lk_decode_split_size): small batches split the
    context finer so 256 CUs stay busy; static per (B, Hkv) for hipGraph capture."""
    bh = B * Hkv
    return DECODE_SPLIT_LARGE if bh >= 512 else 512 if bh >= 128 else 256 if bh >= 32 else DECODE_SPLIT_SMALL


def decode_splits(max_context: int, split: int) -> int:
    return max(1, (int(max_context) + split - 1) // split)


# Split decode: the last split workgroup of each (sequence, kv head) merges the partials
# itself (csrc/attn_decode.hip merge_splits) instead of a decode_reduce launch after the kernel.
# Needs one zero-initialised int32 ticket per (sequence, kv head), reset by its last taker: a
# per-device buffer made before any graph capture.  Used where the batch fills the CUs unsplit
# (B x Hkv >= 512, 2048-key workgroups): rows of <= 2048 keys write their output directly and the
# reduce launch (which round 5 made on every layer of every step, to find nothing to merge) is
# gone.  At small batches, where every row splits, the separate reduce kernel measured faster
# (batch 1, same box, twice each: decode step 3.74 / 3.73 ms fused vs 3.65 / 3.61 ms,
# profiles/r6_fused_merge/): the split workgroups' write-through partials and ticket sit on the
# critical path.  LK_DECODE_FUSED_REDUCE=0: never, =2: always.
DECODE_FUSED_REDUCE = int(os.environ.get("LK_DECODE_FUSED_REDUCE", "1") or 0)
_DECODE_TICKETS: dict = {}


def decode_tickets(device, n: int):
    device = torch.device(device)
    key = device.index if device.index is not None else torch.cuda.current_device()
    t = _DECODE_TICKETS.get(key)
    if t is None or t.numel() < n:
        t = _DECODE_TICKETS[key] = torch.zeros(max(n, 1 << 16), dtype=torch.int32, device=device)
    return t


def paged_decode(q, k_cache, v_cache, block_tables, ctx_lens, scale: float, max_splits: Optional[int] = None,
                 part_o=None, part_ml=None, out=None, split: Optional[int] = None, k_start=None, prefix=None,
                 reduce: bool = True, own_blocks: bool = False):
    """q [B, Hq, D] -> [B, Hq, D].  ``split`` keys per workgroup (default from
    :func:`decode_split_size`), ``max_splits`` = splits covering the block-table width —
    both static, so the launch is hipGraph-capturable.

    Cascade: ``k_start`` (device int32 [1]) keys are a prefix shared by every row whose
    attention was computed once for the batch by :func:`flash_prefill` in partial mode
    into ``prefix`` = (o [B, Hq, D], ml [B, Hq, 2]); this call attends the rest and
    merges (the CPU reference attends everything directly).  ``reduce=False`` (GPU, no
    tickets): rows with more than one split keep their partials in ``part_o`` / ``part_ml`` for
    the consumer to merge (:func:`ws_pro` kind 2).  ``own_blocks``: no cache block belongs to two rows (their
    reads then pass the caches by; without it every split looks whether its rows are shared; the result is the same)."""
    if use_hip(q):
        BS = k_cache.shape[2]
        if split is None:
            split = max(decode_split_size(q.shape[0], k_cache.shape[1]), BS)
        if max_splits is None:
            max_splits = decode_splits(block_tables.shape[1] * BS, split)
        pp_o, pp_ml = prefix if prefix is not None else (None, None)
        bh = q.shape[0] * k_cache.shape[1]
        fused = reduce and (DECODE_FUSED_REDUCE == 2 or (DECODE_FUSED_REDUCE == 1 and bh >= 512))
        tickets = decode_tickets(q.device, bh) if fused else None
        return lib().paged_decode(q, k_cache, v_cache, block_tables, ctx_lens, max_splits, split, scale,
                                  part_o, part_ml, out, k_start, pp_o, pp_ml, tickets, reduce, own_blocks)
    y = ref.paged_decode(q, k_cache, v_cache, block_tables, ctx_lens, scale)
    if out is not None:
        out.copy_(y)
        return out
    return y


def prefill_rows_per_tile(G: int, D: int = 128) -> int:
    """Query rows per flash-prefill tile: the HIP library's choice for (GQA group, head dim)
    (8-wave 64-row workgroups for G >= 4, D >= 64 under LK_PREFILL_WAVES=8), else 32 / 4-wave."""
    try:
        return int(lib().prefill_rows_per_tile(G, D))
    except Exception:  # no extension (CPU): the tiles only matter to the HIP kernel
        return 32 if G >= 4 else 32 * (4 // G)


def prefill_tiles(q_lens: Sequence[int], ctx_lens: Sequence[int], G: int, causal: bool, D: int = 128):
    """Query tiles (seq, q0) for the flash kernel, heaviest first (LPT scheduling:
    with causal masking a tile's cost grows with the keys it sees)."""
    qb = prefill_rows_per_tile(G, D)
    seqs, q0s, cost = [], [], []
    for b, (ql, cl) in enumerate(zip(q_lens, ctx_lens)):
        past = cl - ql
        for q0 in range(0, ql, qb):
            seqs.append(b)
            q0s.append(q0)
            cost.append(min(cl, past + q0 + qb) if causal else cl)
    order = np.argsort(-np.asarray(cost, dtype=np.int64), kind="stable")
    return (np.asarray(seqs, dtype=np.int32)[order], np.asarray(q0s, dtype=np.int32)[order])


def device_tiles(q_lens: Sequence[int], ctx_lens: Sequence[int], G: int, causal: bool, D: int, device):
    """:func:`prefill_tiles` on the device, in one copy: what a forward pass hands to all of its layers."""
    both = torch.from_numpy(np.stack(prefill_tiles(q_lens, ctx_lens, G, causal, D))).to(device, non_blocking=True)
    return both[0], both[1]


def flash_prefill(q, k, v, cu_q, Hq: int, Hkv: int, D: int, scale: float, causal: bool,
                  block_tables=None, ctx_lens=None, q_lens_cpu=None, ctx_lens_cpu=None,
                  tiles=None, out=None, part=None, q_past=None):
    """Varlen flash attention.  Paged when ``block_tables`` is given (K/V caches
    ``[NB, Hkv, BS, D]``), else dense K/V rows ``[T, >=Hkv*D]`` (encoder).
    ``part`` = (o f32 [T, Hq, D], ml f32 [T, Hq, 2]): write unnormalised partials for a
    cascade / context-parallel merge instead of ``out`` (GPU only; ml = (running max, sum) in
    the log2 domain).  ``q_past`` (int32 [B], GPU only): position of each sequence's first
    query relative to its first key for the causal mask (a context-parallel key shard), instead
    of ctx_len - q_len.

    ``q_lens_cpu`` / ``ctx_lens_cpu``: host copies of the lengths (the scheduler has
    them), used to build the tile list without a device sync."""
    if use_hip(q):
        if tiles is None:
            if q_lens_cpu is None:
                cu = cu_q.cpu().tolist()
                q_lens_cpu = [cu[i + 1] - cu[i] for i in range(len(cu) - 1)]
            if ctx_lens_cpu is None:
                ctx_lens_cpu = ctx_lens.cpu().tolist() if ctx_lens is not None else list(q_lens_cpu)
            if block_tables is not None:
                BS = k.shape[2]
                need = max((int(c) + BS - 1) // BS for c in ctx_lens_cpu) if ctx_lens_cpu else 0
                if need > block_tables.shape[1]:
                    raise ValueError("block table too narrow for the context lengths")
            tiles = device_tiles(q_lens_cpu, ctx_lens_cpu, Hq // Hkv, causal, D, q.device)
        pp_o, pp_ml = part if part is not None else (None, None)
        if out is not None and part is None and (out.data_ptr() % 16 or out.stride(0) % 8):
            # the kernel's output rows leave as 16-byte stores: stage a misaligned view
            y = lib().flash_prefill(q, k, v, block_tables, cu_q, ctx_lens, tiles[0], tiles[1], Hq,
                                    Hkv, D, scale, causal, None, None, None, q_past)
            out[:, : Hq * D].copy_(y)
            return out
        return lib().flash_prefill(q, k, v, block_tables, cu_q, ctx_lens, tiles[0], tiles[1], Hq,
                                   Hkv, D, scale, causal, out, pp_o, pp_ml, q_past)
    if q_past is not None:
        raise NotImplementedError("q_past: GPU kernel only")
    y = ref.flash_prefill(q, k, v, block_tables, cu_q, ctx_lens, Hq, Hkv, D, scale, causal)
    if out is not None:
        out[:, : Hq * D].copy_(y)
        return out
    return y


def knn_topk(corpus, cnorm, queries, qnorm, K: int):
    """Cosine top-K (scores f32 [nq,K], indices int32 [nq,K]; -1 pads)."""
    if use_hip(corpus):
        s, i = lib().knn_topk(corpus, cnorm, queries, qnorm, K)
        return s, i
    return ref.knn_topk(corpus, cnorm, queries, qnorm, K)


def knn_packed(corpus, cnorm, queries, K: int):
    """:func:`knn_topk` of few queries on the GPU with both results in one int32 tensor [2, nq, K] (the scores' bits, then
    the indices).  None where the one-pass search does not take the shape."""
    if not (use_hip(corpus) and queries.is_cuda and 1 <= K <= 64 and queries.shape[0] > 0):
        return None
    r = lib().knn_packed(corpus, cnorm, queries, K)
    return r if r.numel() else None


def knn_hits(corpus, cnorm, queries, K: int):
    """:func:`knn_packed` into pinned memory as a handle: ``query()`` whether the hits have arrived, ``synchronize()`` waits for them
    alone (no event behind the kernels), ``rows(k)`` then the (index, score) pairs of each query.  None where the one-pass search does
    not take the shape."""
    if not (use_hip(corpus) and queries.is_cuda and 1 <= K <= 64 and queries.shape[0] > 0):
        return None
    return lib().knn_hits(corpus, cnorm, queries, K)


def knn_merge(cand_s, cand_i, K: int):
    if use_hip(cand_s):
        return tuple(lib().knn_merge(cand_s.contiguous(), cand_i.contiguous(), K))
    nq = cand_s.shape[0]
    out_s = torch.full((nq, K), float("-inf"))
    out_i = torch.full((nq, K), -1, dtype=torch.int32)
    for r in range(nq):
        pairs = [(float(s), int(i)) for s, i in zip(cand_s[r].tolist(), cand_i[r].tolist()) if int(i) >= 0]
        pairs.sort(key=lambda p: (-p[0], p[1]))
        for j, (s, i) in enumerate(pairs[:K]):
            out_s[r, j] = s
            out_i[r, j] = i
    return out_s, out_i


def pool_normalize(hidden, cu, mode: int, normalize: bool = True, out=None):
    """Pooled (mean / CLS), L2-normalised sentence vectors; ``out``: destination rows [B, H]
    (f32 or bf16; the kernel writes them directly), default a new f32 [B, H]."""
    if use_hip(hidden):
        return lib().pool_normalize(hidden, cu, mode, normalize, out)
    y = ref.pool_normalize(hidden, cu, mode, normalize)
    if out is not None:
        out.copy_(y)
        return out
    return y


def row_norms(x):
    if use_hip(x):
        return lib().row_norms(x.contiguous())
    return ref.row_norms(x)


def select_tokens(logits, temps=None, seed: int = 0, step: int = 0, out=None):
    if use_hip(logits):
        return lib().select_tokens(logits, temps, int(seed) & ((1 << 63) - 1), int(step), out)
    return ref.select_tokens(logits, temps, seed, step)


def argmax_key(logits, vocab_lo: int = 0):
    """Per row an order-preserving int64 key of (max value, vocab_lo + first argmax): the larger
    key is the larger value, then the LOWER id (torch.argmax's tie order), so the max of the
    keys gathered from the vocab shards picks the global greedy token (parallel/tp.py)."""
    if use_hip(logits):
        return lib().argmax_key(logits, int(vocab_lo))
    return ref.argmax_key(logits, vocab_lo)


def key_to_id(keys):
    """Global ids from [W, R] gathered argmax keys (max over W), int32 [R]; a [R] key row
    decodes directly."""
    if keys.dim() == 1:
        keys = keys[None]
    if use_hip(keys):
        return lib().keys_to_ids(keys.contiguous())
    return ref.keys_to_ids(keys)


def sample(logits, prm, hist, hist_len, seed: int = 0, out=None):
    """Ollama-default sampling of every row (repeat penalty from the device history ring,
    top-k, top-p, temperature; greedy rows = argmax); appends the tokens to the ring."""
    if use_hip(logits):
        return lib().sample(logits, prm, hist, hist_len, int(seed) & ((1 << 63) - 1), out)
    return ref.sample(logits, prm, hist, hist_len, seed)


def repeat_penalty_(logits, window, penalty):
    if use_hip(logits):
        lib().repeat_penalty_(logits, window, penalty)
        return logits
    return ref.repeat_penalty_(logits, window, penalty)


# Decode-regime GEMMs (csrc/skinny_gemm.hip) vs the library GEMM, from the MI355X
# sweeps in profiles/r1_skinny_gemm.md and profiles/r1_ws_sweep.md:
#  * M <= 256: the LDS-DMA weight-streaming kernel: 1.2-2.3x hipBLASLt on every
#    Llama projection (QKV / O / down; gate_up+SwiGLU fused up to M = 160), and its
#    split-K reduction fused into the consumer (RMSNorm+residual, RoPE+KV write);
#  * the LM head (N >= 65536) at M <= 16: the fragment-load kernel (weights straight to
#    VGPRs, split-K); larger M: the prefill GEMM.
# The fragment-load kernel also served every projection at M <= 16 until round 2; the
# fused weight-streaming path beat it end to end at every small batch (bench.py --batch
# 1/2/4/8 on MI355X: p50 227 -> 201, 235 -> 207, 252 -> 224, 292 -> 259 ms), so
# LK_SKINNY_MAX_M now defaults to 0.
SKINNY_MAX_M = int(os.environ.get("LK_SKINNY_MAX_M", "0"))
LM_HEAD_SKINNY_MAX_M = 16
# LM head (N >= 65536) at 16 < M <= 256: weight-streaming kernel (1) or the prefill GEMM (0)
WS_LM_HEAD = os.environ.get("LK_WS_LM_HEAD", "0") == "1"
WS_MAX_M = int(os.environ.get("LK_WS_MAX_M", "256"))
WS_SWIGLU_MAX_M = 160
# 256 rows of X and a tile's of W within 32-bit offsets (csrc/skinny_gemm.hip ws_too_far); beyond, the fragment-load kernel
WS_MAX_K = 8_000_000


# Measured per-shape choice between the weight-streaming kernel and the prefill GEMM for
# decode batches (``tune_decode``, cold weights, at engine start): the static rule below is
# wrong in both directions on some shapes (benchmarks/decode_route.py on MI355X,
# profiles/r3_decode_route/: the 70B TP=8 gate_up shard at M 192-256 ran the prefill GEMM at
# 0.35x of the ws kernel; the 70B QKV at M 160-256 ran ws at 0.79-0.90x of the GEMM).
# {(M bucket, N, K, swiglu): "ws" | "gemm"}; buckets are the tuned M values, a batch uses the
# smallest bucket >= M.
_DECODE_TABLE: dict = {}
DECODE_TUNE_MS = (32, 64, 96, 128, 160, 192, 224, 256)


def _decode_bucket(M: int) -> Optional[int]:
    for b in DECODE_TUNE_MS:
        if M <= b:
            return b
    return None


# Few rows (csrc/rows_gemm.hip, one launch with any epilogue) or the kernels with larger tiles.  A workgroup of the few-row
# kernel reads 16 (``wide`` True: 32, 2: 64) columns of W -- SwiGLU 2 x 16 or 2 x 32 -- and 16 to 64 rows of X, so its time is
#   2.1 us + rounds of workgroups (one per CU, the 8 XCDs alike) x (their bytes / 58 KB/us + 1 us),
# and not below 2 us and W at 4.9 TB/s, 0.3 of it again for each further row tile (a weight of more than 96 MB, which no L2 keeps, 0.9 for
# the second): within 10 % of 13,000 launches (30 shapes of W, 17 - 1,024 rows, all forms), GELU 0.3 us per round.  64 columns up to 64 rows only
# from N 3072 on: below, the narrower forms fill the chip in one round.  The other side: the weight-streaming kernel (``_ws_cost``) where
# it takes the step, else the prefill tiles (``_tiled_cost``; the choice is the tiles' where they come within 5 % and with SwiGLU, whose tiles
# take longer than that estimate, the few-row kernel's up to 10 % more).  Measured in hipGraphs, weights cold, few-row / other (us):
#    64 x  2048 x 2048  6.0 / 11.6    256 x 2048 x 2048  9.1 / 20.0    768 x 2048 x 2048 18.1 / 27.9     64 x 2048 x 5632 12.1 / 15.1
#    64 x 10496 x 2048 14.4 / 19.3    128 x 4096 x 4096 16.1 / 19.4    192 x 4096 x 4096 18.1 / 21.6    512 x 2048 x 5632 28.3 / 43.8
#   128 x 16384 x 1024 16.1 / 13.2    192 x 16384 x 1024 21.7 / 15.4   768 x 3072 x 768 15.7 / 11.8      65 x 8192 x 8192 52.8 / 42.0
#   SwiGLU: 64 x 11264 x 2048 14.6 / 18.9   192 x 4096 x 5632 26.2 / 97   400 x 6144 x 768 17.6 / 12.8   96 x 32768 x 1024 27.2 / 18.1
#   bias:   19 x  768 x  768  3.0 / 15.6    512 x 2304 x 768 11.4 / 18.0   400 x 576 x 1152 6.4 / 21.3   1000 x 3072 x 768 (GELU) 18.3 / 14.5
# Over 1,200 of them (M x N x K and epilogue) the picks take 0.4 - 1.0 % more than the best of all forms and kernels, where a rule by bytes per CU
# alone took 3.8 % more and up to 1.6 times as long as the other side.
# Widths that neither tiles (N no multiple of 192 or 256) go to the vendor's kernels, which split K for narrow outputs: fitted to
# within 25 % for N 48 - 11,280, K 256 - 8,192, 17 - 1,024 rows, and taken 5 % lower, since an even choice is worth nothing (few-row / vendor):
#    64 x  400 x 1024  3.3 / 6.7      64 x 2064 x 1024  5.5 / 8.8     512 x   48 x 8192 24.9 / 9.1     400 x 2064 x 1024 17.4 / 9.4
# (past K 8192 more than 16 rows of X do not stay in L2.)  Where the streaming kernel's sum rides in its consumer
# (linear_add_rmsnorm, linear_rope_kv) the two are level at decode sizes, and those stay as they are.
ROWS_MAX_M = 1024
_ROWS_RULE: dict = {}


def _ws_cost(M: int, N: int, K: int, swiglu: bool) -> float:
    """us of the weight-streaming kernel: 3.8 ns for each of a workgroup's columns and 2.5 ns for each row per 64 of K, 6 us for each
    further round of workgroups, the weight at 6.4 TB/s at least, and the sum of its parts of K behind it: within 20 % of 510 products
    of 1 - 256 rows (32 shapes, 1024 - 128256 x 768 - 14336).  Given on the scale of the few-row kernel's estimate, which lies 10 % above its
    own times, 16 % up to 64 rows and 25 % up to 16: over 1,100 products (4 - 160 rows, N 256 - 23040, K 512 - 8192) the picks of the two
    take 0.4 % more than the better one, 20 % at most, and 28 of them more than 5 %."""
    def plan(bn):   # (filled share of the CUs, parts of K), as csrc/skinny_gemm.hip lays a launch out
        cols, per = (N // 2, bn // 2) if swiglu else (N, bn)
        if cols % per:
            return -1.0, 1
        s = 1
        while cols // per * s * 2 <= 256 and K % (s * 128) == 0 and K // (s * 2) >= 1024:
            s *= 2
        return cols // per * s / (256 * -(-cols // per * s // 256)), s

    full, half, mid = plan(128), plan(64), (-1.0, 1) if swiglu else plan(96)
    whole = half[0] == full[0] and half[1] == 1 < full[1] and (K <= 3072 or (K <= 4096 and M <= 128))   # 64 columns of all of K
    (fill, parts), bn = (full, 128) if full[0] >= 0.7 or (0 <= full[0] and half[0] <= full[0] and not whole) else (half, 64)
    if mid[0] > fill + 1e-9:
        parts, bn = mid[1], 96
    rounds = -(-(N // bn * parts) // 256)
    chain = 3.0 + rounds * (K / parts) / 64 * (0.0038 * bn + 0.0025 * 64 * -(-M // 64) - 0.16) + 6.3 * (rounds - 1)
    # (of few workgroups the sum's launch is not hidden: 56 x 1280 x 6400 14.7 us, 11.9 without the last term, 12.3 on the few-row kernel)
    us = max(chain, 3.3 + N * K * 2 / 6.35e6) + (2.0 + 2.4e-6 * parts * M * N + (N // bn * parts <= 128) if parts > 1 else 0)
    return us * _few_scale(M)


def _few_scale(M: int) -> float:
    """How far the few-row kernel's estimate lies above its times."""
    return 1.1 if M > 64 else 1.16 if M > 16 else 1.25


def _rows_cost(M: int, N: int, K: int, epi: int, products: int = 1):
    """(us of the few-row kernel, its ``wide`` argument, us of the other kernels), or None where it does not take the shape; of one
    product or of ``products`` like it, in one launch or one after the other."""
    mt = (M + 15) // 16   # 16-row tiles of X
    key = (mt, N, K, epi, products)
    if key in _ROWS_RULE:
        return _ROWS_RULE[key]
    est = None
    if 1 <= M <= ROWS_MAX_M and (K <= 8192 or mt == 1) and lib().rows_supported(M, N, K, epi):
        mb, cus = N * K * 2 / 1e6, device_cus()

        def cost(nt):   # (the row tiles of a workgroup: as csrc/rows_gemm.hip takes them)
            chain, rounds, tiles = min((r * ((m + nt) * (K // 32) / 58 + 1), r, t) for m in range(1, min(mt, 4) + 1) for t in [-(-mt // m)]
                                       for r in [-(-(-(-(t * (N // (16 * nt)) * products) // 8)) * 8 // cus)])
            again = 0.3 * (tiles - 1) + (0.6 if tiles > 1 and products * mb > 96 else 0)   # (the L2s hold 32 MB)
            return max(2.1 + chain, 2 + products * mb * (1 + again) / 4.9) + 0.05 * chain + (0.3 * rounds if epi == 3 else 0)

        t, wide = (cost(2), False) if epi == 1 else (cost(1), False)
        for nt, form in ((2, True), (4, 2)):
            if N % (16 * nt) == 0 and (nt == 2 or N >= 3072 or M > 64) and not (nt == 2 and epi == 1) and cost(nt) < t:
                t, wide = cost(nt), form
        tiled = _tiled_cost(16 * mt, N, K, epi)
        if epi < 2 and M <= (WS_SWIGLU_MAX_M if epi == 1 else WS_MAX_M) and _decode_static_ok(N, K, epi == 1):
            other = _ws_cost(16 * mt, N, K, epi == 1)
        elif tiled is not None:
            other = tiled * (1.1 if epi == 1 else 0.95)
        else:
            rows = 16 * mt if M <= 64 else 64 * ((M + 63) // 64)
            other = 0.95 * (5.2 + K / 2048 + 3.1e-9 * rows * N * K + 0.19 * mb + 2.8e-7 * rows * (N + K) + (0 if epi in (0, 2) else 2.7))
        est = (t, wide, products * other)
    _ROWS_RULE[key] = est
    return est


def _rows_rule(M: int, N: int, K: int, epi: int, products: int = 1) -> Optional[int]:
    """None: not the few-row kernel; else its ``wide`` argument (False, True or 2)."""
    est = _rows_cost(M, N, K, epi, products)
    return est[1] if est is not None and est[0] < est[2] else None


# What ``tune_decode`` measured of the few-row kernel for a plain or SwiGLU projection, {(M bucket, N, K, swiglu): wide, or None
# where another kernel (``_DECODE_TABLE``) was faster}; the rule above holds for shapes and rows that were not measured.
_ROWS_TABLE: dict = {}
# The us of the kernel that those picks run, {(M bucket, N, K, swiglu): us}
_DECODE_US: dict = {}


def _alone_us(M: int, N: int, K: int, swiglu: bool):
    """us of a plain or SwiGLU product as :func:`linear` runs it: what start-up measured, else the estimate; None without one."""
    if M > LM_HEAD_SKINNY_MAX_M and (_decode_bucket(M), N, K, swiglu) in _DECODE_US:
        return _DECODE_US[(_decode_bucket(M), N, K, swiglu)]
    if GEMV and M <= GEMV_MAX_M and gemv_supported(M, N, K, 2 if swiglu else 0):
        return 1.9 + 0.4 * M + N * K * 2 / 6.4e6
    est = _rows_cost(M, N, K, int(swiglu))
    if est is not None:
        return min(est[0], est[2]) / _few_scale(M)
    return _ws_cost(M, N, K, swiglu) / _few_scale(M) if _decode_static_ok(N, K, swiglu) else None


def _rows_choice(M: int, N: int, K: int, epi: int, products: int = 1) -> Optional[int]:
    if epi < 2 and M > LM_HEAD_SKINNY_MAX_M and _ROWS_TABLE:
        key = (_decode_bucket(M), N, K, epi == 1)
        if key in _ROWS_TABLE:
            return _ROWS_TABLE[key]
    return _rows_rule(M, N, K, epi, products)


def decode_route(M: int, N: int, K: int, swiglu: bool) -> str:
    """The kernel that :func:`linear` / :func:`linear_swiglu` run for M rows of a tuned projection: "rows", "rows wide", "ws" or "gemm"."""
    wide = _rows_choice(M, N, K, 1 if swiglu else 0)
    return _DECODE_TABLE.get((_decode_bucket(M), N, K, swiglu), "ws") if wide is None else "rows wide" if wide else "rows"


def _rows(x, w, b, epi: int):
    """The product on the few-row kernel, or None where the measured table, the rule or the operands' layout say otherwise."""
    if not (x.dim() == 2 and w.dim() == 2 and SKINNY_MAX_M < x.shape[0] <= (WS_MAX_M if GEMM_LIBRARY else ROWS_MAX_M)
            and _gemm_ok(x, w) and w.data_ptr() % 16 == 0):
        return None
    wide = _rows_choice(x.shape[0], w.shape[0], w.shape[1], epi)
    return None if wide is None else lib().rows_linear(x, w, b, epi, wide)


def _decode_gemm_kind(x, w, swiglu: bool) -> Optional[str]:
    if not (use_hip(x) and x.dim() == 2 and w.dim() == 2 and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16):
        return None
    M = x.shape[0]
    N, K = w.shape
    if M < 1 or K % 256 or x.stride(1) != 1 or x.stride(0) % 8 or not w.is_contiguous():
        return None
    if swiglu:
        if N % 2 or (N // 2) % 64:
            return None
    elif N % 128:
        return None
    if M <= SKINNY_MAX_M or (K > WS_MAX_K and M <= WS_MAX_M):
        return "skinny"
    if _DECODE_TABLE and M > LM_HEAD_SKINNY_MAX_M:
        b = _decode_bucket(M)
        choice = _DECODE_TABLE.get((b, N, K, bool(swiglu))) if b is not None else None
        if choice is not None:
            return "ws" if choice == "ws" else None
    if N >= 65536 and not swiglu:
        if M <= LM_HEAD_SKINNY_MAX_M:
            return "skinny"
        return "ws" if WS_LM_HEAD and M <= WS_MAX_M else None
    if M <= (WS_SWIGLU_MAX_M if swiglu else WS_MAX_M):
        return "ws"
    return None


# Prefill / encoder-regime GEMMs (M > WS_MAX_M, and every GEMM with a bias / activation
# epilogue): the hand-written 256 x {256, 192} MFMA kernel of csrc/gemm.hip with the SwiGLU /
# bias / GELU / ReLU epilogue fused.  Two tunables per call: the column tile (192 turns
# N = 6144 into whole waves of 256 CUs) and the K-loop schedule (4 or 2 phases per K-tile).
# ``tune_gemm`` measures them per (M bucket, N, K, epilogue) at engine start-up; untuned
# shapes use the wave-quantisation heuristic of ``_gemm_default``.  The vendor library is
# only reached for shapes the kernel does not support (K % 64, N % 192) -- counted in
# ``LIBRARY_FALLBACKS`` so a test can assert the serving path never takes it.
EPI = {None: 0, "swiglu": 1, "bias": 2, "gelu": 3, "relu": 4}
# measurement knob only: LK_GEMM_LIBRARY=1 sends the prefill-regime GEMMs to hipBLASLt (+ the
# separate activation kernels) for in-situ A/B against the hand-written kernel; =2 only the plain
# ones (no bias / activation / SwiGLU epilogue: QKV, O, down), the fused ones stay hand-written.
# Either turns the fused prefill chain off (its epilogues exist only in gemm.hip).
GEMM_LIBRARY = int(os.environ.get("LK_GEMM_LIBRARY", "0") or 0)
# K-loop schedule of untuned shapes (0: 4 phases per K-tile with per-cluster priority flips,
# 1: 2 phases, 2: 4 phases with a static priority for the lagging half of the waves).  Default:
# 2 for the decoder's K >= 4096 projections (1-5 % faster cold on every Llama-3-8B shape at
# M 4096 / 8192), 0 for the encoder's K 768 / 3072 (neutral there, and 2 lost 8 % on the
# bge QKV at M 65536): profiles/r2_gemm_prio.md.  LK_GEMM_SCHED forces one for every shape.
GEMM_SCHED = int(os.environ["LK_GEMM_SCHED"]) if os.environ.get("LK_GEMM_SCHED") else None


def _gemm_sched(K: int) -> int:
    if GEMM_SCHED is not None:
        return GEMM_SCHED
    return 2 if K >= 4096 else 0
_GEMM_TABLE: dict = {}
# key -> (rows that were measured, the fastest there with ranges of K on gemm1w.hip's tiles among the candidates)
_GEMM_MEASURED: dict = {}
LIBRARY_FALLBACKS: dict = {}
# measured (variant, bn, splits) per (M bucket, N, K, epilogue) for the shipped models' projections
# (benchmarks/gemm_table.py on an MI355X; LK_GEMM_STATIC=0 ignores it)
GEMM_TABLE_FILE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "gemm_table_mi355x.json")
_STATIC: Optional[dict] = None
_STATIC_TOP: dict = {}  # (N, K, epi) -> largest measured M bucket


_CUS: Optional[int] = None


def device_cus() -> int:
    """Compute units of the current device (256 on a whole MI355X; fewer on a partitioned one,
    e.g. CPX mode): the wave size every tile-count policy below quantises against.  256 without a
    GPU (CPU runs never dispatch GPU kernels)."""
    global _CUS
    if _CUS is None:
        _CUS = 256
        if torch.cuda.is_available():
            _CUS = int(torch.cuda.get_device_properties(torch.cuda.current_device()).multi_processor_count) or 256
    return _CUS


def _table_matches_device(doc: dict) -> bool:
    """The shipped table was measured on one device configuration: use it only on the same arch
    and CU count (a partitioned MI355X has different waves, so its measured picks do not apply)."""
    if not torch.cuda.is_available():
        return True
    arch = getattr(torch.cuda.get_device_properties(torch.cuda.current_device()), "gcnArchName", "") or ""
    return arch.split(":")[0] == doc.get("arch", "gfx950") and int(doc.get("cus", 256)) == device_cus()


def _static_table() -> dict:
    global _STATIC
    if _STATIC is None:
        _STATIC = {}
        if os.environ.get("LK_GEMM_STATIC", "1") != "0" and os.path.exists(GEMM_TABLE_FILE):
            import json

            with open(GEMM_TABLE_FILE) as f:
                doc = json.load(f)
            if not _table_matches_device(doc):
                logging.getLogger("lk.ops").warning("gemm table %s was measured on %s / %s CUs; this device differs: not used",
                            GEMM_TABLE_FILE, doc.get("arch"), doc.get("cus", 256))
                return _STATIC
            for mb, n, k, epi, v, bn, ks in doc["entries"]:
                _STATIC[(mb, n, k, epi)] = (v, bn, ks)
                _STATIC_TOP[(n, k, epi)] = max(mb, _STATIC_TOP.get((n, k, epi), 0))
    return _STATIC


def _static_cfg(key):
    """The measured entry of an M bucket; past the largest measured bucket of the shape (the
    encoder's 100k-row batches: many whole waves, where the choice no longer moves with M) the
    largest one's."""
    t = _static_table()
    cfg = t.get(key)
    if cfg is None:
        top = _STATIC_TOP.get(key[1:])
        if top is not None and key[0] > top:
            cfg = t.get((top,) + key[1:])
    return cfg


def _gemm_key(M: int, N: int, K: int, epi: int):
    return ((M + 255) // 256, N, K, epi)


def _measured(M: int, N: int, K: int, epi: int):
    """What ``tune_gemm`` found fastest, where these rows are as many tiles of 128, 192 and 256 rows as those it measured, else None."""
    if not _GEMM_MEASURED:   # (asked for every product of a pass)
        return None
    m, best = _GEMM_MEASURED.get(_gemm_key(M, N, K, epi), (0, None))
    return best if all(-(-M // bm) == -(-m // bm) for bm in (128, 192, 256)) else None


# Variants 3 / 4 / 5 = csrc/gemm1w.hip, the one-wave-per-SIMD kernel with 256-wide column tiles and
# 256 / 192 / 128-row tiles.  The smaller row tiles fill the 256 CUs where 256-row tiles leave most of a
# wave idle (M 2664: QKV on 128-row tiles 107 us, O on 192-row tiles 69 us; profiles/gemm1w_slots.md).
# Which tile wins depends on M through the wave quantisation AND the chip's clocks (a partly
# filled wave runs at a higher clock), so the choice is MEASURED: ``tune_gemm`` times every
# candidate per 256-row M bucket, and a table of those measurements for the shipped models
# (gemm_table_mi355x.json, written by benchmarks/gemm_table.py on an MI355X) is the default;
# ``_gemm_default`` below is the fallback for shapes the table does not hold.
# LK_GEMM1W=0 restores round 4's gemm.hip-only choice.
GEMM1W = os.environ.get("LK_GEMM1W", "1") != "0"
GEMM1W_MIN_TILES = 256
GEMM1W_BM = {3: 256, 4: 192, 5: 128, 6: 256, 7: 256}
# Variants 6 / 7: column split (csrc/gemm1w.hip launch1w_tiles) -- the column tiles that fill whole
# waves of the CUs on 256-row tiles, the rest (under a wave) on 128 / 192-row tiles, two launches.
# QKV at M 4096 = 16 x 24 256-row tiles = 1.5 waves: 16 x 16 tiles, then 32 x 8 128-row tiles.
GEMM1W_SPLIT = {6: 128, 7: 192}
SPLIT_ON = os.environ.get("LK_GEMM_SPLIT", "1") != "0"  # 0: measured 6 / 7 entries run as variant 3 (A/B)


def gemm1w_split_cols(M: int, N: int, epi: int, cus: Optional[int] = None) -> int:
    """Column tiles a variant 6 / 7 launch runs on 256-row tiles (mirrors lk_gemm1w_split_cols,
    which uses the device's CU count too); 0 or all of them: no split (the launch is variant 3's)."""
    cus = cus or device_cus()
    tn = N // 256
    tm = (M + 255) // 256
    return min(tn, (tm * tn // cus) * cus // tm)


def _split_applies(M: int, N: int, epi: int) -> bool:
    return 0 < gemm1w_split_cols(M, N, epi) < N // 256


def _gemm_configs(N: int, epi: int):
    """(schedule / variant, column tile) candidates the kernels support for this N / epilogue."""
    bns = [256] if epi == 1 else [bn for bn in (256, 192) if N % bn == 0]
    cfgs = [(sched, bn) for bn in bns for sched in (0, 1, 2)]
    if 256 in bns and GEMM1W:
        cfgs += [(v, 256) for v in GEMM1W_BM]
    return cfgs


def _gemm_default(M: int, N: int, K: int, epi: int):
    """Fallback policy for shapes without a measured entry.  gemm.hip: fewest tile-columns x
    waves, cost(bn) = ceil(tiles / 256 CUs) * bn (ties -> 256), 4-phase schedule (fastest of its
    schedules with weights streamed from HBM: profiles/r2_gemm.md).  gemm1w.hip (256-row tiles)
    instead once its tiles fill a wave, and its 192-row tiles where 256-row tiles would leave
    over a third of a single wave idle while 192-row ones still fit in one."""
    tm = (M + 255) // 256
    cus = device_cus()
    best = None
    for _, bn in _gemm_configs(N, epi):
        n_cols = N // 2 // 128 if epi == 1 else N // bn
        cost = -(-tm * n_cols // cus) * (256 if epi == 1 else bn)
        if best is None or cost < best[0]:
            best = (cost, bn)
    if best is None:
        return None
    bn = best[1]
    ks = _gemm_splits(M, N, K, epi, bn)
    tiles = tm * (N // 2 // 128 if epi == 1 else N // bn)
    if GEMM1W and bn == 256 and ks == 1 and K // 64 >= 3:
        if tiles >= GEMM1W_MIN_TILES:
            return (3, 256, 1)
        tiles192 = -(-M // 192) * (N // 2 // 128 if epi == 1 else N // 256)
        if tiles < 0.7 * cus and tiles192 <= cus:
            return (4, 256, 1)
    return (_gemm_sched(K), bn, ks)


# split-K for shapes with at most half as many tiles as CUs (M <= 2048 O / down projections,
# the 70B TP=8 QKV shard at N 1280), and 3 K-ranges for long-K shapes of 129-160 tiles:
# fp32 partials of up to 4 K-ranges, each of >= 8 K-tiles,
# summed by a reduce kernel that applies the epilogue (profiles/r2_gemm_splitk.md); LK_GEMM_SPLITK=0
# turns it off
GEMM_SPLITK = os.environ.get("LK_GEMM_SPLITK", "1") != "0"


def _gemm_splits(M: int, N: int, K: int, epi: int, bn: int) -> int:
    if not GEMM_SPLITK or epi == 1:
        return 1
    tiles = ((M + 255) // 256) * (N // bn)
    if tiles > 128:
        # long K just past half a wave: three K-ranges give ~1.7-1.9 waves of tiles
        # (M 2304 / 2560 down projection: 295 -> 278, 277 -> 255 us; from 176 tiles on, worse)
        return 3 if tiles <= 160 and K >= 8192 else 1
    return max(1, min(4, device_cus() // tiles, K // 64 // 8))


def _gemm_ok(x, w) -> bool:
    return (use_hip(x) and x.dim() == 2 and w.dim() == 2 and x.dtype == torch.bfloat16
            and w.dtype == torch.bfloat16 and x.stride(1) == 1 and x.stride(0) % 8 == 0
            and w.is_contiguous() and x.data_ptr() % 16 == 0)


def gemm(x, w, b=None, epi: int = 0, out=None):
    """epi(x w^T (+ b)) on the hand-written kernel; None if the shape is unsupported."""
    M, K = x.shape
    N = w.shape[0]
    # the epilogue stores / bias loads are 16-byte vectors
    if b is not None and (b.data_ptr() % 16 or not b.is_contiguous()):
        return None
    if out is not None and (out.data_ptr() % 16 or out.stride(0) % 8 or out.stride(1) != 1):
        return None
    cfg = _cfg_of(M, N, K, epi)
    cfg = _split_rule(M, N, K, epi, cfg, x.stride(0) if out is None else max(x.stride(0), out.stride(0)))
    if cfg is None or not lib().gemm_supported(M, N, K, epi, cfg[1], cfg[2], cfg[0]):
        return None
    return lib().gemm(x, w, b, epi, cfg[1], out, cfg[0], cfg[2])


def _library(x, w, b, act, key):
    LIBRARY_FALLBACKS[key] = LIBRARY_FALLBACKS.get(key, 0) + 1
    y = torch.nn.functional.linear(x, w, b)
    if act == "gelu":
        gelu_(y)
    elif act == "relu":
        relu_(y)
    return y


def tune_gemm(weights, max_m: int, min_m: int = 512, iters: int = 6, cold_bytes: int = 600 << 20,
              ms: Optional[list] = None) -> dict:
    """Time every (schedule / variant, column tile) of the prefill kernels for each 256-row M
    bucket in [min_m, max_m] (or the row counts ``ms``) and each (weight, epilogue) pair; keep
    the fastest.  gemm.hip candidates run with the split-K the policy gives them, gemm1w.hip
    unsplit; where K may also be cut into ranges on gemm1w.hip's tiles (``_split_rule``), those that are estimated
    within 1.3 of the best such split are measured too and kept apart (QKV and SwiGLU of a fused step take no split).  As in serving, the weights arrive from HBM: each launch reads the next of enough
    weight copies to overflow the 256 MB MALL (a warm-weight tuning picks the 2-phase schedule for
    the SwiGLU projection, which is 3 % slower in situ).  Candidates are timed round-robin so
    clock drift hits all alike.  ``weights``: [(w [N, K] bf16 CUDA tensor, epi)].  Returns
    {key: {cfg: us}} and fills the tuned table."""
    import statistics

    L = lib()
    out = {}

    def once(fn):
        a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        a.record()
        fn()
        b.record()
        b.synchronize()
        return a.elapsed_time(b) * 1e3

    rows = ms if ms is not None else [mb * 256 for mb in range(max(min_m, 256) // 256, max_m // 256 + 1)]
    for w, epi in weights:
        N, K = w.shape
        copies = [w] + [w.clone() for _ in range(max(0, -(-cold_bytes // (N * K * 2)) - 1))]
        rot = [0]

        def wn():
            rot[0] = (rot[0] + 1) % len(copies)
            return copies[rot[0]]

        bias = torch.zeros(N, device=w.device, dtype=torch.bfloat16) if epi >= 2 else None
        xmax = torch.randn(max(rows), K, device=w.device, dtype=torch.bfloat16)
        for M in rows:
            x = xmax[:M]
            cfgs = []
            for v, bn in _gemm_configs(N, epi):
                if v in GEMM1W_SPLIT and not _split_applies(M, N, epi):
                    continue  # the same launch as variant 3
                ks = 1 if v in GEMM1W_BM else _gemm_splits(M, N, K, epi, bn)
                if not L.gemm_supported(M, N, K, epi, bn, ks, v):
                    ks = 1
                if L.gemm_supported(M, N, K, epi, bn, ks, v):
                    cfgs.append((v, bn, ks))
            if not cfgs:
                continue
            ranges = _split_costs(M, N, K) if _split_takes(M, N, K, epi, K) else {}
            ranges = {c: t for c, t in ranges.items() if c[2] > 1 and L.gemm_supported(M, N, K, epi, c[1], c[2], c[0])}
            unsplit, cfgs = cfgs, cfgs + [c for c, t in ranges.items() if t <= 1.3 * min(ranges.values())]
            fns = {c: (lambda c=c: L.gemm(x, wn(), bias, epi, c[1], None, c[0], c[2])) for c in cfgs}
            for f in fns.values():
                f()
            ts = {c: [] for c in cfgs}
            for _ in range(iters):
                for c, f in fns.items():
                    ts[c].append(once(f))
            med = {c: statistics.median(v) for c, v in ts.items()}
            key = _gemm_key(M, N, K, epi)
            _GEMM_TABLE[key], _GEMM_MEASURED[key] = min(unsplit, key=med.get), (M, min(med, key=med.get))
            out[key] = {f"v{c[0]}/{c[1]}/k{c[2]}": round(t, 1) for c, t in med.items()}
        del copies
    return out


# decode tuner: also pick the weight-streaming kernel variant per row tile (LK_WS_VARIANT_TUNE=0:
# keep LK_WS_LOADER's default everywhere)
WS_VARIANT_TUNE = os.environ.get("LK_WS_VARIANT_TUNE", "1") != "0"
_WS_VARIANTS: dict = {}  # (row-tile top M, N, K, swiglu) -> 0 ring / 1 loader waves (also set in _C)


def apply_ws_variants(table: dict):
    """Install measured weight-streaming kernel variants (a TP worker applies its leader's)."""
    _WS_VARIANTS.clear()
    _WS_VARIANTS.update(table)
    if table and available():
        L = lib()
        for (M, N, K, sw), v in table.items():
            L.ws_set_variant(M, N, K, sw, v)


def tune_decode(weights, ms: Sequence[int] = DECODE_TUNE_MS, iters: int = 3, cold_bytes: int = 640 << 20) -> dict:
    """For each decode-sized M bucket and each (weight, swiglu) pair, time the weight-streaming
    kernel, the prefill GEMM and the few-row kernel in a hipGraph, each launch on the next copy
    of the weight (enough to overflow the 256 MB MALL for weights of 4 MB and more; below, 64 copies
    lie in it whole), and record the faster of the first two (`_DECODE_TABLE`: what
    steps with a fused consumer choose by) and whether the few-row kernel is faster still
    (`_ROWS_TABLE`: what `linear` chooses by).  The few-row rule's answer stands unless another arm is 5 %
    faster, so that near ties do not change from one start to the next.  Returns
    {(M, N, K, swiglu): {"ws" / "gemm": us}}, {(M, N, K, swiglu, "few", "rows"): {arm: us}} of all arms and,
    per row tile that has two kernels (64 and 128 rows), {(M, N, K, swiglu, "ws_variant"): {"ring" / "loader": us}}."""
    import statistics

    L = lib()
    out = {}
    side = torch.cuda.Stream() if len(weights) else None
    for w, swiglu in weights:
        N, K = w.shape
        swiglu = bool(swiglu)
        # (at most 64 launches per graph: a thousand captured launches per arm took seconds, and for small weights a launch's
        # chain and not the memory decides)
        copies = [w] + [w.clone() for _ in range(min(63, max(1, -(-cold_bytes // (N * K * 2)) - 1)))]

        def timed(fns):
            # as decode steps run: launches of a hipGraph (eager ones of a few microseconds are bound by the
            # host, which favoured the arm with fewer launches: 64 x 2048 x 2048 went to the prefill GEMM,
            # 18.5 us against 10.9 in a graph, and SwiGLU 64 x 11264 x 2048 at random, 32.5 against 19.5)
            ts, graphs = {k: [] for k in fns}, {}
            for fn in fns.values():  # warm-up (and first-launch attributes)
                fn(copies[0])
            torch.cuda.synchronize()
            # (inference mode, as the engine's own captures: the generator's graph state may be an inference tensor by now)
            with torch.inference_mode(), torch.cuda.stream(side):
                for k, fn in fns.items():
                    graphs[k] = torch.cuda.CUDAGraph()
                    graphs[k].capture_begin(capture_error_mode="thread_local")
                    try:
                        for c in copies[1:] + copies[:1]:
                            fn(c)
                    finally:
                        graphs[k].capture_end()
            for i in range(iters):
                for k, g in graphs.items():
                    if i >= 2 and max(ts[k][:2]) < 1.02 * min(ts[k][:2]):   # the launches' own spread: a third round changes nothing
                        continue
                    a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                    a.record()
                    g.replay()
                    b.record()
                    b.synchronize()
                    ts[k].append(a.elapsed_time(b) * 1e3 / len(copies))
            return {k: statistics.median(v) for k, v in ts.items()}

        # the weight-streaming kernel's variant per row tile (64 / 128 rows; past those there is the
        # ring only): one LDS ring vs loader waves (csrc/skinny_gemm.hip wsgemm_lw_kernel), measured
        # at the tile's largest M, before the routing below times the ws arm with it
        if WS_VARIANT_TUNE and _decode_static_ok(N, K, swiglu):
            for M in [m for m in (64, 128) if m in ms]:
                x = torch.randn(M, K, device=w.device, dtype=torch.bfloat16)
                fns = {}
                for v in (0, 1):
                    fns[v] = (lambda c, v=v: (L.ws_set_variant(M, N, K, swiglu, v), L.ws_linear(x, c, swiglu)))
                med = timed(fns)
                best = min(med, key=med.get)
                L.ws_set_variant(M, N, K, swiglu, best)
                _WS_VARIANTS[(M, N, K, swiglu)] = best
                out[(M, N, K, swiglu, "ws_variant")] = {("ring", "loader")[v]: round(t, 1) for v, t in med.items()}
        for M in ms:
            x = torch.randn(M, K, device=w.device, dtype=torch.bfloat16)
            arms = {}
            if M <= 256 and _decode_static_ok(N, K, swiglu):
                arms["ws"] = lambda c, x=x: L.ws_linear(x, c, swiglu)
            epi = 1 if swiglu else 0
            cfg = _gemm_default(M, N, K, epi)
            if cfg is not None and L.gemm_supported(M, N, K, epi, cfg[1], cfg[2], cfg[0]):
                arms["gemm"] = lambda c, x=x, cfg=cfg: L.gemm(x, c, None, epi, cfg[1], None, cfg[0], cfg[2])
            # the few-row kernel in the form that the rule prefers, unless the rule has it beyond 1.5 times the others (its
            # estimates are good to 30 %)
            est = _rows_cost(M, N, K, epi)
            rows = {}
            if (est is not None and est[0] < 1.5 * est[2] and SKINNY_MAX_M < M <= (WS_MAX_M if GEMM_LIBRARY else ROWS_MAX_M)
                    and w.data_ptr() % 16 == 0):
                rows["rows wide" if est[1] else "rows"] = lambda c, x=x, wide=est[1]: L.rows_linear(x, c, None, epi, wide)
            if len(arms) + len(rows) < 2:
                continue
            med = timed({**arms, **rows})
            key = (M, N, K, swiglu)
            if len(arms) > 1:
                _DECODE_TABLE[key] = min(arms, key=med.get)
                out[key] = {k: round(med[k], 1) for k in arms}
            run = min(arms, key=med.get) if arms else None
            if rows and arms:
                best = min(med, key=med.get)
                stay = next(iter(rows)) if est[0] < est[2] else min(arms, key=med.get)
                pick = best if med[best] < 0.95 * med[stay] else stay
                _ROWS_TABLE[key] = est[1] if pick in rows else None
                run = pick
                out[key + ("few", "rows")] = {k: round(v, 1) for k, v in med.items()}
            if run is not None:
                _DECODE_US[key] = med[run]
        del copies
    return out


def _decode_static_ok(N: int, K: int, swiglu: bool) -> bool:
    if K % 256 or K > WS_MAX_K:
        return False
    return (N % 2 == 0 and (N // 2) % 64 == 0) if swiglu else N % 128 == 0


def linear(x, w, b=None, act: Optional[str] = None):
    """Projection GEMM (+ bias, + GELU / ReLU): few rows on the one-launch kernel with any epilogue,
    decode-sized batches without an epilogue on the weight-streaming MFMA kernels (skinny / ws),
    everything else on the prefill kernel with the epilogue fused."""
    if not use_hip(x):
        y = torch.nn.functional.linear(x, w, b)
        if act is not None:
            y = ref.activation_(y, None, 0 if act == "gelu" else 2)
        return y
    if b is None and act is None:
        if _gemv_ok(x, w, 0):
            return lib().gemv_decode(0, x, w)
        y = _rows(x, w, None, 0)
        if y is not None:
            return y
        kind = _decode_gemm_kind(x, w, False)
        if kind == "skinny":
            return lib().skinny_linear(x, w)
        if kind == "ws":
            return lib().ws_linear(x, w)
    epi = EPI["bias" if act is None else act] if b is not None else 0
    if act is not None and b is None:
        b = torch.zeros(w.shape[0], device=x.device, dtype=x.dtype)
        epi = EPI[act]
    lib_arm = GEMM_LIBRARY == 1 or (GEMM_LIBRARY == 2 and epi == 0 and x.shape[0] > WS_MAX_M)
    if epi >= 2 and not lib_arm and b.dtype == torch.bfloat16 and b.is_contiguous() and b.numel() == w.shape[0]:
        y = _rows(x, w, b, epi)
        if y is not None:
            return y
    y = gemm(x, w, b, epi) if _gemm_ok(x, w) and not lib_arm else None
    if y is None:
        y = _library(x, w, b, act, (x.shape[0] > WS_MAX_M, w.shape[0], w.shape[1], epi))
    return y


def linear_pair(x1, w1, x2, w2):
    """(x1 w1^T, x2 w2^T) of two products of the same sizes: one launch where both are the few-row kernel's."""
    if use_hip(x1) and x1.dim() == 2 and x1.shape == x2.shape and w1.shape == w2.shape and not _gemv_ok(x1, w1, 0):
        M, (N, K) = x1.shape[0], w1.shape
        if (SKINNY_MAX_M < M <= (WS_MAX_M if GEMM_LIBRARY else ROWS_MAX_M) and _gemm_ok(x1, w1) and _gemm_ok(x2, w2)
                and w1.data_ptr() % 16 == 0 and w2.data_ptr() % 16 == 0):
            wide = _rows_choice(M, N, K, 0, 2)
            if wide is not None:
                return lib().rows_pair(x1, w1, x2, w2, wide)
    return linear(x1, w1), linear(x2, w2)


# Two products of one x in one launch (csrc/skinny_gemm.hip ws_beside_kernel): a product of a few rows that does not fill the chip leaves CUs and
# the memory idle at its start and its end, and both of these once.  64 W rows per workgroup where all of them run in one round of the CUs
# (two fit a CU's LDS), else 128 where those do: 64 re-read x twice as often, and past one round the CUs with two workgroups hold up the launch.
# Beyond, each product fills the chip by itself and the launch gains nothing; at few rows 128 pay from two thirds of the CUs on (fewer take in
# less than the memory gives).  A workgroup walks the whole of K, which the launches apart cut into ranges: where that chain by itself is as long
# as they are, few workgroups wait for it, and the products stay apart (1 / 128 rows: 384 + 2 x 512, K 8192 8.9 / 25.0 apart, 25.5 / 52.3
# together; 2048 + 2 x 2048, K 2048 8.2 / 16.7, 9.5 / 17.0).  Over 1,172 products (N 64 - 16384, I 64 - 13824, K 256 - 8192, 1 - 128 rows) 0.851 of the
# time apart, 8 of them slower by 3 % or more, 1.105 at most; without the chain in the rule 0.902, 230 and 2.9.
# Plain + SwiGLU apart -> together, us, weights cold, 1 / 4 / 16 / 64 / 128 rows:
#    3072 + 2 x 5632, K 2048   64: 13.3 / 14.4 / 15.2 / 21.4 / 32.0 -> 11.3 / 11.3 / 11.5 / 13.9 / 18.5
#   10496 + 2 x 5632, K 2048  128: 18.2 / 19.2 / 20.3 / 27.6 / 42.7 -> 18.2 / 17.3 / 17.6 / 20.8 / 25.6   (with 64: 20.7 / 19.7 / 20.0 / 24.3 / 31.6)
#    1536 + 2 x 2048, K 1024   64:  7.2 /  7.7 /  7.9 /  9.3 / 11.5 ->  6.2 /  6.3 /  6.4 /  8.0 / 10.5
#    4096 + 2 x 8192, K 4096  128: 30.2 / 29.7 / 30.1 / 38.7 / 54.8 -> 29.8 / 30.1 / 30.8 / 36.0 / 44.9   (taken from 49 rows on)
#    5120 + 2 x 13824, K 5120 128: 57.1 / 57.9 / 60.7 / 75.3 / 90.5 -> 52.3 / 52.1 / 52.3 / 56.6 / 66.7
#    6144 + 2 x 14336, K 4096   -: 47.6 / 49.5 / 49.8 / 57.1 / 70.5    (64: 54.1 / 54.4 / 55.1 / 66.2 / 87.8; 128: 62.9 / 63.3 / 64.2 / 70.9 / 85.6)
BESIDE_MAX_M = 128


def _beside_rule(M: int, N: int, I: int, K: int) -> int:
    """W rows per workgroup for N plain and I SwiGLU output columns in one launch; 0: two launches."""
    if not 1 <= M <= BESIDE_MAX_M or not 64 <= K <= WS_MAX_K or K % 64:
        return 0
    if N < 1 or I < 1:
        return 0
    cus, tiles = device_cus(), N // 128 + I // 64
    if N % 64 == 0 and I % 32 == 0 and N // 64 + I // 32 <= cus:
        bn = 64
    elif N % 128 == 0 and I % 64 == 0 and tiles <= cus and (M > 48 or tiles >= 0.65 * cus):
        bn = 128
    else:
        return 0
    # the chain of one workgroup: per 64 of K the tile's columns, the row tile and the rows in it
    chain = 4.0 + K / 64 * ((0.14 if bn == 64 else 0.32) + 0.056 * (-(-M // 64) - 1) + 0.034 * -(-M // 16))
    alone = _alone_us(M, N, K, False), _alone_us(M, 2 * I, K, True)
    # (one or two rows stream at the matrix-vector kernel's rate, to which a chain has to leave room)
    gemv = GEMV and M <= GEMV_MAX_M and gemv_supported(M, N, K, 0) and gemv_supported(M, 2 * I, K, 2)
    return bn if None not in alone and chain < (0.82 if gemv else 1.0) * sum(alone) else 0


def linear_beside(x, w, w_gate_up):
    """(x w^T, silu(x wg^T) * (x wu^T)) for a fused [wg; wu] weight in one launch; None where two pay."""
    if not GEMM_LIBRARY and _gemm_ok(x, w) and _gemm_ok(x, w_gate_up) and w.data_ptr() % 16 == 0 and w_gate_up.data_ptr() % 16 == 0:
        bn = _beside_rule(x.shape[0], w.shape[0], w_gate_up.shape[0] // 2, w.shape[1])
        if bn and w.shape[1] == w_gate_up.shape[1] == x.shape[1] and w_gate_up.shape[0] % 2 == 0:
            return tuple(lib().ws_beside(x, w, w_gate_up, bn))
    return None


def sums_pay(M: int, N: int, K1: int, K2: int) -> bool:
    """Whether :func:`linear_sums` of weights [N, K1] and [N, K2] is worth its launch.  What decides is the longest range of K that a
    workgroup gets against the mean: where it is longer, part of the chip waits while the weights' stream runs on.  Launches apart and the
    norm / the sums and theirs, us, weights cold, 1 / 4 / 16 / 64 rows (longest over mean):
      2048 x (4096 | 5632)  1.07: 15.2 / 17.2 / 20.7 / 25.2 -> 12.4 / 12.8 / 13.1 / 17.3     5120 x (5120 | 5120)  1.5: 31 / 32 / 37 / 54 -> 31 / 31 / 33 / 43
      4096 x (4096 | 8192)  1.33: 26.5 / 29.1 / 30.9 / 42.7 -> 27.3 / 27.9 / 28.5 / 33.8     8192 x (4096 | 6144)  1.2: 40 / 41 / 42 / 56 -> 42 / 42 / 44 / 53
      6144 x (6144 | 16384) 1.45: 56 / 65 / 69 / 82 -> 68 / 69 / 73 / 96                     8192 x (8192 | 28672) 1.56: 107 / 118 / 120 / 128 -> 128 / 129 / 137 / 177
      8192 x (8192 | 8192)  1.0:  57 / 72 / 73 / 81 -> 65 / 66 / 65 / 67 (one or two rows: the matrix-vector kernel at 4.7 TB/s)
    Weights of up to 64 MB together gain the launch whatever the ranges (8192 x (512 | 960), 1.39: 17.1 / 17.8 / 18.5 / 22.1 -> 16.6 / 17.3 / 18.0 / 21.9)."""
    if N * (K1 + K2) * 2 <= 64e6:
        return True
    parts = device_cus() // max(1, N // 64)
    if parts < 2 or (parts == 2 and M <= 2):
        return False
    longest = min(max(-(-K1 // (256 * s)), -(-K2 // (256 * (parts - s)))) for s in range(1, parts))
    return longest * 256 * parts <= (1.15 if parts == 2 else 1.3 if M <= 2 else 1.5) * (K1 + K2)


def linear_sums(x1, w1, x2, w2):
    """(parts, s1): the f32 parts [n, M, N] of x1 w1^T (the first s1) and x2 w2^T in one launch, for ``stream_rmsnorm(sums=...)``;
    None where the two products run apart (a program asks :func:`sums_pay` too)."""
    if use_hip(x1) and x1.dim() == 2 and x2.dim() == 2 and not GEMM_LIBRARY and x1.shape[0] == x2.shape[0] and w1.shape[0] == w2.shape[0]:
        if (_gemm_ok(x1, w1) and _gemm_ok(x2, w2) and w1.data_ptr() % 16 == 0 and w2.data_ptr() % 16 == 0
                and lib().rows_sums_supported(x1.shape[0], w1.shape[0], w1.shape[1], w2.shape[1])):
            return lib().rows_sums(x1, w1, x2, w2)
    return None


# Encoder passes of few rows: the layer norms and the attention run inside the projections behind them (csrc/encoder_rows.hip).  Every
# workgroup normalises its tile's rows, so what a launch saves is lost again with more of them, sooner where the layers are narrow and each of
# their launches is short: up to 32 rows at width 768, 16 below.  A captured pass, launches apart -> fused, us (cold: 512 MB read before):
#   12 layers of 768, one text of 8 / 16 / 19 / 32 / 40 tokens: 299 / 316 / 314 / 344 / 343 -> 255 / 277 / 275 / 299 / 351,
#     cold 350 / 365 / 357 / 376 / 373 -> 280 / 301 / 300 / 323 / 369; 8 texts of 2 / of 4 tokens 316 / 347 -> 306 / 324
#   6 layers of 384, heads of 64, one text of 8 / 16 / 22 / 32 / 40 tokens: 131 / 133 / 133 / 134 / 136 -> 110 / 115 / 118 / 126 / 156,
#     cold 155 / 158 / 156 / 158 / 158 -> 124 / 128 / 130 / 138 / 173; 8 texts of 2 / 3 / 4 tokens 134 / 134 / 136 -> 132 / 134 / 139
ENCODER_ROWS = 32


def encoder_rows_ok(h, width: int, inner: int) -> bool:
    """Whether :func:`ln_linear` takes these rows in the projections of an encoder layer (``width`` to 3 ``width`` and to ``inner``)."""
    return (use_hip(h) and h.dtype == torch.bfloat16 and not GEMM_LIBRARY and 1 <= h.shape[0] <= (ENCODER_ROWS if width >= 768 else ENCODER_ROWS // 2)
            and all(lib().ln_linear_supported(h.shape[0], n, width) for n in (3 * width, inner)))


def _fused_weight(w, *vectors) -> bool:
    """Whether the fused encoder launches read a projection's weight and the vectors beside it as they lie: contiguous bf16, and the
    weight on a 16-byte line."""
    return all(t is not None and t.dtype == torch.bfloat16 and t.is_contiguous() for t in (w, *vectors)) and w.data_ptr() % 16 == 0


def linear_add(x, w, b, residual):
    """x w^T + b, then + residual (each rounded on its own, as the two operations apart round)."""
    if use_hip(x) and not GEMM_LIBRARY and _fused_weight(w, b) and _gemm_ok(x, w):
        est = _rows_cost(x.shape[0], w.shape[0], w.shape[1], 2)
        if est is not None:
            return lib().rows_linear(x, w, b, 5, est[1], residual)
    return linear(x, w, b) + residual


def ln_linear(s, ln_w, ln_b, eps: float, w, b, act: Optional[str] = None):
    """(act(h w^T + b), h) with h = LN(s); ``act``: None or "gelu"."""
    if use_hip(s) and _fused_weight(w, b, ln_w, ln_b) and ln_w.data_ptr() % 16 == 0 and ln_b.data_ptr() % 16 == 0:
        return lib().ln_linear(s, ln_w, ln_b, eps, w, b, act == "gelu")
    h = layernorm(s, ln_w, ln_b, eps)
    return linear(h, w, b, act=act), h


def attn_linear_add(qkv, cu, lens_cpu, nh: int, head_dim: int, scale: float, w, b, residual, tiles=None):
    """Bidirectional attention over packed rows [q | k | v], the projection of its output and the residual; one launch for one short
    text."""
    K = nh * head_dim
    if (use_hip(qkv) and not GEMM_LIBRARY and head_dim == 64 and lens_cpu is not None and len(lens_cpu) == 1 and lens_cpu[0] == qkv.shape[0]
            and _fused_weight(w, b) and lib().attn_linear_supported(qkv.shape[0], nh, w.shape[0])):
        return lib().attn_linear(qkv, nh, scale, w, b, residual)
    a = flash_prefill(qkv[:, :K], qkv[:, K:2 * K], qkv[:, 2 * K:], cu, nh, nh, head_dim, scale, False, q_lens_cpu=lens_cpu, tiles=tiles)
    return linear_add(a, w, b, residual)


def linear_swiglu(x, w_gate_up):
    """silu(x Wg^T) * (x Wu^T) for a fused [Wg; Wu] weight: one kernel (GEMM with the
    SwiGLU epilogue) in every regime."""
    if not use_hip(x):
        return silu_mul(linear(x, w_gate_up))
    if _gemv_ok(x, w_gate_up, 2):
        return lib().gemv_decode(2, x, w_gate_up)
    y = _rows(x, w_gate_up, None, 1)
    if y is not None:
        return y
    kind = _decode_gemm_kind(x, w_gate_up, True)
    if kind == "skinny":
        return lib().skinny_linear(x, w_gate_up, True)
    if kind == "ws":
        return lib().ws_linear(x, w_gate_up, True)
    y = gemm(x, w_gate_up, None, 1) if _gemm_ok(x, w_gate_up) and GEMM_LIBRARY != 1 else None
    if y is None:
        y = silu_mul(_library(x, w_gate_up, None, None, (True, w_gate_up.shape[0], w_gate_up.shape[1], 1)))
    return y


# Decode-step fusions: when the weight-streaming GEMM splits K (S >= 2 partial slabs),
# the consumer kernel does the split-K reduction itself -- RMSNorm(+residual) after the
# o / down projections, RoPE + paged-KV write after QKV -- so each of those projections
# costs one launch fewer (three per layer; bit-identical to the unfused ops).
DECODE_FUSION = os.environ.get("LK_DECODE_FUSION", "1") != "0"
_WS_PLANS: dict = {}


def _ws_split_plan(x, w):
    """(BN, S) of the weight-streaming GEMM when it runs split-K for this shape, else None."""
    if not DECODE_FUSION or _decode_gemm_kind(x, w, False) != "ws":
        return None
    key = (x.shape[0], w.shape[0], w.shape[1])
    plan = _WS_PLANS.get(key)
    if plan is None:
        plan = _WS_PLANS[key] = tuple(lib().ws_plan(*key, False))
    return plan if plan[1] in (2, 4, 8) else None


# Split-K decode GEMMs whose reduction runs in their own last workgroup(s) (csrc/skinny_gemm.hip
# WsTail): the QKV projection's RoPE + paged-KV write (one ticket per head), and for <= 4 rows the
# o / down projections' residual + RMSNorm -- no reduce launch after them.  Measured OFF: at batch 1
# (same box, twice each, profiles/r6_ws_tail/) a decode step took 4.34 / 4.32 ms with the tails vs
# 3.685 / 3.672 ms with the three ~5 us reduce launches per layer (p50 161.8 vs 139.4 ms): the
# write-through partials and the one-workgroup reductions cost more than the launches they save.
# LK_WS_FUSED_TAIL=1 turns them on (numerics: tests/test_kernels_gpu.py *fused_tail*).
WS_FUSED_TAIL = os.environ.get("LK_WS_FUSED_TAIL", "0") == "1"
_WS_TICKETS: dict = {}


def ws_tickets(device):
    """Zeroed int32 tickets of the fused split-K tails (one buffer per device, made before any
    graph capture by the model runner; every ticket is reset by its last taker)."""
    device = torch.device(device)
    key = device.index if device.index is not None else torch.cuda.current_device()
    t = _WS_TICKETS.get(key)
    if t is None:
        t = _WS_TICKETS[key] = torch.zeros(4096, dtype=torch.int32, device=device)
    return t


# Consumer-side prologues in the decode step (csrc/skinny_gemm.hip WsPro, rows <= XPRO_MAX_M, one
# GPU without TP): the O projection merges the paged-decode split partials itself (no
# decode_reduce launch) and gate_up / the next layer's QKV compute residual add + RMSNorm of the
# previous projection's split-K slabs themselves (no rmsnorm launch) -- three launches fewer per
# layer, bit-identical values (models/llama.py _forward_decode_xpro).  Measured slower at batch 1
# (decode step 4.23 vs 3.58 ms: every workgroup re-reads and re-normalises the producer's fp32 slabs,
# and the O projection's merge prologue costs 17 us; profiles/r6_xpro/): off unless LK_DECODE_XPRO=1.
XPRO = os.environ.get("LK_DECODE_XPRO", "0") == "1"
XPRO_MAX_M = int(os.environ.get("LK_DECODE_XPRO_MAX_M", "16"))
_PLAN_CACHE: dict = {}


def ws_plan(M: int, N: int, K: int, swiglu: bool = False) -> tuple:
    """(BN, S) of the weight-streaming GEMM for this shape (lk_wsgemm_plan)."""
    key = (M, N, K, swiglu)
    p = _PLAN_CACHE.get(key)
    if p is None:
        p = _PLAN_CACHE[key] = tuple(lib().ws_plan(M, N, K, swiglu))
    return p


def ws_pro(x, w, plan, kind: int, swiglu: bool = False, reduce: bool = False, **kw):
    """Weight-streaming GEMM with a consumer-side X prologue (``kind`` 1: x = RMSNorm(bf16(sum of
    ``pp``) + ``res_in``) * ``gamma``, ``res_out`` = the summed residual; 2: x = the paged-decode
    output with its split partials ``po`` / ``pml`` merged; 0: plain x).  Returns the f32 partial
    slabs [S, M, N] (S > 1 and not ``reduce``) or the bf16 / SwiGLU output."""
    return lib().ws_pro(x, w, swiglu, plan[0], plan[1], kind, reduce, **kw)


# Decode GEMV for one or two rows (csrc/gemv_decode.hip): no split-K slabs, the RMSNorm in the
# consumer's prologue, residual add / SwiGLU / RoPE + paged-KV write in the epilogue -- a Llama
# block's batch-1 decode step is QKV -> paged decode -> O -> gate_up -> down, with no reduce, norm
# or RoPE launch (models/llama.py _forward_decode_gemv).  LK_DECODE_GEMV=0: the weight-streaming path.
GEMV = os.environ.get("LK_DECODE_GEMV", "1") != "0"
GEMV_MAX_M = 2
# LK_GEMV_MERGE=1: the O projection's GEMV merges the paged-decode split partials itself (no
# decode_reduce launch).  Measured slightly slower at batch 1 (decode step 3.129 / 3.133 vs 3.104 /
# 3.110 ms: every workgroup re-reads all split partials), so the reduce kernel stays the default
GEMV_MERGE = os.environ.get("LK_GEMV_MERGE", "0") == "1"
_GEMV_OK: dict = {}


# The long-K projections (K split into an even number >= 2 of streaming blocks: down at K 14,336,
# the 70B QKV / gate_up at K 8,192) take two waves per pair of W rows, a K half each, their sums
# joined in LDS (LK_GEMV_KSPLIT=0: one wave per pair).  The first W block is requested behind X's
# LDS-DMA and ahead of the prologue's waits; requested before X it held X up (loads return in order:
# 3.199 vs 3.17 ms; by LDS-DMA 3.31 vs 3.10, profiles/r6_gemv/).  Workgroup target (LK_GEMV_WGS, 0: 512)
GEMV_KSPLIT = os.environ.get("LK_GEMV_KSPLIT", "1") != "0"
GEMV_WGS = int(os.environ.get("LK_GEMV_WGS", "0") or 0)


# Batch-1 decode: while the latency-bound paged-decode kernels leave HBM idle, a side stream reads
# the O projection's weights (and the first LK_GEMV_L3_PREFETCH_MB of gate_up's gate / up rows)
# through the 256 MiB Infinity Cache so the GEMVs behind the attention read them from L3.
# -1: off; 0: O only.
GEMV_L3_MB = int(os.environ.get("LK_GEMV_L3_PREFETCH_MB", "-1") or -1)
GEMV_L3_WGS = int(os.environ.get("LK_GEMV_L3_WGS", "128") or 128)
_L3_SINK: dict = {}


def l3_prefetch(t, r0: int, r1: int):
    """Read rows [r0, r1) of a contiguous 2-D GPU tensor (values unused) on the current stream."""
    s = _L3_SINK.get(t.device)
    if s is None:
        s = _L3_SINK[t.device] = torch.zeros(1, dtype=torch.int32, device=t.device)
    lib().l3_prefetch(t, r0, r1, GEMV_L3_WGS, s)


def gemv_supported(M: int, N: int, K: int, mode: int) -> bool:
    key = (M, N, K, mode)
    ok = _GEMV_OK.get(key)
    if ok is None:
        if not _GEMV_OK:  # first use: the launch knobs
            lib().gemv_set_ksplit(GEMV_KSPLIT)
            lib().gemv_set_wgs(GEMV_WGS)
        ok = _GEMV_OK[key] = bool(lib().gemv_supported(M, N, K, mode))
    return ok


def _gemv_ok(x, w, mode: int) -> bool:
    """A plain / SwiGLU projection of <= 2 rows goes to the decode GEMV (faster than the weight-
    streaming kernels at every decode shape measured: benchmarks/gemv_bench.py, profiles/r6_gemv/)."""
    M = x.shape[0]
    return (GEMV and M <= GEMV_MAX_M and x.dim() == 2 and x.dtype == torch.bfloat16 and w.dtype == torch.bfloat16
            and w.is_contiguous() and x.stride(-1) == 1
            and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0 and gemv_supported(M, w.shape[0], w.shape[1], mode))


def gemv_decode(mode: int, x, w, gamma=None, eps: float = 1e-5, res=None, positions=None, cos_sin=None,
                Hq: int = 0, Hkv: int = 0, D: int = 0, k_cache=None, v_cache=None, slots=None, neox: bool = True,
                po=None, pml=None, ctx=None, max_splits: int = 0, split: int = 0):
    """mode 0: x W^T; 1: ``res`` += x W^T in place (returned); 2: SwiGLU(x [Wg; Wu]^T) [M, N/2];
    3: packed QKV with RoPE applied to q (and to k in the paged cache, k kept unrotated in the
    row), K/V written at ``slots``.  ``gamma``: the GEMV's input is RMSNorm(x) * gamma.  ``po`` /
    ``pml`` (mode 1, GPU): x's rows that :func:`paged_decode` (``reduce=False``) left as split
    partials are merged in the GEMV's prologue (no decode_reduce launch)."""
    if use_hip(x):
        return lib().gemv_decode(mode, x, w, gamma, eps, res, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache,
                                 slots, neox, po, pml, ctx, max_splits, split)
    if po is not None:
        raise NotImplementedError("gemv_decode: the split-merge prologue is a GPU kernel")
    xin = ref.rmsnorm(x, gamma, eps) if gamma is not None else x
    y = xin.float() @ w.float().t()
    if mode == 0:
        return y.to(x.dtype)
    if mode == 1:
        res.copy_((y.to(res.dtype).float() + res.float()).to(res.dtype))
        return res
    if mode == 2:
        I = w.shape[0] // 2
        g, u = y[:, :I].to(x.dtype).float(), y[:, I:].to(x.dtype).float()
        return (torch.nn.functional.silu(g).to(x.dtype).float() * u).to(x.dtype)
    qkv = y.to(x.dtype)
    rope_kv_(qkv, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots, neox, False)
    return qkv


def splitk_rope_kv(part, positions, cos_sin, Hq: int, Hkv: int, D: int, k_cache, v_cache, slots, neox: bool,
                   write_k_inplace: bool = False):
    return lib().splitk_rope_kv(part, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots, neox, write_k_inplace)


def splitk_rmsnorm(part, residual, w, eps: float):
    """RMSNorm(bf16(sum of part's slabs) + residual) * w; residual updated in place."""
    return lib().splitk_rmsnorm(part, residual, w, eps)


def linear_add_rmsnorm(x, w, residual, norm_w, eps: float):
    """RMSNorm(x W^T + residual) * norm_w, with ``residual`` updated in place to
    x W^T + residual (the pre-norm block's "o / down projection -> add -> norm")."""
    plan = _ws_split_plan(x, w)
    if plan is not None and residual.is_contiguous():
        tk = ws_tickets(x.device) if WS_FUSED_TAIL and x.shape[0] <= 4 else None
        return lib().ws_linear_rmsnorm(x, w, residual, norm_w, eps, plan[0], plan[1], tk)
    return rmsnorm(linear(x, w), norm_w, eps, residual=residual)


def linear_rope_kv(x, w, positions, cos_sin, Hq: int, Hkv: int, D: int, k_cache=None, v_cache=None,
                   slots=None, neox: bool = True, write_k_inplace: bool = False):
    """qkv = x W^T, then :func:`rope_kv_` on it (one launch fewer on split-K decode shapes; on
    prefill-sized steps of a folded model -- interleaved RoPE, e.g. the tensor-parallel block,
    where the whole fused chain does not apply -- the QKV GEMM's epilogue does the RoPE and the
    paged-KV write).  Rows <= 2 (the tensor-parallel decode step at batch 1-2): the decode GEMV
    with its RoPE + paged-KV epilogue."""
    if (not write_k_inplace and k_cache is not None and slots is not None and _gemv_ok(x, w, 3)
            and w.shape[0] == (Hq + 2 * Hkv) * D):
        return lib().gemv_decode(3, x, w, None, 1e-5, None, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache,
                                 slots, neox)
    plan = _ws_split_plan(x, w)
    if plan is not None:
        # (rows <= 64: past that the last workgroup of a head reduces >= 128 KB of partials alone,
        # as long as the reduce kernel's whole launch)
        tk = ws_tickets(x.device) if WS_FUSED_TAIL and plan[0] == D == 128 and x.shape[0] <= 64 else None
        return lib().ws_linear_rope_kv(x, w, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots, neox,
                                       write_k_inplace, plan[0], plan[1], tk)
    if _qkv_epilogue_ok(x, w, neox, write_k_inplace, k_cache, slots):
        return linear_qkv_fused(x, w, None, 1e-5, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots)
    qkv = linear(x, w)
    rope_kv_(qkv, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots, neox, write_k_inplace)
    return qkv


def _qkv_epilogue_ok(x, w, neox: bool, write_k_inplace: bool, k_cache, slots) -> bool:
    if neox or write_k_inplace or not PREFILL_CHAIN or GEMM_LIBRARY or not _gemm_ok(x, w):
        return False
    if x.shape[0] <= WS_MAX_M or (k_cache is not None and slots is None):
        return False
    M, K = x.shape
    N = w.shape[0]
    c = _cfg_of(M, N, K, 0)
    return c is not None and c[2] == 1 and lib().gemm_supported(M, N, K, EPI_QKV, c[1], 1, c[0])


# ---------------------------------------------------------------- fused prefill chain
# Prefill-sized steps (M > WS_MAX_M rows) of a decoder whose norm weights are folded into its
# projections (LlamaModel.fold_norms) run the pre-norm block as four GEMMs and nothing else:
#   QKV     x_or_r W_qkv'^T  * s_in(row)  -> interleaved RoPE, K / V into the paged cache  (epi QKV)
#   O       r += attn W_o^T, partial sums of squares of r per 256 columns               (epi RESID)
#   gate_up silu / mul of r W_gu'^T * s_post(row)                                       (epi SWIGLU)
#   down    r += a W_down^T, partial sums of squares                                    (epi RESID)
# s(row) = rsqrt(sum of the partials / H + eps) is recomputed by each consumer tile from the
# producer's partials (no norm pass, no normalised activation in HBM, no RoPE / KV pass).
# LK_PREFILL_CHAIN=0 keeps the round-3 path (GEMM -> rmsnorm / rope_kv kernels).
PREFILL_CHAIN = os.environ.get("LK_PREFILL_CHAIN", "1") != "0"
EPI_RESID, EPI_QKV = 6, 7


def _cfg_of(M: int, N: int, K: int, epi: int):
    """(schedule / variant, bn, splits) of the prefill GEMM for this shape: the start-up tuned
    table (LK_GEMM_TUNE=1), else the shipped measurements (gemm_table_mi355x.json), else the
    fallback policy.  What start-up measured stays as it is for rows that make as many tiles; the rest by these very rows (``_fill_rule``)."""
    key = _gemm_key(M, N, K, epi)
    cfg = _GEMM_TABLE.get(key)
    if cfg is not None and _measured(M, N, K, epi) is not None:
        return cfg
    if cfg is None:
        cfg = _static_cfg(key)
        if cfg is not None and (not GEMM1W and cfg[0] in GEMM1W_BM):
            cfg = None
        elif cfg is not None and not SPLIT_ON and cfg[0] in GEMM1W_SPLIT:
            cfg = (3, 256, 1)
    return _fill_rule(M, N, epi, cfg if cfg is not None else _rounds_rule(M, N, K, epi) or _tile_rule(M, N, K, epi), K)


# Shapes without a measured entry, more than 256 rows: gemm1w.hip's 128 / 192 / 256-row tiles against the fallback.  Its
# waves of tiles cost 0.6 / 0.78 / 1.0 us per 64 columns of K each (128-row tiles from K 4096 on 1.1 of that) however few the tiles are, its
# start and end 4 / 5.5 / 6.5 us (GELU 2 / 3.5 / 4.5 more), and the output's stores 0.5 / 0.3 / 0.38 us per MB; gemm.hip's split-K with its
# reduction 16 + 8 f us and 0.8 + 0.8 f us per 64 columns of a range and 256 of N's tile (f: how much of the chip its workgroups
# fill), unsplit 8 us + 1.35 us per wave and 64 columns.  Measured, weights cold, fallback / the rule's pick (us):
#   3072 x 2048: M 320 26.5 / 27.2 (128-row tiles)   M 949 31.3 / 26.9   M 2048 41.5 / 29.9   M 2900 43.0 / 34.7 (192)   M 4096 47.8 / 46.3 (256)
#   2048 x 5632: M 1500 52.7 / same (128-row: 72.4)   M 2900 77.1 / 74.8 (128)   M 4096 96.9 / 79.4
#   1536 x 4096: M 1500 38.3 / same (128-row: 50.6)   M 2048 41.3 / same (51.8)   M 2900 54.4 / 51.1 (128)   M 4096 59.8 / 54.2
#   3072 x 768 GELU: M 949 22.4 / 15.0 (128)   M 2048 23.6 / 17.0   M 2900 25.7 / 22.7 (192)   768 x 3072: M 2048 30.6 / same (34.8)
#   11264 x 2048 SwiGLU: M 640 35.9 / 33.3 (128)   M 2048 99.7 / 81.6 (192)   M 2900 141.6 / 119.5   M 4096 156.9 / same (256)
#   8192 x 14336: M 640 159 / same (128-row: 195)   7168 x 6144: M 640 69.6 / same (87.4)   11264 x 512 GELU: M 2500 41.7 / 50.1 (192)
# Over 132 widths (N 768 - 11,264, K 512 - 14,336) at 12 row counts with three epilogues it takes 0.861 of the fallback's time, and 0.8 % more than
# the best of the four; 18 of the 4,752 picks are more than 8 % slower than the fallback, 20 % at most (the last shape above).
# v: (rows, start and end, per 64 columns, from K 4096 on, stores per MB, GELU)
_TILE_COST = {5: (128, 4.0, 0.6, 1.1, 0.5, 2.0), 4: (192, 5.5, 0.78, 1.0, 0.3, 3.5), 3: (256, 6.5, 1.0, 1.0, 0.38, 4.5)}
_TILE_RULE: dict = {}


def _tile_times(M: int, N: int, K: int, epi: int, d):
    """(us of a ``_TILE_COST`` variant, us of the fallback's choice ``d``), by the costs above."""
    cus, steps = device_cus(), K / 64
    out_mb = M * (N // 2 if epi == 1 else N) * 2 / 1e6

    def cost(v):
        bm, ends, c, deep, store, gelu = _TILE_COST[v]
        waves = -(-(-(-M // bm) * (N // 256)) // cus)
        return ends + (gelu if epi == 3 else 0) + waves * c * (deep if K >= 4096 else 1.0) * steps + store * out_mb

    if d[0] in _TILE_COST:
        return cost, cost(d[0])
    if d[2] > 1:
        f = min(1.0, -(-M // 256) * (N // d[1]) * d[2] / cus)
        return cost, 16 + 8 * f + (0.8 + 0.8 * f) * d[1] / 256 * steps / d[2]
    cols = N // 256 if epi == 1 else N // d[1]
    return cost, 8 + 1.35 * steps * -(-(-(-M // 256) * cols) // cus)


def _tiled_cost(M: int, N: int, K: int, epi: int) -> Optional[float]:
    """us that :func:`gemm` is estimated to take, or None where no tile takes the width."""
    d = _gemm_default(M, N, K, epi)
    if d is None or not (N % 256 == 0 or (epi != 1 and N % 192 == 0)):
        return None
    cost, other = _tile_times(M, N, K, epi, d)
    cfg = _cfg_of(M, N, K, epi)
    split = _split_rule(M, N, K, epi, cfg, 0)
    if split != cfg and split[2] > 1:
        # (the few-row kernel runs 10 - 20 % ahead of its estimate at these rows, and within a forward pass the sum's launch has a gap before it:
        # at 512 rows 2048 x 5632 28.7 split and 28.3 in it, 3072 x 2048 22.9 and 18.6)
        return 1.2 * (_split_cost(M, N, K, split[0], split[2]) + (2.5 if epi == 3 else 0))
    return cost(cfg[0]) if cfg is not None and cfg != d and cfg[0] in _TILE_COST else other


def _remember(table: dict, key, value):
    """table[key] = value in a table of bounded size, and the value back: a caller never reads the table again, which another thread may empty."""
    if len(table) > 4096:
        table.clear()
    table[key] = value
    return value


def _tile_rule(M: int, N: int, K: int, epi: int):
    d = _gemm_default(M, N, K, epi)
    # (past the rows it was fitted on a launch is several waves, whose stores overlap and which this cost does not describe: _rounds_rule)
    if not GEMM1W or not 256 < M <= 4608 or epi > 4 or K // 64 < 3 or N % 256 or d is None:
        return d
    key = (M, N, K, epi, d)
    pick = _TILE_RULE.get(key)
    if pick is not None:
        return pick
    cost, other = _tile_times(M, N, K, epi, d)
    best = min(_TILE_COST, key=cost)
    # (the pick has to be clear where the estimates are least sure: between two of these tiles 3 % of them, at K up to 1,024 7 %, and
    # against split-K 20 % from K 5,632 on, where 100 - 200 tiles of deep K run up to a quarter longer than estimated)
    if d[0] in _TILE_COST:
        clear = 0.93 if K <= 1024 else 0.97
    else:
        clear = 0.8 if d[2] > 1 and K >= 5632 else 1.0
    return _remember(_TILE_RULE, key, (best, 256, 1) if cost(best) < clear * other else d)


def _rounds_cost(M: int, N: int, bm: int) -> float:
    """Time of one K-tile over all rounds of ``bm`` x 256 tiles: a tile takes a + b * (share of the CUs at work beside it), with the constants
    of grouped_tile_rows in csrc/gemm.hip."""
    cus, f = device_cus(), bm / 256
    a, b = 1.41 * f - 0.17, 0.69 - 0.18 * f
    whole, part = divmod(-(-M // bm) * (N // 256), cus)
    return whole * (a + b) + (a + b * part / cus if part else 0.0)


_FILL_RULE: dict = {}


def _fill_cost(M: int, N: int, epi: int, v: int, K: int = 4096) -> float:
    """us that a variant's launches are estimated to differ by from another's: 0.71 of ``_rounds_cost`` per K-tile (of a column split the sum of its
    two launches, of which a short last round costs up to 0.3 more), 2 us per round of 256-row tiles for their ends, 2 us for a second launch."""
    cus, tn, steps = device_cus(), N // 256, K / 64

    def launch(bm, cols):
        return 0.71 * steps * _rounds_cost(M, cols * 256, bm) + 2.0 * bm / 256 * -(-(-(-M // bm) * cols) // cus)

    if v not in GEMM1W_SPLIT:
        return launch(GEMM1W_BM[v], tn)
    cols, bm = gemm1w_split_cols(M, N, epi, cus), GEMM1W_SPLIT[v]
    last = -(-M // bm) * (tn - cols) % cus
    return launch(256, cols) + launch(bm, tn - cols) + 2.0 + (0.71 * steps * 0.3 * (1 - last / cus) if last else 0.0)


def _fill_rule(M: int, N: int, epi: int, cfg, K: int = 4096):
    """A pick of 256 or 192-row tiles or of a column split, at this very number of rows: a table's entry was measured at the top of a bucket of
    256, and the rules above know no column split.  Another of the four where it is estimated to cost 1.5 % and 1 us less.  28,672 x 4,096 with SwiGLU:
    300 rows 84.2 -> 73.5 us (two tiles of either, 192 rows each), 949 rows 177.6 -> 167.0 (64 columns of 256 rows, the rest in 192), 1,100 rows
    234 -> 206; 10,496 x 2,048 at 4,095 rows 142.7 -> 135.4 (32 columns, the rest in 192); 14,336 x 4,096 at 2,589 248 -> 228.  Over 610 products (N 2,304 -
    28,672, K 192 - 4,096, 257 - 4,600 rows, three epilogues) it changes 233 of the picks before it, 15 to over 2 % slower (12 % the worst, 10,496 x 320), all to
    0.979 of their time on average.  By the rounds alone, without what a round and a launch cost whatever K is, 391 were changed and 61 slower,
    most by a column split at K up to 1,024: 6,144 x 192 with GELU at 4,099 rows 1.12, 11,264 x 1,024 at 3,733 1.16."""
    if cfg is None or cfg[0] not in (3, 4, 6, 7) or cfg[2] != 1 or not 256 < M <= 4608 or not GEMM1W or N % 256:
        return cfg
    key = (M, N, K, epi, cfg[0], device_cus(), SPLIT_ON)
    pick = _FILL_RULE.get(key)
    if pick is not None:
        return pick
    forms = (3, 4, 6, 7) if SPLIT_ON and _split_applies(M, N, epi) else (3, 4)
    costs = {v: _fill_cost(M, N, epi, v, K) for v in forms}
    best = min(costs, key=costs.get)
    # (a split that does not apply runs as 3)
    return _remember(_FILL_RULE, key, (best, 256, 1) if costs[best] + 1.0 < 0.985 * costs.get(cfg[0], costs[3]) else cfg)


def _rounds_rule(M: int, N: int, K: int, epi: int):
    """Tile of an unsplit product past the rows that ``_tile_rule`` covers, or None: 256 or 192 rows of gemm1w.hip by their rounds over the CUs
    alone, 192 where those take 3 % less.  Over 98 products (4,700 - 66,000 rows, N 768 - 28,672, K 768 - 5,632, four epilogues) the pick is
    1.3 % behind the better of the two.  Where N is a multiple of 192 the fallback takes gemm.hip's 192 columns, whose kernel needs 1.1 - 1.3
    times as long: 58,963 x 2304 x 768 248 -> 205 us, 8,925 x 2304 x 1536 70 -> 56, 44,104 x 768 x 768 65 -> 56, 5,500 x 3072 x 2048 89 -> 69."""
    if not GEMM1W or M <= 4608 or epi > 4 or K // 64 < 3 or N % 256 or (M + 256) * max(N, K) * 2 >= 0x7FFFFFF0:   # (its 32-bit offsets)
        return None
    d = _gemm_default(M, N, K, epi)
    if d is None or d[2] != 1:
        return None
    return (4, 256, 1) if _rounds_cost(M, N, 192) < 0.97 * _rounds_cost(M, N, 256) else (3, 256, 1)


# A plain, bias, activation or residual product of 257 - 4,608 rows may also run as 2 - 8 ranges of K on gemm1w.hip's tiles, f32 partials
# and a sum behind them.  Unsplit, N 2048 at 300 rows is 24 tiles of 128 rows on 256 CUs that each walk all of K; gemm.hip's
# split has 256-row tiles, four ranges at most and twice the time per 64 columns.  A round of workgroups costs a + f b us per 64 columns of its range
# (f: how much of the chip the launch fills), a further one c more, the launch 6.3 - 9.9 us, the sum 2.9 us and 0.46 us per range and MB of
# bf16 output: within 5.1 % (rms) of 20,000 launches, N 512 - 10,240, K 512 - 14,336.  An unsplit tile is left where that is 5 % less,
# gemm.hip's split for the best of all of these (it was the fastest of none).  Weights cold, before / the pick (us):
#   4096 x 4096: M 350 39.7 / 25.7 (4 of 128 rows)   M 512 41.6 / 31.6   M 1024 45.1 / 42.1 (2)   from M 1152 on the same (unsplit)
#   4096 x 14336: M 512 89.3 / 66.9 (4)   M 768 98.9 / 86.2 (4 of 192)   M 1024 115.2 / 106.0 (4 of 256)   M 1536 170 / 140 (2 of 192)
#   2048 x 5632: M 300 40.6 / 21.2 (8)   M 768 44.4 / 30.1 (4)   M 2048 63.3 / 51.0 (2)   M 3072 85.6 / 64.6 (1)
#   1024 x 4096: M 300 33.3 / 16.5 (8)   M 1024 35.8 / 22.9   M 3072 47.7 / 36.6 (2)      2048 x 2048: M 300 22.6 / 14.9 (4)   M 768 24.1 / 20.8 (3)
# Over the 1,325 products of two sweeps (one of them of random shapes) the picks take 0.9 % more than the best of all kernels, those before 28 %.
# v: (rows, start and end, a, b, c)
_SPLIT_COST = {5: (128, 6.3, 0.451, 0.319, 5.0), 4: (192, 8.1, 0.658, 0.357, 6.4), 3: (256, 9.9, 0.868, 0.409, 8.1)}
_SPLIT_RULE: dict = {}


def _split_cost(M: int, N: int, K: int, v: int, ks: int) -> float:
    bm, ends, a, b, c = _SPLIT_COST[v]
    cus = device_cus()
    wgs = -(-M // bm) * (N // 256) * ks
    rounds = -(-wgs // cus)
    return (ends + rounds * -(-(K // 64) // ks) * (a + b * wgs / (rounds * cus)) + (rounds - 1) * c
            + (2.9 + 0.46e-6 * ks * M * N * 2 if ks > 1 else 0.0))


def _split_costs(M: int, N: int, K: int) -> dict:
    return {(v, 256, ks): _split_cost(M, N, K, v, ks) for v in _SPLIT_COST for ks in (1, 2, 3, 4, 6, 8) if K // 64 >= 3 * ks}


def _split_takes(M: int, N: int, K: int, epi: int, ld: int) -> bool:
    return (GEMM1W and GEMM_SPLITK and 256 < M <= 4608 and epi in (0, 2, 3, 4) and N % 256 == 0 and K % 64 == 0
            and max(N, ld) * (M + 256) < 1 << 26 and N * K * 2 < 0x7FFFFFF0)


def _split_rule(M: int, N: int, K: int, epi: int, cfg, ld: int):
    """The pick ``cfg`` of :func:`_cfg_of`, or what the costs above take instead: (variant, 256, ranges of K).  ``ld``: the longest of the
    operands' row strides -- a split needs them whole within 32-bit offsets, where rows further apart go in chunks unsplit and in gemm.hip.
    Where start-up has measured, that decides."""
    if cfg is None or not 256 < M <= 4608 or not _split_takes(M, N, K, epi, ld):
        return cfg
    best = _measured(M, N, K, epi)
    if best is not None or cfg[0] in GEMM1W_SPLIT:
        return best or cfg
    key = (M, N, K, cfg)
    best = _SPLIT_RULE.get(key)
    if best is not None:
        return best
    costs = _split_costs(M, N, K)
    best = min(costs, key=costs.get, default=cfg)
    if cfg in costs and (best[2] == 1 or costs[best] > 0.95 * costs[cfg]):
        best = cfg
    return _remember(_SPLIT_RULE, key, best)


def _resid_cfg(M: int, N: int, K: int, ld: int = 0):
    c = _cfg_of(M, N, K, 0)
    if c is None or c[0] not in GEMM1W_BM:
        c = (c[0] if c is not None else _gemm_sched(K), 256, _gemm_splits(M, N, K, 0, 256))
    return _split_rule(M, N, K, 0, c, ld)


def prefill_chain_ok(x, w_qkv, w_o, w_gate_up, w_down) -> bool:
    """Whether a step of x.shape[0] rows can run the fused chain on the HIP kernels: prefill-sized,
    every projection on the hand-written GEMM, the QKV GEMM unsplit (its epilogue is in-kernel)."""
    if not (PREFILL_CHAIN and use_hip(x) and not GEMM_LIBRARY and x.dtype == torch.bfloat16):
        return False
    M = x.shape[0]
    if M <= WS_MAX_M:
        return False
    L = lib()
    N, K = w_qkv.shape
    c = _cfg_of(M, N, K, 0)
    if c is None or c[2] != 1 or not L.gemm_supported(M, N, K, EPI_QKV, c[1], 1, c[0]):
        return False
    N, K = w_gate_up.shape
    c = _cfg_of(M, N, K, 1)
    if c is None or c[2] != 1 or not L.gemm_supported(M, N, K, 1, c[1], 1, c[0]):
        return False
    for w in (w_o, w_down):
        N, K = w.shape
        sched, bn, ks = _resid_cfg(M, N, K)
        if not L.gemm_supported(M, N, K, EPI_RESID, bn, ks, sched):
            return False
    return True


def ss_buffer(M: int, N: int, device) -> torch.Tensor:
    """Partial sums of squares of a [M, N] residual: [N / 256, M] f32."""
    return torch.empty((N // 256, M), dtype=torch.float32, device=device)


def linear_resid(x, w, residual, ss_out):
    """residual += x W^T (bf16 rounding as the unfused linear -> add), and the partial sums of
    squares of the new residual per 256 columns into ss_out [N / 256, >= M] (one GEMM)."""
    if not use_hip(x):
        return ref.linear_resid(x, w, residual, ss_out)
    M, K = x.shape
    N = w.shape[0]
    sched, bn, ks = _resid_cfg(M, N, K, max(x.stride(0), residual.stride(0)))
    return lib().gemm_fused(x, w, EPI_RESID, bn, None, sched, ks, resid=residual, ss_out=ss_out)


def linear_swiglu_scaled(x, w_gate_up, ss, eps: float):
    """silu(s * x Wg^T) * (s * x Wu^T), s = the folded norm's per-row rsqrt from ``ss``."""
    if not use_hip(x):
        return ref.gemm_scaled(x, w_gate_up, ss, x.shape[1], eps, swiglu=True)
    M, K = x.shape
    N = w_gate_up.shape[0]
    sched, bn, _ = _cfg_of(M, N, K, 1)
    return lib().gemm_fused(x, w_gate_up, 1, bn, None, sched, 1, ss_in=ss, eps=eps)


def linear_qkv_fused(x, w, ss, eps: float, positions, cos_sin, Hq: int, Hkv: int, D: int,
                     k_cache=None, v_cache=None, slots=None):
    """qkv = s * x W^T (ss None: unscaled), interleaved-pair RoPE on q / k, K / V into the paged
    cache: the QKV projection, the input norm's scale and rope_kv_ in one GEMM."""
    if not use_hip(x):
        return ref.qkv_fused(x, w, ss, x.shape[1], eps, positions, cos_sin, Hq, Hkv, D, k_cache, v_cache, slots)
    M, K = x.shape
    N = w.shape[0]
    sched, bn, _ = _cfg_of(M, N, K, 0)
    return lib().gemm_fused(x, w, EPI_QKV, bn, None, sched, 1, ss_in=ss, eps=eps, positions=positions,
                            cos_sin=cos_sin, slots=slots, k_cache=k_cache, v_cache=v_cache, hq=Hq, hkv=Hkv, hd=D)


# ---------------------------------------------------------------- per-step gathers (csrc/step_ops.hip)
def embed_rows(table, ids, lo: int = 0, n_local: Optional[int] = None):
    """Rows of ``table`` for int32 ``ids``; with ``lo`` / ``n_local`` a vocab-parallel shard:
    ids outside [lo, lo + n_local) give zero rows (summed over the TP group afterwards)."""
    whole = lo == 0 and n_local is None
    n_local = table.shape[0] if n_local is None else n_local
    if use_hip(table) and ids.dtype == torch.int32:
        # the whole table: an out-of-range id is counted on the device (lib().embed_errors(),
        # polled by the engine's health check) instead of becoming a silent zero row
        return lib().embed_rows(table, ids.contiguous(), lo, -1 if whole else n_local)
    if whole:
        return table[ids.long()]  # raises on a bad id, like an nn.Embedding lookup
    local = ids.long() - lo
    mask = (local < 0) | (local >= n_local)
    return table[local.clamp(0, max(0, n_local - 1))].masked_fill(mask[:, None], 0)


def set_ids(ids, host):
    """ids (int32) = host (CPU int32); on the GPU a few travel in a launch's own arguments, without a pinned copy."""
    if not (use_hip(ids) and lib().set_ids(ids, host)):
        ids.copy_(host.pin_memory() if ids.is_cuda else host, non_blocking=True)


def scatter_ids(ids, dst, prev, src):
    """ids[dst] = prev[src] (the in-flight decode inputs of a pipelined step), one launch."""
    if use_hip(ids) and ids.dtype == torch.int32 and prev.dtype == torch.int32:
        lib().scatter_ids(ids, dst.contiguous(), prev.contiguous(), src.contiguous())
        return ids
    ids.index_copy_(0, dst, prev.index_select(0, src).to(ids.dtype))
    return ids


def gather_rows(x, idx):
    """x[idx] (rows), one launch on the GPU."""
    if (use_hip(x) and x.dtype == torch.bfloat16 and idx.dtype == torch.int64 and x.dim() == 2
            and x.stride(-1) == 1 and x.shape[1] % 8 == 0 and x.stride(0) % 8 == 0 and x.data_ptr() % 16 == 0):
        return lib().gather_rows(x, idx.contiguous())
    return x.index_select(0, idx)


def softmax_scale(D: int) -> float:
    return 1.0 / math.sqrt(D)
