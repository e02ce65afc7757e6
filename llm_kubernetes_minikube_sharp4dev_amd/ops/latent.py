"""Entry points of attention over a cached latent (``csrc/latent_attn.hip``, ``csrc/head_linear.hip``): a token's cache row is
``[latent c | zeros | rotated key part | zeros]``, common to all query heads and to every layer that reads it.  A head's key
``[W_uk c | common part]`` and value ``W_uv c`` are never formed: its query goes through ``W_uk^T`` once (so the score is a dot
product with the cache row), and the softmax average of the latents goes through ``W_uv`` afterwards.

    s(i, j) = scale * <[W_uk^T q | rotated q]_i, row_j>     for first(i) <= j <= i
    p(i, j) = exp(s(i, j)) / (exp(sink_h) + sum_j' exp(s(i, j')))          out_i = W_uv sum_j p(i, j) c_j

Cache ``[blocks, BS, KD]`` in the activation dtype, ``KD = RP + RDP`` (``latent_row``).  GPU tensors go to the HIP kernels, CPU
tensors to the torch implementations below.
"""
from __future__ import annotations

import torch

from ._ext import lib, use_hip

__all__ = ["latent_row", "latent_prep", "latent_query_rot", "latent_query", "head_linear", "latent_attention_prefill", "latent_attention_decode",
           "latent_decode_splits"]


def latent_row(kv_rank: int, rot_dim: int) -> tuple:
    """(RP, RDP): columns of a cache row that hold the latent and the rotated part, padded to the kernels' sizes."""
    rp = next((p for p in (128, 256, 512) if kv_rank <= p), -(-kv_rank // 64) * 64)
    rdp = next((p for p in (64, 128) if rot_dim <= p), -(-rot_dim // 64) * 64)
    return rp, rdp


def _rotate_pairs(x, positions, freq, rd: int, adjacent: bool = False, mag: float = 1.0):
    """x f32 [T, ..., rd]: dimension i pairs with i + rd / 2 (``adjacent``: 2 i with 2 i + 1), angle position * freq[i], cos and sin
    times ``mag``."""
    half = rd // 2
    ang = positions.float().view(-1, *([1] * (x.dim() - 1))) * freq.float()[:half]
    c, s = torch.cos(ang) * mag, torch.sin(ang) * mag
    u, v = (x[..., 0:rd:2], x[..., 1:rd:2]) if adjacent else (x[..., :half], x[..., half:rd])
    y = (u * c - v * s, v * c + u * s)
    return torch.stack(y, -1).flatten(-2) if adjacent else torch.cat(y, -1)


def latent_prep(u, dq_col: int, q_rank: int, dq_norm, dkv_col: int, kv_rank: int, dkv_norm, rot_dim: int, freq, positions, eps: float,
                cache, slots, rp: int, adjacent: bool = False, mag: float = 1.0):
    """cq [T, q_rank] = the columns ``[dq_col, dq_col + q_rank)`` of ``u`` divided by their RMS times ``dq_norm`` (f32 arithmetic).
    With ``dkv_norm`` (None: this layer reads another layer's cache) also the token's cache row at ``slots`` (< 0: none): the
    normed latent of the columns behind ``dkv_col`` and the ``rot_dim`` columns that follow, rotated by position (``adjacent`` pairs or halves; cos and
    sin times ``mag``)."""
    if use_hip(u):
        return lib().latent_prep(u, int(dq_col), int(q_rank), dq_norm, int(dkv_col), int(kv_rank), dkv_norm, int(rot_dim), freq, positions,
                                 float(eps), cache, slots, int(rp), bool(adjacent), float(mag))
    T = u.shape[0]

    def rms(x, w):
        return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + eps) * w

    cq = rms(u[:, dq_col:dq_col + q_rank].float(), dq_norm).to(u.dtype)
    if dkv_norm is not None:
        row = torch.zeros(T, cache.shape[2], dtype=torch.float32, device=u.device)
        row[:, :kv_rank] = rms(u[:, dkv_col:dkv_col + kv_rank].float(), dkv_norm)
        kr = u[:, dkv_col + kv_rank:dkv_col + kv_rank + rot_dim].float()
        row[:, rp:rp + rot_dim] = _rotate_pairs(kr, positions[:T], freq, rot_dim, adjacent, mag)
        BS = cache.shape[1]
        sl = slots[:T].long()
        ok = sl >= 0
        cache[sl[ok] // BS, sl[ok] % BS] = row[ok].to(cache.dtype)
    return cq


def latent_query_rot(q, qa, H: int, qdim: int, dim: int, rot_dim: int, freq, positions, rp: int, adjacent: bool = False, mag: float = 1.0):
    """Rotated parts of the queries: ``q`` rows hold H heads of ``qdim`` columns, ``[dim plain | rot_dim | padding]``; their rotated
    columns go to ``qa[..., rp : rp + rot_dim]`` (``qa`` [T, H, KD]), zeros behind them."""
    if use_hip(q):
        lib().latent_query(q, None, qa, int(H), int(qdim), int(dim), int(rot_dim), freq, positions, int(rp), bool(adjacent), float(mag))
        return qa
    T = q.shape[0]
    r = q[:, : H * qdim].view(T, H, qdim)[..., dim:dim + rot_dim].float()
    qa[..., rp:] = 0
    qa[..., rp:rp + rot_dim] = _rotate_pairs(r, positions[:T], freq, rot_dim, adjacent, mag).to(qa.dtype)
    return qa


def head_linear(x, w, x_head: int, out, parts: int = 1):
    """Per-head products: ``out[t, h, :N] = w[h] x[t, h * x_head : h * x_head + K]`` for ``w`` [H, N, K] and ``out`` [T, H, >= N]
    (a view whose last dimension is contiguous); f32 accumulation.  ``parts`` 2 (bf16): the K columns behind those add to them, an
    operand that is kept in two bf16 parts."""
    if use_hip(x):
        lib().head_linear(x, w, int(x_head), out, int(parts))
        return out
    H, N, K = w.shape
    T = x.shape[0]
    xs = torch.stack([x[:, h * x_head:h * x_head + parts * K].float().view(T, parts, K).sum(1) for h in range(H)], 0)   # [H, T, K]
    out[..., :N] = torch.bmm(xs, w.float().transpose(1, 2).contiguous()).transpose(0, 1).to(out.dtype)
    return out


def latent_query(q, w, qa, qdim: int, dim: int, rot_dim: int, freq, positions, rp: int, adjacent: bool = False, mag: float = 1.0):
    """Attention queries over a cached latent in one launch: ``qa[t, h, :rp] = w[h] q[t, h * qdim : h * qdim + K]`` for ``w`` [H, rp, K]
    (:func:`head_linear`) and the rotated part behind them (:func:`latent_query_rot`)."""
    if use_hip(q):
        lib().latent_query(q, w, qa, int(w.shape[0]), int(qdim), int(dim), int(rot_dim), freq, positions, int(rp), bool(adjacent), float(mag))
        return qa
    head_linear(q, w, qdim, qa)
    return latent_query_rot(q, qa, w.shape[0], qdim, dim, rot_dim, freq, positions, rp, adjacent, mag)


def latent_decode_splits(B: int, H: int, span: int) -> int:
    """Workgroups per (sequence, head block) of the decode kernel: about one workgroup per CU, never more than one per 128 keys."""
    blocks = max(1, B * -(-H // 16))
    return int(max(1, min(256 // blocks if blocks <= 256 else 1, -(-span // 128))))


def _rows(qa, kv, qpos, window: int, scale: float, sink, rp: int):
    """qa f32 [S, H, KD] at positions qpos [S]; kv f32 [n, KD] at positions 0 .. n - 1 -> [S, H, rp]."""
    s = torch.einsum("ihd,jd->hij", qa, kv) * scale
    j, i = torch.arange(kv.shape[0], device=kv.device).view(1, -1), qpos.view(-1, 1)
    seen = j <= i
    if window > 0:
        seen = seen & (i - j < window)
    s = s.masked_fill(~seen[None], float("-inf"))
    m = s.amax(-1, keepdim=True)
    if sink is not None:
        m = torch.maximum(m, sink.view(-1, 1, 1))
    e = torch.exp(s - m)
    den = e.sum(-1, keepdim=True) + (torch.exp(sink.view(-1, 1, 1) - m) if sink is not None else 0.0)
    return torch.einsum("hij,jd->ihd", e / den, kv[:, :rp])


def _gather(cache, table, n):
    BS = cache.shape[1]
    return cache[table[: (n + BS - 1) // BS].long()].reshape(-1, cache.shape[2])[:n].float()


def _put(out, v, rp: int):
    out[..., :rp] = v.to(out.dtype)
    if out.shape[-1] > rp:
        out[..., rp:] = (v - out[..., :rp].float()).to(out.dtype)


def latent_attention_prefill(qa, cache, block_tables, cu_q, ctx_lens, window: int, scale: float, sink, rp: int, out, max_len: int, gate=None):
    """Query chunks over their sequences' cached rows (their own included).  ``qa`` [T, H, KD]; ``sink`` f32 [H] or None; ``window`` 0:
    causal; ``out`` [T, H, rp] receives the averaged latents (head h times ``sigmoid(gate[:, h])`` with a ``gate`` [T, H]).  With
    ``out`` [T, H, 2 rp] (bf16) they come in two parts, the rounded value and the rest behind it."""
    if use_hip(qa):
        lib().latent_attn_prefill(qa, cache, block_tables, cu_q, ctx_lens, int(window), float(scale), sink, int(rp), out, int(max_len), gate)
        return out
    cu = cu_q.tolist()
    for b in range(len(cu) - 1):
        s0, s1 = cu[b], cu[b + 1]
        n = int(ctx_lens[b])
        r = _rows(qa[s0:s1].float(), _gather(cache, block_tables[b], n), torch.arange(n - (s1 - s0), n, device=qa.device), window, scale,
                  sink, rp)
        _put(out[s0:s1], r if gate is None else r * torch.sigmoid(gate[s0:s1, : r.shape[1], None].float()), rp)
    return out


def latent_attention_decode(qa, cache, block_tables, ctx_lens, window: int, scale: float, sink, rp: int, out, splits: int = 1, gate=None):
    """One query row per sequence at its last position (ctx - 1).  ``gate`` and an ``out`` in two parts: as in :func:`latent_attention_prefill`."""
    if use_hip(qa):
        lib().latent_attn_decode(qa, cache, block_tables, ctx_lens, window, float(scale), sink, int(rp), out, int(splits), gate)
        return out
    for b in range(qa.shape[0]):
        n = int(ctx_lens[b])
        if n < 1:
            continue
        r = _rows(qa[b:b + 1].float(), _gather(cache, block_tables[b], n), torch.tensor([n - 1], device=qa.device), window, scale, sink, rp)
        _put(out[b:b + 1], r if gate is None else r * torch.sigmoid(gate[b:b + 1, : r.shape[1], None].float()), rp)
    return out
