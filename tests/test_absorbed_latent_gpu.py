"""Windowed latent attention on the cached latent (``LatentAttnSpec.absorb``) against the float64 oracle and against
the same mixer over expanded keys and values: whole prompts, portions and decode rows, head counts that do and do not
fill a block of 16, ranks and rotated parts with and without padding, adjacent rotation pairs with a magnitude, gates."""
import pytest
import torch

from test_fusasun_mixers import one_layer, q16, rnd, run_mixer, step_meta, want_mixer

YARN = {"base": 1000.0, "scaling": {"factor": 4.0, "original": 64, "fast": 4.0, "slow": 1.0}}


def err(got, want):
    return float((got.double() - want).norm() / want.norm())


def mixer(H, dim, rd, vdim, q_rank, kv_rank, window):
    return {"heads": H, "dim": dim, "rot_dim": rd, "vdim": vdim, "q_rank": q_rank, "kv_rank": kv_rank, "scale": (dim + rd) ** -0.5,
            "mask": {"size": window}, "rot": dict(YARN, dims=rd)}


@pytest.mark.gpu
@pytest.mark.parametrize("H,dim,rd,vdim,q_rank,kv_rank,window,T", [
    (16, 128, 64, 128, 96, 512, 24, 70), (16, 50, 10, 40, 32, 100, 33, 90), (20, 52, 8, 44, 40, 128, 16, 65), (40, 96, 32, 64, 64, 256, 300, 150)])
def test_absorbed_mixer(H, dim, rd, vdim, q_rank, kv_rank, window, T):
    mx = mixer(H, dim, rd, vdim, q_rank, kv_rank, window)
    m, sd = one_layer("latent_attention", mx, 64, "cuda", torch.bfloat16, taps=2)
    M = m.layers[0].mix
    assert M.spec.absorbed and len(m.make_caches(2, 16, 1)[0]) == 2          # the latent rows and the convolution state
    h = q16(rnd(torch.Generator().manual_seed(3), T, 64))
    want = want_mixer("latent_attention", h, mx, sd)
    cuts = ([T], [T - 40, 1, 30], [5])
    absorbed = [err(run_mixer(m, h, c, "cuda", torch.bfloat16), want) for c in cuts]
    M.spec.absorbed = False
    expanded = [err(run_mixer(m, h, c, "cuda", torch.bfloat16), want) for c in cuts]
    print(H, dim, kv_rank, "absorbed", absorbed, "expanded", expanded)
    # both round five times on the way to the output projection (query latent, query, key side, averages, output): the same size of
    # error; T x W outputs of independent roundings leave a few per cent between two such figures
    assert max(absorbed) <= 1.1 * max(expanded) and max(absorbed) < 1.5e-2


def attention_of(M, u, T):
    """The gated averages from the down projections ``u``, in float64 and without any rounding on the way."""
    s, H, u = M.spec, M.spec.heads, u.double()
    rms = lambda x, w: x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w.double()
    dq, dkv, g = (M.rows.off[k] for k in ("dq", "dkv", "g"))
    c = rms(u[:, dkv:dkv + s.kv_rank], M.dkv_norm)
    q = (rms(u[:, dq:dq + s.q_rank], M.dq_norm) @ M.w_uq.double().T).view(T, H, -1)
    ang = torch.arange(T, device=u.device).double()[:, None] * M.freq.double()[None, :s.rot_dim // 2]
    cs, sn = ang.cos() * s.rot.magnitude, ang.sin() * s.rot.magnitude

    def turn(x, cs, sn):
        a, b = x[..., 0::2], x[..., 1::2]
        return torch.stack([a * cs - b * sn, b * cs + a * sn], -1).flatten(-2)

    qr = turn(q[..., s.dim:s.dim + s.rot_dim], cs[:, None], sn[:, None])
    kr = turn(u[:, dkv + s.kv_rank:dkv + s.kv_rank + s.rot_dim], cs, sn)
    w = M.w_ukv.double()
    k = (c @ w[:H * s.dim].T).view(T, H, s.dim)
    v = (c @ w[M.up_rows.off["uv"]:][:H * s.vdim_p].T).view(T, H, s.vdim_p)
    sc = (torch.einsum("thd,jhd->htj", q[..., :s.dim], k) + torch.einsum("thr,jr->htj", qr, kr)) * s.scale
    i = torch.arange(T, device=u.device)
    sc = sc.masked_fill(~((i[None] <= i[:, None]) & (i[:, None] - i[None] < s.window)), float("-inf"))
    return torch.einsum("htj,jhv->thv", sc.softmax(-1), v) * torch.sigmoid(u[:, g:g + H, None])


@pytest.mark.gpu
@pytest.mark.parametrize("H,dim,rd,vdim,q_rank,kv_rank,window", [(16, 128, 64, 128, 96, 512, 64), (32, 128, 64, 128, 96, 512, 200), (16, 64, 32, 64, 64, 128, 33)])
def test_absorbed_attention_is_as_exact(monkeypatch, H, dim, rd, vdim, q_rank, kv_rank, window):
    """Behind the same down projections the cached latent's gated averages are no further from float64 than those over expanded keys and
    values: W_uv takes the averages in two bf16 parts, so they are rounded once (the output), where expanded values are rounded twice."""
    from llm_kubernetes_minikube_sharp4dev_amd.models import fusasun
    mx = mixer(H, dim, rd, vdim, q_rank, kv_rank, window)
    T = 2 * window + 40
    m, _ = one_layer("latent_attention", mx, 64, "cuda", torch.bfloat16, taps=2)
    M = m.layers[0].mix
    h = q16(rnd(torch.Generator().manual_seed(3), T, 64))
    fn, calls = fusasun.latent_window_attention, []
    monkeypatch.setattr(fusasun, "latent_window_attention", lambda u, *a, **k: calls.append((u.clone(), fn(u, *a, **k))) or calls[-1][1])
    errs = []
    for cuts in ([T], [T - 20]):
        for absorbed in (True, False):
            M.spec.absorbed = absorbed
            calls.clear()
            run_mixer(m, h, cuts, "cuda", torch.bfloat16)
            u, got = torch.cat([c[0] for c in calls]), torch.cat([c[1] for c in calls])
            errs.append(err(got.view(T, H, -1), attention_of(M, u, T)))
    print(errs)
    assert errs[0] <= errs[1] and errs[2] <= errs[3]


@pytest.mark.parametrize("dtype,device,change", [
    (torch.float32, "cuda", {}), (torch.bfloat16, "cpu", {}), (torch.bfloat16, "cuda", {"kv_rank": 600}), (torch.bfloat16, "cuda", {"dim": 96}), (torch.bfloat16, "cuda", {"heads": 4}),
    (torch.bfloat16, "cuda", {"rot_dim": 0}), (torch.bfloat16, "cuda", {"rot_dim": 130})])
def test_absorb_rule(dtype, device, change):
    from llm_kubernetes_minikube_sharp4dev_amd.models.window_attention import LatentAttnSpec
    from dataclasses import replace
    s = LatentAttnSpec.from_dict(mixer(16, 128, 64, 128, 96, 512, 24))
    assert s.absorb(torch.bfloat16, "cuda") and s.absorb(torch.bfloat16, torch.device("cuda", 0))
    assert not replace(s, **change).absorb(dtype, device)
    assert not replace(s, window=0).absorb(torch.bfloat16, "cuda") and not replace(s, gate_elem=True).absorb(torch.bfloat16, "cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T", [1, 16, 17, 33, 65, 129, 200])
@pytest.mark.parametrize("H,dim,rd,qdim,K,rp,kd,adjacent", [(3, 12, 6, 24, 16, 40, 64, True), (2, 128, 64, 192, 128, 512, 576, False),
                                                          (16, 44, 10, 56, 48, 128, 192, True), (2, 20, 8, 28, 20, 72, 80, False)])
def test_latent_query(T, H, dim, rd, qdim, K, rp, kd, adjacent, dtype):
    """Products and rotated part of one launch, over the row tiles of both kernels, against float64; nothing outside is touched."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    g = torch.Generator().manual_seed(T + H)
    q, w = q16(rnd(g, T, H * qdim)), q16(rnd(g, H, rp, K, scale=K ** -0.5))
    freq = torch.tensor([30.0 ** (-2.0 * i / rd) for i in range(rd // 2)], dtype=torch.float32)
    pos = torch.randint(0, 3000, (T,), generator=g, dtype=torch.int32)
    buf = torch.full((T + 1, H, kd), 7.0, dtype=dtype, device="cuda")
    ops.latent_query(q.to(dtype).cuda(), w.to(dtype).cuda(), buf[:T], qdim, dim, rd, freq.cuda(), pos.cuda(), rp, adjacent=adjacent, mag=1.2)
    qh = q.view(T, H, qdim)
    ang = pos.double()[:, None, None] * freq.double()
    c, s = ang.cos() * 1.2, ang.sin() * 1.2
    r = qh[..., dim:dim + rd]
    a, b = (r[..., 0::2], r[..., 1::2]) if adjacent else (r[..., :rd // 2], r[..., rd // 2:])
    rot = (a * c - b * s, b * c + a * s)
    rot = torch.stack(rot, -1).flatten(-2) if adjacent else torch.cat(rot, -1)
    want = torch.cat([torch.einsum("thk,hnk->thn", qh[..., :K], w), rot, torch.zeros(T, H, kd - rp - rd, dtype=torch.float64)], -1)
    # f32: angles up to 3000 are 2^-13 apart in f32, times values of at most 5; bf16: half a step of the result
    got, atol = buf[:T].double().cpu(), 5 * 1.2 * 2 ** -12
    assert bool(((got - want).abs() <= atol + (2 ** -8 if dtype == torch.bfloat16 else 2 ** -18) * want.abs()).all())
    assert bool((buf[T] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rp,rdp", [(512, 64), (512, 128), (256, 64), (128, 128)])
@pytest.mark.parametrize("H,lens,past,window,loud", [(16, [1, 3, 4, 5], [0, 40, 31, 32], 24, False), (16, [70, 33], [0, 7], 0, False), (5, [29, 8], [3, 64], 33, True),
                                                    (40, [65], [17], 48, False), (1, [130, 64], [0, 1], 512, True)])
def test_prompt_rows(rp, rdp, H, lens, past, window, loud):
    """Prompt portions behind cached rows on both prompt kernels: queries per workgroup that do and do not divide a portion, heads that do and do not
    fill a block, windows inside and across 32-key tiles, a sink, gates; loud: later keys so far above the first tile's that the pass is
    repeated.  Against float64."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    g = torch.Generator().manual_seed(rp + H)
    BS, kd, T = 16, rp + rdp, sum(lens)
    blocks = [-(-(n + p) // BS) for n, p in zip(lens, past)]
    cache, q = q16(rnd(g, sum(blocks) + 2, BS, kd)), q16(rnd(g, T, H, kd, scale=0.3))
    order = torch.randperm(sum(blocks) + 2, generator=g)[:sum(blocks)].int()
    table, at = torch.zeros(len(lens), max(blocks), dtype=torch.int32), 0
    for i, n in enumerate(blocks):
        table[i, :n] = order[at:at + n]
        at += n
    if loud:   # the last keys of every sequence point along its last query's
        for i, (n, p) in enumerate(zip(lens, past)):
            for k in range(max(0, n + p - 6), n + p):
                cache[table[i, k // BS].long(), k % BS] = q16(q[sum(lens[:i + 1]) - 1, 0] * 60)
    gate, sink = q16(rnd(g, T, H)), rnd(g, H).float()
    out = torch.full((T + 1, H, 2 * rp), 7.0, dtype=torch.bfloat16, device="cuda")
    cu = torch.tensor([0] + lens).cumsum(0).int().cuda()
    ctx = torch.tensor([n + p for n, p in zip(lens, past)]).int().cuda()
    ops.latent_attention_prefill(q.bfloat16().cuda(), cache.bfloat16().cuda(), table.cuda(), cu, ctx, window, kd ** -0.5, sink.cuda(), rp, out[:T], max(lens),
                                 gate=gate.bfloat16().cuda())
    got, t0 = out[:T, :, :rp].double().cpu() + out[:T, :, rp:].double().cpu(), 0
    for i, (n, p) in enumerate(zip(lens, past)):
        rows = cache[table[i, :blocks[i]].long()].reshape(-1, kd)[:n + p].double()
        s = torch.einsum("qhd,kd->hqk", q[t0:t0 + n].double(), rows) * kd ** -0.5
        qi, ki = torch.arange(p, p + n)[:, None], torch.arange(n + p)[None]
        s = s.masked_fill(((ki > qi) | ((ki <= qi - window) if window else torch.zeros_like(ki, dtype=torch.bool)))[None], float("-inf"))
        s = torch.cat([sink.double().view(H, 1, 1).expand(H, n, 1), s], -1)
        w = s.softmax(-1)[..., 1:]
        want = torch.einsum("hqk,kd->qhd", w, rows[:, :rp]) * torch.sigmoid(gate[t0:t0 + n].double())[..., None]
        size = torch.einsum("hqk,kd->qhd", w, rows[:, :rp].abs())
        # weights rounded to bf16 (2^-9), scores in f32: up to kd products of the size of the row's largest score
        big = float(s[s.isfinite()].abs().max())
        assert bool(((got[t0:t0 + n] - want).abs() <= (2.0 ** -8 + big * 2.0 ** -18) * size + 1e-5).all()), float(((got[t0:t0 + n] - want).abs() / (size + 1e-9)).max())
        t0 += n
    assert bool((out[T] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("splits", [1, 2, 4, 5, 70])
def test_decode_splits_agree_with_gates(splits):
    """One query row per sequence over any number of key splits, gated: against float64."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    g = torch.Generator().manual_seed(5)
    B, H, rp, rdp, BS, n = 3, 16, 128, 64, 16, 150
    qa, cache = q16(rnd(g, B, H, rp + rdp, scale=0.3)), q16(rnd(g, 40, BS, rp + rdp))
    table = torch.randperm(40, generator=g)[:30].view(3, 10).int()
    ctx = torch.tensor([150, 1, 77], dtype=torch.int32)
    gate = q16(rnd(g, B, H + 8, scale=3.0))
    out = torch.zeros(B, H, rp, dtype=torch.bfloat16, device="cuda")
    b16 = lambda t: t.to(torch.bfloat16).cuda()
    ops.latent_attention_decode(b16(qa), b16(cache), table.cuda(), ctx.cuda(), 100, 0.1, None, rp, out, splits=splits, gate=b16(gate)[:, 8:])
    for b in range(B):
        kv = cache[table[b].long()].reshape(-1, rp + rdp)[max(0, int(ctx[b]) - 100):int(ctx[b])]
        p = ((qa[b] @ kv.T) * 0.1).softmax(-1)
        want = (p @ kv[:, :rp]) * torch.sigmoid(gate[b, 8:, None])
        assert float((out[b].double().cpu() - want).abs().max()) < 2 ** -7 * float(want.abs().max())


@pytest.mark.gpu
@pytest.mark.parametrize("rows,splits", [(1, 1), (3, 4), (0, 0)])
@pytest.mark.parametrize("rp", [128, 512, 64])
def test_averages_in_two_parts(rows, splits, rp):
    """The same averages rounded once and as value and rest (decode rows in one and several splits, a prompt; the matrix kernels and, at
    rank 64, the plain one): the first part is the rounded one, the rest is at most half a step of it and not all zero."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    g = torch.Generator().manual_seed(rp + rows)
    B, H, rdp, n = 3, 16, 64, 150
    b16 = lambda t: t.to(torch.bfloat16).cuda()
    cache, table = b16(q16(rnd(g, 40, 16, rp + rdp))), torch.randperm(40, generator=g)[:30].view(3, 10).int().cuda()
    ctx = torch.tensor([n, 33, 77], dtype=torch.int32, device="cuda")
    T = B if rows else 60
    qa, gate = b16(rnd(g, T, H, rp + rdp, scale=0.3)), b16(rnd(g, T, H))
    one, two = (torch.full((T, H, w), 7.0, dtype=torch.bfloat16, device="cuda") for w in (rp, 2 * rp))
    for out in (one, two):
        if rows:
            ops.latent_attention_decode(qa, cache, table, ctx, 100, 0.1, None, rp, out, splits=splits, gate=gate)
        else:
            cu = torch.tensor([0, 20, 40, 60], dtype=torch.int32, device="cuda")
            ops.latent_attention_prefill(qa, cache, table, cu, ctx, 100, 0.1, None, rp, out, 20, gate=gate)
    assert torch.equal(two[..., :rp], one)
    rest = two[..., rp:].float()
    assert bool((rest.abs() <= 2 ** -8 * one.float().abs()).all()) and float((rest != 0).float().mean()) > 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [1, 17, 40, 129, 300])
@pytest.mark.parametrize("H,N,K", [(16, 128, 512), (3, 40, 128), (2, 64, 50), (2, 36, 72)])
def test_head_products_of_two_parts(rows, H, N, K):
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    g = torch.Generator().manual_seed(rows + K)
    v, w = rnd(g, rows, H, K).double(), q16(rnd(g, H, N, K, scale=K ** -0.5))
    hi = v.bfloat16()
    lo = (v - hi.double()).bfloat16()
    out = torch.full((rows, H, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.head_linear(torch.cat([hi, lo], -1).view(rows, -1).cuda(), w.bfloat16().cuda(), 2 * K, out, parts=2)
    want = torch.einsum("thk,hnk->thn", hi.double() + lo.double(), w)
    # half a step of the result, f32 sums of 2 K terms
    assert bool(((out.double().cpu() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("rows", [16, 33, 63, 64, 65, 127, 128])
@pytest.mark.parametrize("H,N", [(16, 128), (40, 128), (130, 128)])   # one, two and four 16-row tiles per workgroup among the rows
@pytest.mark.parametrize("parts", [1, 2])
def test_head_products_row_tiles(rows, H, N, parts):
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    K = 64
    g = torch.Generator().manual_seed(rows + H)
    x, w = q16(rnd(g, rows, H, parts, K)), q16(rnd(g, H, N, K, scale=K ** -0.5))
    buf = torch.full((rows + 1, H, N), 7.0, dtype=torch.bfloat16, device="cuda")
    ops.head_linear(x.reshape(rows, -1).bfloat16().cuda(), w.bfloat16().cuda(), parts * K, buf[:rows], parts=parts)
    want = torch.bmm(x.double().sum(2).transpose(0, 1), w.double().transpose(1, 2).contiguous()).transpose(0, 1)
    assert bool(((buf[:rows].double().cpu() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all())   # as above
    assert bool((buf[rows] == 7.0).all())


@pytest.mark.gpu
def test_head_products_of_many_columns():
    """More 32-column workgroups than a grid's second dimension has places."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    N, K = 32 * 65536 + 40, 8
    g = torch.Generator(device="cuda").manual_seed(1)
    x, w = torch.randn(2, K, generator=g, device="cuda").bfloat16(), torch.randn(1, N, K, generator=g, device="cuda").bfloat16()
    out = torch.empty(2, 1, N, dtype=torch.bfloat16, device="cuda")
    ops.head_linear(x, w, K, out)
    want = x.double() @ w[0].double().T
    assert bool(((out[:, 0].double() - want).abs() <= 2 ** -8 * want.abs() + 1e-5).all())


@pytest.mark.gpu
@pytest.mark.parametrize("kv_rank", [128, 100])
def test_weights_of_another_model(kv_rank):
    """A model that took another's weights by ``load_state_dict`` attends with them: the projections by head follow."""
    mx = mixer(16, 50, 10, 40, 32, kv_rank, 33)
    h = q16(rnd(torch.Generator().manual_seed(3), 40, 64))
    a, _ = one_layer("latent_attention", mx, 64, "cuda", torch.bfloat16, seed=5)
    b, _ = one_layer("latent_attention", mx, 64, "cuda", torch.bfloat16, seed=6)
    assert a.layers[0].mix.spec.absorbed
    b.load_state_dict(a.state_dict())
    assert torch.equal(run_mixer(a, h, [30], "cuda", torch.bfloat16), run_mixer(b, h, [30], "cuda", torch.bfloat16))
    assert (a.layers[0].mix.w_uv_h is None) == (kv_rank == 128)
