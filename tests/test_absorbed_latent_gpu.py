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
