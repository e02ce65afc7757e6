"""Expert products of decode-sized steps (csrc/moe.hip: weight rows through private LDS rings) against float64: one to four row tiles per
walk, experts with more pairs than a walk takes (the rings are filled again behind the sums) beside experts without any, and fewer
64-column stages than waves; and the sizes from which the grouped dense product takes over."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops

pytestmark = pytest.mark.gpu


def choices(T, E, top, skew, g):
    t = torch.stack([torch.randperm(E, generator=g)[:top] for _ in range(T)])
    if skew:   # nearly all tokens choose expert 1, experts from E - 2 on nobody
        t = t % (E - 2)
        t[: T - T // 8, 0] = 1
    return t.int()


def check(T, E, top, W, ff, skew):
    g = torch.Generator().manual_seed(T * 7 + W + ff + skew)
    table = choices(T, E, top, skew, g)
    b16 = lambda t: t.to(torch.bfloat16)
    h = b16(torch.randn(T, W, generator=g))
    gu, dn = b16(torch.randn(E, 2 * ff, W, generator=g) * W ** -0.5), b16(torch.randn(E, W, ff, generator=g) * ff ** -0.5)
    seg, order = ops.moe_route(None, table.cuda(), E)
    pairs = table.reshape(-1).long()[order.cpu().long()]
    assert torch.equal(pairs, pairs.sort().values)
    mid = ops.lib().moe_gemm(h.cuda(), order, seg, gu.cuda(), top, True).cpu()
    y = torch.stack([gu[e].double() @ h[p // top].double() for p, e in zip(order.cpu().tolist(), pairs.tolist())])
    gate, up = y[:, :ff], y[:, ff:]
    want = gate * torch.sigmoid(gate) * up
    # one rounding (2^-8 covers half a step); f32 sums of K products of standard deviation 1, the fast exponential and reciprocal
    tol = 2 ** -8 * want.abs() + 1e-4
    assert bool(((mid.double() - want).abs() <= tol).all()), float(((mid.double() - want).abs() - tol).max())
    out = ops.lib().moe_gemm(mid.cuda(), order, seg, dn.cuda(), top, False).cpu().double()
    want = torch.empty(T * top, W, dtype=torch.float64)
    for i, (p, e) in enumerate(zip(order.cpu().tolist(), pairs.tolist())):
        want[p] = dn[e].double() @ mid[i].double()
    tol = 2 ** -8 * want.abs() + 1e-4
    assert bool(((out - want).abs() <= tol).all()), float(((out - want).abs() - tol).max())
    return h, table, gu, dn


@pytest.mark.parametrize("skew", [False, True])
@pytest.mark.parametrize("T,E,top", [(1, 8, 1), (4, 8, 2), (32, 8, 2), (43, 8, 2), (64, 8, 2), (92, 8, 2), (160, 8, 2), (220, 8, 2)])
def test_row_tiles_and_walks(T, E, top, skew):
    check(T, E, top, 256, 128, skew)   # 0 .. 55 pairs per expert on average, up to 200 in one


@pytest.mark.parametrize("W,ff", [(64, 192), (192, 64), (64, 64), (320, 128)])
def test_waves_without_a_stage(W, ff):
    check(40, 6, 2, W, ff, True)


@pytest.mark.parametrize("T,dense", [(255, False), (256, True), (400, True), (511, True), (512, True)])
def test_route_to_the_grouped_product(monkeypatch, T, dense):
    """64 to 127 pairs per expert: one dense product per expert on small row tiles; below, the rings."""
    E, top, W, ff = 8, 2, 256, 256
    h, table, gu, dn = check(T, E, top, W, ff, False)
    lib, ran = ops.lib(), []

    class Spy:
        def __getattr__(self, name):
            if name in ("gemm_grouped", "moe_gemm"):
                ran.append(name)
            return getattr(lib, name)

    monkeypatch.setattr(ops.window, "lib", lambda: Spy())
    got = ops.window.run_experts(h.cuda(), None, table.cuda(), gu.cuda(), dn.cuda(), top).cpu().double()
    assert ran == ["gemm_grouped" if dense else "moe_gemm"] * 2
    want = torch.empty(T * top, W, dtype=torch.float64)
    for p, e in enumerate(table.reshape(-1).tolist()):
        y = gu[e].double() @ h[p // top].double()
        mid = (y[:ff] * torch.sigmoid(y[:ff]) * y[ff:]).bfloat16().double()
        want[p] = dn[e].double() @ mid
    # the result's rounding, and the middle's where its f32 value fell on the other side of a rounding boundary (2^-8 of single terms)
    assert float((got - want).norm() / want.norm()) < 2 ** -8


@pytest.mark.parametrize("T,top,E,n", [(1, 1, 1, 1), (64, 2, 16, 8), (513, 2, 16, 3), (700, 3, 40, 65)])
def test_routes_of_several_layers(hip, T, top, E, n):
    """One launch for all tables sorts each as a launch for it alone (the order inside an expert's segment is free)."""
    g = torch.Generator().manual_seed(T)
    tables = [torch.randint(0, E, (50, top), generator=g, dtype=torch.int32).cuda() for _ in range(n)]
    ids = torch.randint(0, 50, (T,), generator=g, dtype=torch.int32).cuda()
    got = ops.moe_routes(ids, tables, E)
    assert len(got) == n
    for t, (seg, order) in zip(tables, got):
        want, worder = ops.moe_route(ids, t, E)
        assert torch.equal(seg, want)
        for e in range(E):
            a, b = int(seg[e]), int(seg[e + 1])
            assert torch.equal(order[a:b].sort().values, worder[a:b].sort().values)


@pytest.mark.parametrize("dim,vdim,P,BS", [(128, 128, 64, 16), (72, 40, 8, 16), (64, 96, 24, 48), (256, 8, 32, 32), (16, 200, 64, 128)])
def test_pooled_means(hip, dim, vdim, P, BS):
    """Blocks that end in the step, of sequences with and without a past, against the f32 means."""
    G, lens = 2, [(5 * P, 5 * P), (3, 2 * P), (1, P - 1), (P + 1, 3 * P + 1), (1, 4 * P)]
    g = torch.Generator().manual_seed(dim)
    nb = [-(-c // BS) for _, c in lens]
    bt = torch.zeros(len(lens), max(nb), dtype=torch.int32)
    perm, at = torch.randperm(sum(nb), generator=g).to(torch.int32), 0
    for s, n in enumerate(nb):
        bt[s, :n] = perm[at:at + n]
        at += n
    kc, vc = torch.randn(sum(nb), G, BS, dim, generator=g).bfloat16(), torch.randn(sum(nb), G, vdim, BS, generator=g).bfloat16()
    cu = torch.tensor([0] + [n for n, _ in lens]).cumsum(0).to(torch.int32)
    ctx = torch.tensor([c for _, c in lens], dtype=torch.int32)
    slots = torch.zeros(int(cu[-1]), dtype=torch.int32)
    out = []
    for dev in ("cpu", "cuda"):
        pk, pv = torch.zeros_like(kc).to(dev), torch.zeros_like(vc).to(dev)
        ops.pool_kv_write(kc.to(dev), vc.to(dev), pk, pv, P, bt.to(dev), ctx.to(dev), cu.to(dev), slots.to(dev), 0, max(n for n, _ in lens))
        out.append((pk.cpu().float(), pv.cpu().float()))
    for a, b in zip(*out):   # f32 means in another order may round to the other neighbour: one bf16 step
        assert ((a - b).abs() <= 2.0 ** -7 * a.abs() + 1e-6).all() and ((a != 0) == (b != 0)).all()


@pytest.mark.parametrize("T,top,E,dead", [(1, 2, 4, 1), (48, 2, 16, 15), (48, 2, 16, 0), (64, 2, 16, 64), (17, 3, 8, 9), (600, 2, 128, 31)])
def test_rows_that_are_not_live_run_through_no_expert(T, top, E, dead):
    """The pairs of rows without a live word are no expert's and stand behind the others; their results are zeros, the others' the same bits."""
    W, ff, V = 128, 64, 40
    g = torch.Generator().manual_seed(T + dead)
    bf = lambda *s: (torch.randn(*s, generator=g) * 0.1).to(torch.bfloat16).cuda()
    h, gu, dn = bf(T, W), bf(E, 2 * ff, W), bf(E, W, ff)
    table = torch.rand(V, E, generator=g).argsort(1)[:, :top].to(torch.int32).contiguous().cuda()
    ids = torch.randint(0, V, (T,), generator=g, dtype=torch.int32).cuda()
    live = torch.arange(T, dtype=torch.int32)
    live[torch.randperm(T, generator=g)[:dead]] = -1
    live = live.cuda()
    assert ops.moe_skips_rows(T, top, E, W, ff)
    (seg, order), = ops.moe_routes(ids, [table], E, live)
    seg, order_h = seg.tolist(), order.tolist()
    assert seg[-1] == (T - dead) * top and sorted(order_h) == list(range(T * top))
    assert all(live[p // top] >= 0 for p in order_h[:seg[-1]]) and all(live[p // top] < 0 for p in order_h[seg[-1]:])
    route = ops.moe_routes(ids, [table], E, live)[0]
    got = ops.table_experts(h, ids, table, gu, dn, top, route).view(T, top, W)
    want = ops.table_experts(h, ids, table, gu, dn, top).view(T, top, W).clone()
    want[(live < 0)] = 0
    assert torch.equal(got, want)
    y, got = ops.linear_table_experts(h, gu[0].contiguous(), ids, table, gu, dn, top, route)
    assert torch.equal(got.view(T, top, W), want)
    exact = h.double() @ gu[0].double().t()
    assert ((y.double() - exact).norm() / exact.norm()).item() < 4e-3   # (one rounding to bf16: 2^-9)
