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
