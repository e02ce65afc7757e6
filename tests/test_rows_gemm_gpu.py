"""Few-row GEMM (csrc/rows_gemm.hip) against float64: row tiles and their edges, K ranges that the four waves share
evenly and not (fewer 64-steps than waves among them), every epilogue; and the routes that lead there."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _ref(x, w, b, epi):
    y = x.double() @ w.double().t()
    if epi == 1:
        g, u = (t.to(torch.bfloat16).double() for t in y.chunk(2, 1))
        return torch.nn.functional.silu(g).to(torch.bfloat16).double() * u
    if epi >= 2:
        y = y + b.double()
    return torch.nn.functional.gelu(y) if epi == 3 else torch.relu(y) if epi == 4 else y


@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 48, 49, 64, 65, 130, 257])
@pytest.mark.parametrize("N,K,epi", [(16, 64, 0), (48, 128, 2), (2048, 2048, 0), (160, 320, 1), (768, 768, 2), (3072, 768, 3),
                                     (96, 832, 4), (64, 14336, 0), (2048, 5632, 1)])
def test_rows_linear(hip, M, N, K, epi, wide):
    torch.manual_seed(M + N + K)
    x = torch.randn(M + 1, K + 8, device=DEV).to(torch.bfloat16)[1:, :K]   # rows of a wider tensor
    w = (torch.randn(N, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    b = torch.randn(N, device=DEV).to(torch.bfloat16) if epi >= 2 else None
    y, r = hip.rows_linear(x, w, b, epi, wide), _ref(x, w, b, epi)
    # one bf16 rounding (half a step: 2^-8 of the value) of an f32 sum of K products.  SwiGLU: the rounding of the
    # result and of silu(g), and a step (2^-7) of u and of g (silu's relative slope is below 1.3) where a sum
    # lies so near a rounding edge that f32 and f64 fall on different sides: below 7 half steps
    assert ((y.double() - r).abs() <= (7 if epi == 1 else 1) * 2.0 ** -8 * r.abs() + 2e-5 * K ** 0.5).all()


def test_rows_linear_refuses():
    lib = ops.lib()
    x, w = torch.zeros(4097, 128, device=DEV, dtype=torch.bfloat16), torch.zeros(32, 128, device=DEV, dtype=torch.bfloat16)
    for bad in ((x, w, None, 0), (x[:4], w[:24], None, 0), (x[:4], w, None, 2), (x[:4, :96], w[:, :96].contiguous(), None, 0)):
        with pytest.raises(RuntimeError):
            lib.rows_linear(*bad)


@pytest.mark.parametrize("M,N,K", [(19, 2304, 768), (64, 2048, 2048), (3, 10368, 2048), (64, 10368, 2048), (20, 4096, 14336), (40, 1152, 384),
                                   (200, 2048, 2048), (700, 2048, 2048), (1000, 768, 768), (1100, 768, 768), (333, 2304, 768)])
def test_routes_agree(M, N, K):
    """ops.linear / linear_swiglu give the same product whichever kernel the rule names."""
    torch.manual_seed(N)
    x = torch.randn(M, K, device=DEV).to(torch.bfloat16)
    w = (torch.randn(N, K, device=DEV) / K ** 0.5).to(torch.bfloat16)
    b = torch.randn(N, device=DEV).to(torch.bfloat16)
    for y, r in ((ops.linear(x, w), _ref(x, w, None, 0)), (ops.linear(x, w, b), _ref(x, w, b, 2)),
                 (ops.linear(x, w, b, act="gelu"), _ref(x, w, b, 3)), (ops.linear_swiglu(x, w), _ref(x, w, None, 1))):
        assert ((y.double() - r).norm() / r.norm()) < 4e-3


@pytest.fixture(autouse=True)
def tables():
    """The measured decode tables, put back behind a test that fills them."""
    saved = [(t, dict(t)) for t in (ops._DECODE_TABLE, ops._ROWS_TABLE, ops._WS_VARIANTS)]
    for t, _ in saved[:2]:
        t.clear()
    yield
    for t, v in saved:
        t.clear()
        t.update(v)
    ops.apply_ws_variants(saved[2][1])


class Spy:
    """The kernel library with the names of the products that ran."""

    def __init__(self, lib):
        self.lib, self.ran = lib, []

    def __getattr__(self, name):
        f = getattr(self.lib, name)
        if name in ("rows_linear", "ws_linear", "gemm", "skinny_linear", "gemv_decode"):
            return lambda *a, **k: (self.ran.append(name), f(*a, **k))[1]
        return f


@pytest.mark.parametrize("N,K,swiglu", [(2048, 2048, False), (1024, 1024, False), (4096, 1024, True), (10368, 2048, False)])
def test_measured_routes_win(monkeypatch, N, K, swiglu):
    """What start-up measured is what linear runs: each bucket's choice, also against the rule; shapes without an entry take the rule."""
    w = torch.randn(N, K, device="cuda").bfloat16() * K ** -0.5
    ms = (32, 64, 256)
    res = ops.tune_decode([(w, swiglu)], ms=ms)
    ms = [m for m in ms if (m, N, K, swiglu) in ops._ROWS_TABLE]
    assert ms
    spy = Spy(ops.lib())
    monkeypatch.setattr(ops, "lib", lambda: spy)
    run = ops.linear_swiglu if swiglu else ops.linear
    for m in ms:
        key = (m, N, K, swiglu)
        us = res[key + ("few", "rows")]
        assert {"ws", "gemm"} < set(us)
        route = ops.decode_route(m, N, K, swiglu)
        assert us[route] <= min(us.values()) / 0.94 + 0.1   # within the margin of a near tie (times rounded to 0.1 us)
        x = torch.randn(m - 3, K, device="cuda").bfloat16()
        for choice in (ops._ROWS_TABLE[key], None, False):      # the measured one, then both others forced
            ops._ROWS_TABLE[key] = choice
            spy.ran.clear()
            run(x, w)
            want = {None: "ws_linear" if ops._DECODE_TABLE[key] == "ws" else "gemm"}.get(choice, "rows_linear")
            assert spy.ran == [want]
        del ops._ROWS_TABLE[key]
        spy.ran.clear()
        run(x, w)
        assert (spy.ran == ["rows_linear"]) == (ops._rows_rule(m - 3, N, K, 1 if swiglu else 0) is not None)


@pytest.mark.parametrize("M,N,I,K,bn", [(1, 64, 32, 64, 64), (3, 192, 96, 128, 64), (64, 3072, 5632, 512, 64), (65, 128, 64, 320, 128), (128, 384, 192, 704, 128),
                                        (48, 10496, 5632, 256, 128), (128, 192, 32, 1088, 64)])
def test_two_products_beside(hip, M, N, I, K, bn):
    """A plain and a SwiGLU product of one x in one launch, both tile widths, fewer K stages than the rings have, rows apart: one bf16
    rounding of the plain result (2^-9 of it), SwiGLU also of g, u and silu(g), g's moving silu(g) by at most 1.1 times as much (twice that allowed)."""
    torch.manual_seed(M + N + K)
    rows = torch.randn(M, K + 64, device="cuda", dtype=torch.bfloat16)
    w, wgu = (torch.randn(n, K, device="cuda", dtype=torch.bfloat16) / K ** 0.5 for n in (N, 2 * I))
    for x in (rows[:, :K], rows[:, :K].contiguous()):
        got, f = hip.ws_beside(x, w, wgu, bn)
        y, gu = x.double() @ w.double().t(), x.double() @ wgu.double().t()
        g, u = gu[:, :I], gu[:, I:]
        assert ((got.double() - y).abs() <= 2.0 ** -8 * y.abs() + 1e-5).all()
        want = torch.nn.functional.silu(g) * u
        assert ((f.double() - want).abs() <= 2.0 ** -8 * (3 * want.abs() + 1.1 * (g * u).abs()) + 1e-5).all()


@pytest.mark.parametrize("M,N,I,bn", [(4, 128, 128, 0), (4, 128, 128, -64), (4, 128, 128, 1), (4, 128, 128, 32), (4, 128, 128, 256), (129, 128, 128, 64), (4, 96, 128, 64),
                                      (4, 128, 48, 64)])
def test_two_products_beside_refuses(hip, M, N, I, bn):
    """Tile widths that there are none of, none among them, and sizes that they do not divide: an error, not the end of the process."""
    x, w, wgu = (torch.zeros(n, 64, device="cuda", dtype=torch.bfloat16) for n in (M, N, 2 * I))
    with pytest.raises(RuntimeError, match="ws_beside"):
        hip.ws_beside(x, w, wgu, bn)


def test_two_products_beside_takes_what_apart_takes(hip):
    """ops.linear_beside returns what the two calls return, to the roundings of their sums' orders, or leaves the operands to them: rows and
    widths inside and outside the rule, an x of transposed memory, f32."""
    torch.manual_seed(0)
    big = torch.randn(300, 1024, device="cuda", dtype=torch.bfloat16)
    wn, wgu = (torch.randn(n, 256, device="cuda", dtype=torch.bfloat16) / 16 for n in (192, 256))
    cases = [(big[:m, :256], wn, wgu) for m in (1, 2, 17, 128, 129, 300)]
    cases += [(big[:256, :64].t(), wn, wgu), (big[:5, 8:264], wn, wgu), (big[:40, :256], wn[:40], wgu[:48]),
              (big[:40, :256].float(), wn.float(), wgu.float())]
    for x, w, gu in cases:
        if x.dtype == torch.bfloat16:
            a, b = ops.linear(x, w), ops.linear_swiglu_any(x, gu)
        else:
            a, b = torch.nn.functional.linear(x, w), ops.linear_swiglu_any(x, gu)
        both = ops.linear_beside(x, w, gu)
        assert (both is not None) == (x.dtype == torch.bfloat16 and x.stride(1) == 1 and x.shape[0] <= 128 and w.shape[0] == 192)
        if both is None:
            continue
        y, f = both
        assert y.shape == a.shape and f.shape == b.shape and y.dtype == a.dtype
        for p, q in ((y, a), (f, b)):
            assert (p.float() - q.float()).abs().max() <= 2.0 ** -6 * q.float().abs().max()
