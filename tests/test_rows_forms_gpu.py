"""The few-row product's residual epilogue and its widest form."""
import functools

import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops

pytestmark = pytest.mark.gpu


def _r(g, *shape, scale=1.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale).to(torch.bfloat16)


@pytest.mark.parametrize("M,N,K,wide", [(19, 768, 3072, False), (65, 32, 128, True), (1, 16, 64, False), (64, 96, 320, False)])
def test_product_plus_residual(hip, M, N, K, wide):
    """Rounded as the product and the sum apart."""
    g = torch.Generator("cuda").manual_seed(M)
    x, w, b, res = _r(g, M, K), _r(g, N, K, scale=K ** -0.5), _r(g, N), _r(g, M, N + 8)[:, :N]
    assert torch.equal(hip.rows_linear(x, w, b, 5, wide, res), hip.rows_linear(x, w, b, 2, wide) + res)


@pytest.mark.parametrize("M,N,K,epi", [(1, 64, 64, 0), (17, 192, 320, 2), (64, 10496, 2048, 0), (65, 128, 832, 1), (120, 11264, 2048, 1), (33, 320, 64, 3)])
def test_64_columns_per_workgroup(hip, M, N, K, epi):
    """The product's widest form sums K in the same order as the narrow one."""
    g = torch.Generator("cuda").manual_seed(M + N)
    x, w = _r(g, M, K), _r(g, N, K, scale=K ** -0.5)
    b = _r(g, N) if epi >= 2 else None
    assert torch.equal(hip.rows_linear(x, w, b, epi, 2), hip.rows_linear(x, w, b, epi, 0))


@pytest.mark.parametrize("wide", [0, 1, 2])
@pytest.mark.parametrize("M,N,K", [(1, 16, 64), (17, 128, 128), (64, 2048, 2048), (65, 192, 832)])
def test_two_products_in_one_launch(hip, M, N, K, wide):
    g = torch.Generator("cuda").manual_seed(M)
    x1, x2 = _r(g, M, K), _r(g, M, K + 8)[:, :K]
    w1, w2 = _r(g, N, K, scale=K ** -0.5), _r(g, N, K, scale=K ** -0.5)
    y1, y2 = hip.rows_pair(x1, w1, x2, w2, wide)
    assert torch.equal(y1, hip.rows_linear(x1, w1, None, 0, wide)) and torch.equal(y2, hip.rows_linear(x2, w2, None, 0, wide))


@pytest.mark.parametrize("M", [1, 2, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("N,K1,K2", [(2048, 4096, 5632), (2048, 2048, 5632), (1024, 4096, 4160), (4096, 1024, 1088), (8192, 512, 960)])
@pytest.mark.parametrize("picked", [False, True])
def test_sums_of_two_products(hip, M, N, K1, K2, picked):
    """Two products as f32 parts and the norm that adds them up, against the same in float64 with each product rounded to bf16 once."""
    g = torch.Generator(device="cuda").manual_seed(M + N + K2)
    rn = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    x1, x2 = rn(M, K1 + 8).bfloat16()[:, :K1], rn(M, K2).bfloat16()
    w1, w2 = (rn(N, K1) / K1 ** 0.5).bfloat16(), (rn(N, K2) / K2 ** 0.5).bfloat16()
    sums = ops.linear_sums(x1, w1, x2, w2)
    assert sums is not None and sums[0].shape[1:] == (M, N) and 1 <= sums[1] < sums[0].shape[0]
    a, b = x1.double() @ w1.double().T, x2.double() @ w2.double().T
    got1, got2 = (functools.reduce(torch.add, s.unbind(0)) for s in (sums[0][:sums[1]], sums[0][sums[1]:]))   # in the norm's order: the same bits
    for got, want in ((got1, a), (got2, b)):
        assert (got.double() - want).norm() <= 2 ** -21 * want.norm()   # f32 sums of exact products: some 2^-24 each
    x, e, bias, w = rn(M, N), rn(M, N), rn(N), rn(N + 1)[1:]   # (weights that are not aligned to four)
    idx = torch.arange(M - 1, -1, -3, device="cuda") if picked else None
    want = x.double() + 0.5 * (got1.bfloat16().double() + bias.double() + got2.bfloat16().double()) + e.double()
    out = want if idx is None else want[idx]
    out = out / (out.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt() * (1.0 + w.double())
    x0 = x.clone()
    y = ops.stream_rmsnorm(x, None, None, e, 0.5, w, 1.0, 1e-5, idx=idx, a_bias=bias, sums=sums)
    # one bf16 rounding of the result; the stream itself a few f32 roundings of terms of its own size
    assert (y.double() - out).norm() <= 2 ** -8 * out.norm()
    assert torch.equal(x, x0) if picked else (x.double() - want).norm() <= 2 ** -18 * want.norm()


@pytest.mark.parametrize("M,N,K1,K2", [(0, 2048, 2048, 5632), (65, 2048, 2048, 5632), (64, 2080, 2048, 2048), (64, 2048, 256, 256), (64, 64, 4096, 4096)])
def test_sums_not_taken(hip, M, N, K1, K2):
    z = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    assert ops.linear_sums(z(M, K1), z(N, K1), z(M, K2), z(N, K2)) is None


@pytest.mark.parametrize("M,N,K,epi,wide", [(400, 576, 1152, 3, 1), (400, 1152, 384, 0, 1), (320, 3136, 128, 1, 2), (257, 400, 64, 2, 0), (1000, 2112, 64, 0, 2),
                                            (16, 16, 64, 0, 0), (4096, 48, 64, 0, 0)])
def test_last_columns_over_all_xcds(hip, M, N, K, epi, wide):
    """Column tiles that are no multiple of 8, of several row tiles: every row tile of the last columns is computed once."""
    g = torch.Generator("cuda").manual_seed(M + N)
    x, w = _r(g, M, K), _r(g, N, K, scale=K ** -0.5)
    b = _r(g, N) if epi >= 2 else None
    y = hip.rows_linear(x, w, b, epi, wide)
    p = x.double() @ w.double().T
    if epi == 1:
        u, v = (t.to(torch.bfloat16).double() for t in p.chunk(2, 1))
        p = torch.nn.functional.silu(u).to(torch.bfloat16).double() * v
    elif epi >= 2:
        p = p + b.double()
        p = torch.nn.functional.gelu(p) if epi == 3 else p
    # as tests/test_rows_gemm_gpu.py: one bf16 rounding of an f32 sum, SwiGLU below 7 half steps
    assert ((y.double() - p).abs() <= (7 if epi == 1 else 1) * 2.0 ** -8 * p.abs() + 2e-5 * K ** 0.5).all()
    if epi == 0:
        x2, w2 = _r(g, M, K), _r(g, N, K, scale=K ** -0.5)
        y1, y2 = hip.rows_pair(x, w, x2, w2, wide)
        assert torch.equal(y1, y) and torch.equal(y2, hip.rows_linear(x2, w2, None, 0, wide))


@pytest.mark.parametrize("M", [1, 64])
def test_sums_of_odd_column_tiles(hip, M):
    """33 column tiles of 7 parts: 35 of them on one XCD, unless the last column's parts go around."""
    g = torch.Generator("cuda").manual_seed(M)
    x1, x2, w1, w2 = _r(g, M, 2112), _r(g, M, 2816), _r(g, 2112, 2112, scale=2112 ** -0.5), _r(g, 2112, 2816, scale=2816 ** -0.5)
    parts, s1 = hip.rows_sums(x1, w1, x2, w2)
    assert parts.shape == (7, M, 2112)
    for got, want in ((parts[:s1], x1.double() @ w1.double().T), (parts[s1:], x2.double() @ w2.double().T)):
        assert (got.double().sum(0) - want).norm() <= 2 ** -21 * want.norm()
