"""The few-row product's residual epilogue and its widest form."""
import pytest
import torch

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
