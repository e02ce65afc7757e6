"""GELU in the one-wave product's epilogue (csrc/gemm1w.hip): every bf16 argument, as a table (256 and 192-row tiles, the persistent walk)
and computed (128-row tiles), and arguments inside and outside the table in one row."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _all_bf16(g):
    """All 65,536 bf16 values in a random order: a wave meets some that the table holds and some that it does not."""
    return torch.randperm(65536, generator=g, device="cuda").to(torch.int32).to(torch.int16).view(torch.bfloat16)


@pytest.mark.parametrize("M,K", [(257, 192), (1200, 128 * 3)])
@pytest.mark.parametrize("inside", [False, True])
def test_every_argument(hip, M, K, inside):
    g = torch.Generator("cuda").manual_seed(M)
    b = _all_bf16(g)
    if inside:   # (and all of them where whole waves stay inside)
        b = b[(b.abs() >= 2.0 ** -16) & (b.abs() < 16)]
        b = b[:b.numel() // 256 * 256].contiguous()
    N = b.numel()
    x, w = torch.zeros(M, K, device="cuda", dtype=torch.bfloat16), torch.zeros(N, K, device="cuda", dtype=torch.bfloat16)
    y3, y4, y5 = (hip.gemm(x, w, b, 3, 256, None, v, 1) for v in (3, 4, 5))
    for y in (y3, y4):
        assert torch.equal(y.view(torch.int16), y5.view(torch.int16))
    want = torch.nn.functional.gelu(b.double())
    ok = b.isfinite()
    # the polynomial's 2e-4 of the value in the negative tail (3.9e-7 elsewhere), half a bf16 step
    err = (y3.double() - want[None]).abs()[:, ok]
    assert bool((err <= (2.0 ** -8 + 1e-3) * want[ok].abs() + 1e-6).all()), float(err.max())


def test_persistent_walk(hip):
    """More tiles than two per CU: the table outlives the first one."""
    g = torch.Generator("cuda").manual_seed(3)
    M, N, K = 23 * 256 + 17, 24 * 256, 256
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w, b = (torch.randn(N, K, generator=g, device="cuda") / 8).bfloat16(), torch.randn(N, generator=g, device="cuda").bfloat16()
    x[::7] = 0   # rows of the bias alone
    assert torch.equal(hip.gemm(x, w, b, 3, 256, None, 3, 1), hip.gemm(x, w, b, 3, 256, None, 5, 1))
