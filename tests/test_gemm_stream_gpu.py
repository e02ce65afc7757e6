"""K loop of the one-wave GEMM (csrc/gemm1w.hip): numbers of K-tiles around its prologue and tail, odd and even, on every row tile, with
row counts at a tile's edge, against float64; the persistent walk takes an even number of K-tiles and leaves the odd ones to the plain form."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops


def check(M, N, K, variant, swiglu):
    g = torch.Generator(device="cuda").manual_seed(M * 31 + K + variant)
    x = torch.randn(M, K, generator=g, device="cuda").bfloat16()
    w = (torch.randn(N, K, generator=g, device="cuda") * K ** -0.5).bfloat16()
    got = ops.lib().gemm(x, w, None, 1 if swiglu else 0, 256, None, variant, 1).double()
    y = x.double() @ w.double().T
    # half a bf16 step (2^-8 of the value) per rounding: the product; SwiGLU: gate (its slope in silu is at most 1.1), up, silu, result
    if swiglu:
        gate, up = y[:, :N // 2], y[:, N // 2:]
        want = gate * torch.sigmoid(gate) * up
        tol = 2 ** -8 * (3 * want.abs() + 1.1 * (gate * up).abs())
    else:
        want, tol = y, 2 ** -8 * y.abs()
    tol = 1.05 * tol + 1e-4      # second order terms, f32 sums of K products of standard deviation 1
    assert got.shape == want.shape and bool(((got - want).abs() <= tol).all()), float(((got - want).abs() - tol).max())


@pytest.mark.gpu
@pytest.mark.parametrize("variant,bm", [(3, 256), (4, 192), (5, 128)])
@pytest.mark.parametrize("tiles", [3, 4, 5, 6, 9])
def test_k_tiles(variant, bm, tiles):
    for M in (1, bm - 1, bm + 1):
        check(M, 512, 64 * tiles, variant, False)
        check(M, 512, 64 * tiles, variant, True)


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [3, 4, 11, 12, 16])
def test_many_tiles_of_short_k(tiles):
    check(256 * 180 + 17, 768, 64 * tiles, 3, False)   # 543 tiles: three per CU, the last ones partly filled
