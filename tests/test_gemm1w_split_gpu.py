"""Ranges of K on the one-wave-per-SIMD tiles: their sum and its epilogues, against the product in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    return ops.lib()


# (ranges of 3 K-tiles and uneven ones; rows at and past the tiles' edges and no multiple of the four that a workgroup of the sum takes)
@pytest.mark.parametrize("variant", [3, 4, 5])
@pytest.mark.parametrize("M,N,K,splits", [(257, 256, 384, 2), (259, 768, 640, 3), (384, 256, 1024, 4), (511, 512, 1088, 5), (130, 256, 1216, 6),
                                          (258, 256, 1344, 7), (641, 1024, 1600, 8), (1, 256, 1536, 8)])
def test_split_epilogues(hip, M, N, K, splits, variant):
    torch.manual_seed(M + N + splits)
    x = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    b = torch.randn(N, device="cuda").bfloat16()
    y = x.double() @ w.double().t()
    # a product's error: its f32 sums (each of K additions rounds to 2^-24 of the sum of magnitudes at most), then bf16 (half of its 2^-7 steps: 2^-8 of the value)
    acc = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs().t())
    rnd = 2.0 ** -8
    for epi in (0, 2, 3, 4):
        assert hip.gemm_supported(M, N, K, epi, 256, splits, variant)
        out = hip.gemm(x, w, None if epi == 0 else b, epi, 256, None, variant, splits).double()
        e = y if epi == 0 else y + b.double()
        want = torch.nn.functional.gelu(e) if epi == 3 else e.clamp_min(0) if epi == 4 else e
        # (before an activation the sum is rounded too; GELU's slope is below 1.13, its own f32 error below 2^-20 of its argument)
        before = 0 if epi == 0 else 1.13 * (rnd * (1 + rnd) * (e.abs() + acc)) + 2.0 ** -20 * e.abs()
        bound = (1.13 * acc + before) * (1 + rnd) + rnd * want.abs()
        assert bool(((out - want).abs() <= bound).all()), (epi, float(((out - want).abs() - bound).max()))
    r0 = torch.randn(M, N, device="cuda").bfloat16()
    r, ss = r0.clone(), torch.full((N // 256, M), -1.0, device="cuda")
    hip.gemm_fused(x, w, 6, 256, None, variant, splits, resid=r, ss_out=ss)
    want = r0.double() + y
    bound = (acc + rnd * (y.abs() + acc)) * (1 + rnd) + rnd * want.abs()
    assert bool(((r.double() - want).abs() <= bound).all())
    sq = r.double().square().view(M, N // 256, 256).sum(-1).t()
    assert bool(((ss.double() - sq).abs() <= 256 * 2.0 ** -24 * sq).all())


def test_far_rows_keep_an_unsplit_kernel(hip):
    """A residual product takes its split by the operands' row strides as well: the same values either way."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    M, N, K = 300, 256, 2048
    torch.manual_seed(5)
    big = torch.empty(M, 122880, device="cuda", dtype=torch.bfloat16)
    big[:, :K] = torch.randn(M, K, device="cuda").bfloat16()
    w = (torch.randn(N, K, device="cuda") * K ** -0.5).bfloat16()
    far, near = big[:, :K], big[:, :K].contiguous()
    assert ops._resid_cfg(M, N, K, near.stride(0))[2] > 1 and ops._resid_cfg(M, N, K, far.stride(0)) != ops._resid_cfg(M, N, K, near.stride(0))
    outs = [ops.linear(v, w).double() for v in (far, near)]
    want = near.double() @ w.double().t()
    bound = K * 2.0 ** -24 * (near.double().abs() @ w.double().abs().t()) + 2.0 ** -8 * want.abs()
    assert all(bool(((o - want).abs() <= bound).all()) for o in outs)
