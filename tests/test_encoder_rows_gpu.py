"""The encoder layer's fused launches for few rows (csrc/encoder_rows.hip) against float64, at the edges of their row tiles."""
import pytest
import torch

pytestmark = pytest.mark.gpu
EPS = 2.0 ** -8   # twice bf16's unit roundoff: one rounding, and the f32 sums' share


def _r(g, *shape, scale=1.0, shift=0.0):
    return (torch.randn(*shape, generator=g, device="cuda") * scale + shift).to(torch.bfloat16)


@pytest.mark.parametrize("M", [1, 15, 16, 17, 33, 48, 49, 64, 65, 100])
@pytest.mark.parametrize("K,N,gelu", [(768, 2304, False), (768, 3072, True), (384, 1152, False), (64, 48, True), (320, 16, False)])
def test_ln_linear(hip, M, K, N, gelu):
    g = torch.Generator("cuda").manual_seed(M * 7 + K + N)
    wide = _r(g, M, K + 8)
    x = wide[:, :K]
    lw, lb, w, b = _r(g, K, scale=0.1, shift=1), _r(g, K, scale=0.1), _r(g, N, K, scale=K ** -0.5), _r(g, N, scale=0.1)
    y, h = hip.ln_linear(x, lw, lb, 1e-12, w, b, gelu)
    s = x.double()
    d = s - s.mean(1, keepdim=True)
    want = d / torch.sqrt((d * d).mean(1, keepdim=True) + 1e-12) * lw.double() + lb.double()
    assert ((h.double() - want).abs() <= EPS * want.abs() + 1e-5).all()
    p = h.double() @ w.double().T + b.double()
    q = torch.nn.functional.gelu(p) if gelu else p
    # the product's f32 sum: K roundings of terms up to sum |h w|; GELU's slope is at most 1.13
    bound = EPS * q.abs() + 1.13 * K * 2.0 ** -24 * (h.double().abs() @ w.double().abs().T + b.double().abs()) + 1e-6
    assert ((y.double() - q).abs() <= bound).all()


@pytest.mark.parametrize("M", [1, 2, 15, 16, 17, 31, 32])
@pytest.mark.parametrize("nh,N", [(12, 768), (2, 128), (1, 16), (7, 448)])
def test_attn_linear(hip, M, nh, N):
    g = torch.Generator("cuda").manual_seed(M * 3 + nh)
    K = nh * 64
    qkv, w, b = _r(g, M, 3 * K, scale=1.5), _r(g, N, K, scale=K ** -0.5), _r(g, N, scale=0.1)
    res = _r(g, M, N + 8)[:, :N]
    y = hip.attn_linear(qkv, nh, 0.125, w, b, res)
    q, k, v = (t.view(M, nh, 64).transpose(0, 1) for t in qkv.double().view(M, 3, K).unbind(1))
    p = torch.softmax(q @ k.transpose(1, 2).contiguous() * 0.125, -1)
    a, av = (p @ v).transpose(0, 1).reshape(M, K), (p @ v.abs()).transpose(0, 1).reshape(M, K)
    want = a @ w.double().T + b.double()
    # P and A rounded to bf16 once each, the result once; f32 scores of size up to s move P by 64 * 2^-24 * s, below that
    bound = (2 * EPS * av) @ w.double().abs().T + EPS * want.abs() + EPS * (want + res.double()).abs() + 1e-5
    assert ((y.double() - want - res.double()).abs() <= bound).all()


def test_short_texts_take_the_fused_layers(hip):
    """One text and several packed ones give the rows that the layers apart give, up to the order of the attention's sums."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    from llm_kubernetes_minikube_sharp4dev_amd.models import build_encoder

    m = build_encoder("bge-base", device="cuda").random_init(3)
    for lens in ([19], [33], [64], [5, 9, 33]):
        ids = torch.randint(1000, 30000, (sum(lens),), dtype=torch.int32, device="cuda")
        pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).cuda()
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
        got, keep = m(ids, cu, pos, lens), ops.ENCODER_ROWS
        try:
            ops.ENCODER_ROWS = 0
            apart = m(ids, cu, pos, lens)
        finally:
            ops.ENCODER_ROWS = keep
        assert torch.nn.functional.cosine_similarity(got, apart).min() > 0.9999


@pytest.mark.parametrize("lens", [[9], [3, 9]])
def test_parameters_anywhere(hip, lens):
    """Biases that begin between two 16-byte lines (views of a larger tensor) are taken, as by the launches apart; the rows are the same."""
    from llm_kubernetes_minikube_sharp4dev_amd.models import build_encoder

    m = build_encoder("bert-tiny", device="cuda").random_init(3)
    g = torch.Generator("cuda").manual_seed(1)
    for L in m.layers:
        for name in ("qkv_b", "o_b", "fc1_b", "fc2_b"):
            getattr(L, name).copy_(_r(g, getattr(L, name).numel(), scale=0.1))
    ids = torch.randint(1000, 30000, (sum(lens),), dtype=torch.int32, device="cuda")
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).cuda()
    cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
    want = m(ids, cu, pos, lens)
    for L in m.layers:
        for name in ("qkv_b", "o_b", "fc1_b", "fc2_b"):
            v = getattr(L, name)
            wide = torch.empty(v.numel() + 1, dtype=v.dtype, device="cuda")
            wide[1:] = v
            setattr(L, name, torch.nn.Parameter(wide[1:], requires_grad=False))
            assert getattr(L, name).data_ptr() % 16
    assert torch.equal(m(ids, cu, pos, lens), want)
