"""Filing kernels of normed and of rotated keys (csrc/kv_rows.h) against float64: single rows and 16-row tiles with
remainders, blocks entered in the middle, rows that cache nothing, head sizes of 8 to 32 lanes with padding columns,
shared key parts and blended values; and a head size that only the general kernels take."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops

pytestmark = pytest.mark.gpu
DEV, BS = "cuda", 16
BF = torch.bfloat16


def _slots(T, start):
    s = (torch.arange(T, device=DEV) + start).int()
    if T > 5:
        s[3] = -1
    return s


def _filed(cache, rows, slots, keys_last):
    r, ok = cache.double(), slots >= 0
    s = slots[ok].long()
    if keys_last:
        r[s // BS, :, :, s % BS] = rows[ok]
    else:
        r[s // BS, :, s % BS] = rows[ok]
    return r


def _near(a, r):
    assert ((a.double() - r).abs() <= 2.0 ** -8 * r.abs() + 1e-5).all()   # one bf16 rounding of an f32 value


@pytest.mark.parametrize("T,start", [(1, 0), (37, 5), (511, 3), (512, 0), (1031, 9)])
@pytest.mark.parametrize("H,G,dim,vdim,bias", [(16, 4, 128, 128, True), (3, 1, 40, 24, False), (4, 2, 256, 64, True)])
def test_unitnorm(hip, T, start, H, G, dim, vdim, bias):
    torch.manual_seed(T + dim)
    W = (H + G) * dim + G * vdim
    u = torch.randn(T, W, device=DEV).to(BF)
    b = torch.randn(W, device=DEV).to(BF) if bias else None
    x = u.double() + (b.double() if bias else 0)
    nb, slots, tail = (T + start) // BS + 2, _slots(T, start), u[:, H * dim:].clone()
    kc, vc = torch.zeros(nb, G, BS, dim, device=DEV, dtype=BF), torch.zeros(nb, G, vdim, BS, device=DEV, dtype=BF)
    qk = x[:, :(H + G) * dim].view(T, H + G, dim)
    qk = qk / (qk.pow(2).mean(-1, keepdim=True) + 1e-5).sqrt()
    k_want, v_want = _filed(kc, qk[:, H:], slots, False), _filed(vc, x[:, (H + G) * dim:].view(T, G, vdim), slots, True)
    ops.unitnorm_kv_write(u, H, G, dim, vdim, 1e-5, kc, vc, slots, bias=b)
    _near(u[:, :H * dim].view(T, H, dim), qk[:, :H])
    _near(kc, k_want)
    _near(vc, v_want)
    assert torch.equal(u[:, H * dim:], tail)


@pytest.mark.parametrize("T,start", [(1, 0), (37, 5), (511, 3), (512, 0), (1031, 9)])
@pytest.mark.parametrize("H,G,qd,kd,sd,v,VD,KD,off,rot,blend", [(16, 4, 128, 128, 0, 128, 128, 128, 0, 128, False),
                                                                (4, 4, 192, 128, 64, 128, 128, 192, 128, 64, False),
                                                                (6, 3, 48, 24, 16, 40, 48, 48, 8, 32, True),
                                                                (2, 2, 20, 20, 0, 20, 24, 24, 0, 12, False)])
def test_rot(hip, T, start, H, G, qd, kd, sd, v, VD, KD, off, rot, blend):
    torch.manual_seed(T + qd)
    rn = lambda n: torch.randn(T, n + 8, device=DEV).to(BF)[:, :n]  # noqa: E731
    q, k, sh, vv, v2 = rn(H * qd), rn(G * kd), rn(sd) if sd else None, rn(G * v), rn(G * v) if blend else None
    pos = (torch.arange(T, device=DEV) + start).int()
    freq, mag = (0.5 ** torch.arange(rot // 2, device=DEV)).float(), 1.25
    ang = pos.double()[:, None] * freq.double()
    c, s = (ang.cos() * mag)[:, None], (ang.sin() * mag)[:, None]

    def turn(x):
        y, a, b = x.clone(), x[..., off:off + rot:2], x[..., off + 1:off + rot:2]
        y[..., off:off + rot:2], y[..., off + 1:off + rot:2] = a * c - b * s, b * c + a * s
        return y

    f = lambda t, n: t.double().view(T, -1, n)  # noqa: E731
    zeros = torch.zeros(T, G, max(KD, VD), device=DEV, dtype=torch.float64)
    kw = torch.cat([f(k, kd)] + ([sh.double()[:, None].expand(T, G, sd)] if sd else []) + [zeros[..., :KD - kd - sd]], -1)
    vw = 0.75 * f(vv, v) + 0.25 * f(v2, v) if blend else f(vv, v)
    nb, slots, q_want = (T + start) // BS + 2, _slots(T, start), turn(f(q.clone(), qd))
    kc, vc = torch.ones(nb, G, BS, KD, device=DEV, dtype=BF), torch.ones(nb, G, VD, BS, device=DEV, dtype=BF)
    k_want, v_want = _filed(kc, turn(kw), slots, False), _filed(vc, torch.cat([vw, zeros[..., :VD - v]], -1), slots, True)
    ops.rot_kv_write(q, H, qd, k, G, kd, sh, sd, vv, v, off, rot, freq, mag, pos, kc, vc, slots, v2, 0.25 if blend else 0.0)
    for a, r in ((q.reshape(T, H, qd), q_want), (kc, k_want), (vc, v_want)):
        # one bf16 rounding; a rotation of an angle up to 1,040 whose f32 rounding is 2^-24 of it (6e-5), times values up to ~6
        assert ((a.double() - r).abs() <= 2.0 ** -8 * r.abs() + 6e-4).all()
