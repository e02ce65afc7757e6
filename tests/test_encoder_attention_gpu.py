"""The encoder's attention in the order of large grids: every tile and head once, whatever their numbers."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# (tiles no multiple of the sixteen that a round of the order takes, one short of it and one more; heads from few to many, grouped ones)
@pytest.mark.parametrize("n,nh,hkv,D", [(175, 12, 12, 64), (176, 12, 12, 64), (177, 12, 12, 64), (1100, 2, 2, 32), (231, 16, 4, 128), (118, 32, 16, 64)])
@pytest.mark.parametrize("longest", [128, 256])
def test_large_grids(hip, n, nh, hkv, D, longest):
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    g = torch.Generator(device="cuda").manual_seed(n)
    lens = [1 + (i * 37) % longest for i in range(n)]
    lens[3], lens[-1] = 300, 129
    T = sum(lens)
    q = torch.randn(T, nh * D, device="cuda", generator=g).bfloat16()
    k, v = (torch.randn(T, hkv * D, device="cuda", generator=g).bfloat16() for _ in range(2))

    def run(seqs):
        r0, r1 = sum(lens[:seqs[0]]), sum(lens[:seqs[-1] + 1])
        part = [lens[i] for i in seqs]
        cu = torch.tensor([sum(part[:i]) for i in range(len(part) + 1)], dtype=torch.int32, device="cuda")
        return ops.flash_prefill(q[r0:r1], k[r0:r1], v[r0:r1], cu, nh, hkv, D, D ** -0.5, False, q_lens_cpu=part)

    tiles = len(ops.prefill_tiles(lens, lens, nh // hkv, False, D)[0])
    assert tiles * (nh // min(4, nh // hkv) if nh != hkv else nh) > 2048
    # (heads of their own: a tile is 128 rows, so that texts of up to 128 are one each and keep the plain order, but for heads of 32)
    assert hip.prefill_order(tiles, n, T, nh, D) == (longest > 128 or nh != hkv or D == 32)
    whole = run(range(n))
    step = 12   # (grids of at most 2,048 workgroups keep their order)
    parts = torch.cat([run(range(a, min(a + step, n))) for a in range(0, n, step)])
    assert torch.equal(whole, parts)
