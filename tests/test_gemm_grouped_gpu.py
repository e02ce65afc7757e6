"""One product per expert over rows sorted by expert (the prompt form of the routed feed-forward): row counts on both sides of the row
tiles (128, 192 and 256 rows, chosen by the mean), against float64; gathered sources, scattered results, SwiGLU."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops


# whole rounds of tiles on 256 CUs: 192 rows (one tile per expert instead of two of 128), 256 rows
FULL192, FULL256 = [150, 192, 191, 1, 129, 193, 185, 160, 190, 170, 175, 0, 180, 188, 65, 192], [256, 250, 193, 240, 255, 257, 230, 245] * 2


# 224 and 288 rows (and 256 at a width of 3072)
FULL224 = [448, 449, 447, 224, 225, 223, 400, 385, 390, 672, 673, 0, 380, 370, 1, 395]
FULL288 = [576, 575, 512, 513, 288, 289, 577, 545, 560, 0, 864, 500, 561, 1, 529, 512]


@pytest.mark.gpu
@pytest.mark.parametrize("counts,swiglu,N,K", [(FULL224, True, 4096, 192), (FULL224, False, 2048, 256), (FULL288, True, 4096, 192),
                                               (FULL288, False, 2048, 256), (FULL288, False, 2048, 320), (FULL256, True, 3072, 192),
                                               (FULL256, False, 3072, 256)])
def test_rounds_of_taller_tiles(counts, swiglu, N, K):
    test_rows_per_expert(counts, swiglu, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("counts,swiglu,N,K", [(FULL192, True, 8192, 192), (FULL192, False, 4096, 192), (FULL256, True, 4096, 192),
                                               (FULL256, False, 4096, 256)])
def test_full_rounds(counts, swiglu, N, K):
    test_rows_per_expert(counts, swiglu, N, K)


@pytest.mark.gpu
@pytest.mark.parametrize("counts", [[1, 64, 65], [128, 0, 129, 192, 17], [193, 256, 257, 17], [130, 191, 192, 193, 0, 385], [319, 320, 321, 384, 385, 512, 513]])
@pytest.mark.parametrize("swiglu,N,K", [(True, 512, 192), (True, 768, 256), (False, 256, 128), (False, 512, 320), (False, 192, 320)])
def test_rows_per_expert(counts, swiglu, N, K):
    g = torch.Generator().manual_seed(sum(counts))
    E, R = len(counts), sum(counts)
    x = torch.randn(R, K, generator=g).bfloat16()
    w = (torch.randn(E, N, K, generator=g) * K ** -0.5).bfloat16()
    seg = torch.tensor([0] + counts).cumsum(0).int()
    perm = torch.randperm(R, generator=g).int()
    cols = N // 2 if swiglu else N
    want, tol = torch.zeros(R, cols, dtype=torch.float64), torch.zeros(R, cols, dtype=torch.float64)
    for e in range(E):
        a, b = int(seg[e]), int(seg[e + 1])
        y = x[perm[a:b].long()].double() @ w[e].double().T
        # half a bf16 step (2^-8 of the value) per rounding: the product; SwiGLU: gate (its slope in silu is at most 1.1), up, silu, result
        if swiglu:
            gate, up = y[:, :cols], y[:, cols:]
            want[a:b] = gate * torch.sigmoid(gate) * up
            tol[a:b] = 2 ** -8 * (3 * want[a:b].abs() + 1.1 * (gate * up).abs())
        else:
            want[a:b], tol[a:b] = y, 2 ** -8 * y.abs()
    got = ops.lib().gemm_grouped(x.cuda(), seg.cuda(), w.cuda(), swiglu, perm.cuda(), None).double().cpu()
    tol = 1.05 * tol + 1e-4      # second order terms, f32 sums of K products of standard deviation 1
    assert bool(((got - want).abs() <= tol).all()), float(((got - want).abs() - tol).max())
    pairs = ops.lib().gemm_grouped(x.cuda(), seg.cuda(), w.cuda(), swiglu, (3 * perm + perm % 3).cuda(), None, 3).double().cpu()
    assert torch.equal(pairs, got)
    back = ops.lib().gemm_grouped(x[perm.long()].cuda(), seg.cuda(), w.cuda(), swiglu, None, perm.cuda()).double().cpu()
    assert torch.equal(back[perm.long()], got)


@pytest.mark.gpu
@pytest.mark.parametrize("T,top,E,by_id", [(1, 1, 1, True), (4096, 2, 16, True), (4097, 2, 16, True), (3000, 3, 200, False), (20000, 2, 1024, True), (5, 8, 65, False),
                                             (1024, 1, 64, True), (341, 3, 128, False), (1025, 1, 7, False), (512, 2, 63, True),
                                             (8192, 1, 129, True)])
def test_pairs_sorted_by_expert(T, top, E, by_id):
    g = torch.Generator().manual_seed(T)
    vocab = 50 if by_id else T
    table = torch.randint(-1, E + 1, (vocab, top), generator=g, dtype=torch.int32)
    ids = torch.randint(-2, vocab + 2, (T,), generator=g, dtype=torch.int32) if by_id else None
    seg, order = ops.lib().moe_route(None if ids is None else ids.cuda(), table.cuda(), E)
    e = (table[ids.long().clamp(0, vocab - 1)] if by_id else table).clamp(0, E - 1).reshape(-1)
    assert torch.equal(seg.cpu()[1:].long(), torch.bincount(e, minlength=E).cumsum(0)) and int(seg[0]) == 0
    order = order.cpu().long()
    assert torch.equal(order.sort().values, torch.arange(T * top)) and torch.equal(e[order], e.sort().values)
