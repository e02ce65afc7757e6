"""The one-pass search (csrc/knn.hip knn_scan_kernel) against float64 cosines in stable order: corpora of less than a tile to
more tiles than waves, every width, the most queries and hits it takes, equal rows, and the shapes around it."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops
from llm_kubernetes_minikube_sharp4dev_amd.rag.index import PendingSearch, RagChunk, RagIndex

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("N,D,nq,K", [(1, 128, 1, 1), (15, 256, 16, 8), (17, 384, 3, 5), (65, 512, 16, 8), (4097, 1024, 7, 3),
                                      (20011, 768, 1, 5), (70003, 768, 16, 8), (300, 768, 17, 8), (300, 768, 4, 9), (300, 192, 4, 4), (5, 768, 2, 8)])
def test_scan(hip, N, D, nq, K):
    g = torch.Generator(device=DEV).manual_seed(N)
    c = torch.randn(N, D, device=DEV, generator=g).to(torch.bfloat16)
    c[N // 2:] = c[:N - N // 2].clone()                     # every row of the first half again
    q = torch.randn(nq, D, device=DEV, generator=g).to(torch.bfloat16)
    cn, qn = ops.row_norms(c), ops.row_norms(q)
    ref = (q.double() @ c.double().t()) / (q.double().norm(dim=1)[:, None] * c.double().norm(dim=1)[None] + 1e-9)
    s, i = ops.knn_topk(c, cn, q, qn, K)
    k = min(K, N)
    want = ref.sort(dim=1, descending=True, stable=True)
    # f32 sums of D products and one division: a few 2^-24 of the products' sizes (rows are unit after the division)
    assert ((s[:, :k].double() - want[0][:, :k]).abs() <= 1e-6).all()
    assert ((ref.gather(1, i[:, :k].long()) - want[0][:, :k]).abs() <= 1e-6).all()
    same = s[:, 1:k] == s[:, :k - 1]
    assert (i[:, 1:k][same] > i[:, :k - 1][same]).all()     # equal scores: the lower row first
    assert (i[:, k:] == -1).all() and (s[:, k:] == float("-inf")).all()
    both = ops.knn_packed(c, cn, q, K)
    assert (both is not None) == (nq <= 16 and K <= 8 and D != 192 and K <= N)
    if both is not None:
        assert torch.equal(both[1], i) and ((both[0].view(torch.float32) - s).abs() <= 1e-6).all()


@pytest.mark.parametrize("N,D,nq,K", [(150001, 128, 5, 4), (131072, 128, 1, 8), (100003, 256, 16, 8), (60007, 384, 2, 5), (49169, 512, 1, 1),
                                      (16384, 768, 1, 5), (16385, 768, 2, 8), (33000, 1024, 3, 8)])
def test_scan_ring(hip, N, D, nq, K):
    """Waves of one tile to more than the ring holds, and a wave's last stages, which are waited for together."""
    test_scan(hip, N, D, nq, K)


def test_hits_as_they_arrive(hip):
    """The handle of a search: rows as the packed form's, -1 and rows without a comparable score left out; handles dropped unread."""
    g = torch.Generator(device=DEV).manual_seed(9)
    c = torch.randn(20011, 768, device=DEV, generator=g).to(torch.bfloat16)
    c[5:9] = float("nan")
    few = torch.full((3, 768), float("nan"), device=DEV, dtype=torch.bfloat16)
    few[1] = 1.0
    for corpus in (c, few):
        cn = ops.row_norms(corpus)
        for nq, K in ((1, 1), (1, 3), (16, 3)):
            q = torch.randn(nq, 768, device=DEV, generator=g).to(torch.bfloat16)
            s, i = ops.knn_packed(corpus, cn, q, K).cpu()
            for _ in range(20):
                ops.knn_hits(corpus, cn, q.flip(1).contiguous(), K)      # dropped at once
                h = ops.knn_hits(corpus, cn, q, K)
                h.synchronize()
                assert h.query()
                for k in (K, 1):
                    want = [[(int(b), float(a)) for a, b in zip(x, y) if b >= 0][:k] for x, y in zip(s.view(torch.float32), i)]
                    assert h.rows(k) == want
    assert ops.knn_hits(c, ops.row_norms(c), torch.randn(17, 768, device=DEV).to(torch.bfloat16), 3) is None


def test_a_long_wait_sleeps(hip):
    """A search behind tens of milliseconds of other work: its waiting thread leaves the CPU to others."""
    import time

    g = torch.Generator(device=DEV).manual_seed(4)
    c, q = (torch.randn(n, 768, device=DEV, generator=g).to(torch.bfloat16) for n in (20011, 2))
    cn, m = ops.row_norms(c), torch.randn(8192, 8192, device=DEV, generator=g).to(torch.bfloat16)
    want = ops.knn_packed(c, cn, q, 5)
    m @ m
    torch.cuda.synchronize()
    for _ in range(40):
        y = m @ m
    h = ops.knn_hits(c, cn, q, 5)
    t, cpu = time.perf_counter(), time.thread_time()
    h.synchronize()
    t, cpu = time.perf_counter() - t, time.thread_time() - cpu
    assert t > 0.01, t   # (40 products of 1.1 TFLOP are 17 ms at the card's peak)
    assert cpu < 0.3 * t, (cpu, t)
    assert [[i for i, _ in r] for r in h.rows(5)] == want[1].tolist()
    del y


def test_index_search_agrees(hip):
    """RagIndex gives the same hits whether or not the one-pass search takes the shape."""
    g = torch.Generator(device=DEV).manual_seed(3)
    c = torch.randn(3000, 768, device=DEV, generator=g).to(torch.bfloat16)
    q = torch.randn(20, 768, device=DEV, generator=g)
    index = RagIndex(None, backend="gpu", device=DEV)
    index.chunks = [RagChunk("d#0", "d", "")] * 3000
    index.set_gpu_corpus(c)
    many, few = index.search_vectors(q, 6), [index.search_vectors(q[j:j + 1], 6)[0] for j in range(20)]
    assert [[i for i, _ in h] for h in many] == [[i for i, _ in h] for h in few]
    assert max(abs(a - b) for x, y in zip(many, few) for (_, a), (_, b) in zip(x, y)) <= 1e-6


def test_hits_in_pinned_memory(hip):
    """The form that leaves the hits on the host: the device form's, also when the result of a search before it was dropped unread."""
    g = torch.Generator(device=DEV).manual_seed(4)
    c = torch.randn(20011, 768, device=DEV, generator=g).to(torch.bfloat16)
    cn = ops.row_norms(c)
    for nq in (1, 5, 16):
        q = torch.randn(nq, 768, device=DEV, generator=g).to(torch.bfloat16)
        want, idx = ops.knn_packed(c, cn, q, 5).cpu()
        for _ in range(3):
            ops.knn_hits(c, cn, q.flip(1).contiguous(), 5)
            got = ops.knn_hits(c, cn, q, 5)
            torch.cuda.current_stream().synchronize()
            assert got.query() and got.rows(5) == [list(zip(i, s)) for i, s in zip(idx.tolist(), want.view(torch.float32).tolist())]


def test_a_search_waits_for_its_own_work(hip, monkeypatch):
    """Work that another thread enqueues on the stream behind the search's kernels is not waited for."""
    g = torch.Generator(device=DEV).manual_seed(6)
    c, q = (torch.randn(n, 768, device=DEV, generator=g).to(torch.bfloat16) for n in (3000, 2))
    index = RagIndex(None, backend="gpu", device=DEV)
    index.chunks = [RagChunk("d#0", "d", "")] * 3000
    index.set_gpu_corpus(c)
    want, result = index.search_vectors(q, 5), PendingSearch.result
    big, out, behind = torch.ones(8192, 8192, device=DEV).bfloat16(), torch.empty(8192, 8192, device=DEV).bfloat16(), torch.cuda.Event()
    torch.mm(big, big, out=out)
    torch.cuda.synchronize()

    def work_before_the_wait(pending):
        for _ in range(200):   # 1.1 TFLOP each: at least 0.08 s
            torch.mm(big, big, out=out)
        behind.record()
        return result(pending)

    monkeypatch.setattr(PendingSearch, "result", work_before_the_wait)
    got = index.search_vectors(q, 5)
    done = behind.query()
    torch.cuda.synchronize()
    assert got == want and not done
