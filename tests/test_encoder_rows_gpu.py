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


def _double_forward(m, ids, pos, lens):
    """The encoder's rows in float64, of the same bf16 weights and nothing rounded on the way."""
    F, cfg = torch.nn.functional, m.cfg
    d = lambda t: t.double()  # noqa: E731
    ln = lambda x, w, b: F.layer_norm(x, (cfg.hidden,), d(w), d(b), cfg.norm_eps)  # noqa: E731
    h = ln(d(m.tok)[ids.long()] + d(m.pos)[pos.long()] + d(m.typ)[0], m.emb_ln_w, m.emb_ln_b)
    for L in m.layers:
        q, k, v = (t.view(-1, m.nh, m.D).transpose(0, 1) for t in F.linear(h, d(L.qkv), d(L.qkv_b)).chunk(3, 1))
        at, out = 0, []
        for n in lens:
            s = slice(at, at + n)
            p = torch.softmax(q[:, s] @ k[:, s].transpose(1, 2).contiguous() * m.scale, -1)
            out.append((p @ v[:, s]).transpose(0, 1).reshape(n, -1))
            at += n
        h = ln(F.linear(torch.cat(out), d(L.o), d(L.o_b)) + h, L.ln1_w, L.ln1_b)
        h = ln(F.linear(F.gelu(F.linear(h, d(L.fc1), d(L.fc1_b))), d(L.fc2), d(L.fc2_b)) + h, L.ln2_w, L.ln2_b)
    return h


def _inputs(lens):
    ids = torch.randint(1000, 30000, (sum(lens),), dtype=torch.int32, device="cuda")
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).cuda()
    return ids, torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda(), pos


class _Spy:
    """The native library, counting calls by name."""

    def __init__(self, lib):
        self.lib, self.calls = lib, []

    def __getattr__(self, name):
        f = getattr(self.lib, name)

        def call(*a, **k):
            if not name.endswith("_supported"):
                self.calls.append((name, a[3]) if name == "rows_linear" else name)
            return f(*a, **k)
        return call


@pytest.mark.parametrize("name,lens,norms,attention", [
    ("bge-base", [1], True, True), ("bge-base", [19], True, True), ("bge-base", [32], True, True), ("bge-base", [33], False, False),
    ("bge-base", [64], False, False), ("bge-base", [5, 9, 17], True, False), ("bge-base", [5, 9, 33], False, False),
    ("minilm-l6", [16], True, False), ("minilm-l6", [17], False, False), ("bert-tiny", [16], True, True), ("bert-tiny", [17], False, False), ("bert-tiny", [4, 12], True, False)])
def test_short_texts_take_the_fused_layers(hip, monkeypatch, name, lens, norms, attention):
    """Which passes run the norms, and the attention of one text, inside the projections; their rows against float64, no farther from it
    than the layers apart."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    from llm_kubernetes_minikube_sharp4dev_amd.models import build_encoder

    m = build_encoder(name, device="cuda").random_init(3)
    ids, cu, pos = _inputs(lens)
    spy = _Spy(hip)
    monkeypatch.setattr(ops, "lib", lambda: spy)
    got = m(ids, cu, pos, lens, pool=False)
    n = m.cfg.num_layers
    assert spy.calls.count("ln_linear") == (2 * n - 1 if norms else 0)
    assert spy.calls.count("attn_linear") == (n if attention else 0)
    assert spy.calls.count(("rows_linear", 5)) == ((n if attention else 2 * n) if norms else 0)
    monkeypatch.setattr(ops, "ENCODER_ROWS", 0)
    apart, want = m(ids, cu, pos, lens, pool=False), _double_forward(m, ids, pos, lens)
    e, a = ((y.double() - want).norm() / want.norm() for y in (got, apart))
    # each layer rounds eight tensors on the way to bf16, 2^-9 of a value at most and a third of that on average, alike on both ways
    assert e <= (8 * n) ** 0.5 * 2.0 ** -9 and e <= 1.2 * a + 2.0 ** -12, (float(e), float(a))


def test_product_plus_residual_routes(hip, monkeypatch):
    """``linear_add`` and ``linear_pair``: one launch where the few-row kernel takes the operands, the same rows where it does not."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    g = torch.Generator("cuda").manual_seed(5)
    x, w, b, r = _r(g, 19, 768), _r(g, 768, 768, scale=768 ** -0.5), _r(g, 768), _r(g, 19, 768)
    odd = torch.empty(19, 769, dtype=torch.bfloat16, device="cuda")[:, :768].copy_(x)   # rows that begin between two 16-byte lines
    spy = _Spy(hip)
    monkeypatch.setattr(ops, "lib", lambda: spy)
    one = ops.linear_add(x, w, b, r)
    assert spy.calls == [("rows_linear", 5)]
    want = x.double() @ w.double().T + b.double()
    for y in (one, ops.linear_add(odd, w, b, r), ops.linear_add(x, w, torch.stack([b, b], 1)[:, 0], r)):
        # the product's and the sum's rounding
        assert ((y.double() - want - r.double()).abs() <= EPS * (want.abs() + (want + r.double()).abs()) + 1e-4).all()
    spy.calls.clear()
    w2 = _r(g, 768, 768, scale=768 ** -0.5)
    y1, y2 = ops.linear_pair(x, w, r, w2)
    assert spy.calls == ["rows_pair"]
    z1, z2 = ops.linear_pair(odd, w, r, w2)
    assert spy.calls.count("rows_pair") == 1
    for y, z, p in ((y1, z1, x.double() @ w.double().T), (y2, z2, r.double() @ w2.double().T)):
        assert ((y.double() - p).abs() <= EPS * p.abs() + 1e-4).all() and ((z.double() - p).abs() <= EPS * p.abs() + 1e-4).all()


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


@pytest.mark.parametrize("name", ["minilm-l6", "bert-tiny", "nomic-tiny"])
@pytest.mark.parametrize("lens", [[9], [3, 9], [40], [30, 1, 12]])
def test_lengths_from_the_device(hip, name, lens):
    """``lens_cpu`` may be left out: the lengths are read from ``cu``, or only the given tiles are used."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    from llm_kubernetes_minikube_sharp4dev_amd.models import build_encoder

    m = build_encoder(name, device="cuda").random_init(3)
    ids, cu, pos = _inputs(lens)
    want = m(ids, cu, pos, lens)
    assert torch.equal(m(ids, cu, pos, None), want)
    got = m(ids, cu, pos, None, tiles=ops.device_tiles(lens, lens, 1, False, m.D, ids.device))
    # (one text of heads of 64 has its attention inside a projection where its length is known: eight bf16 roundings a layer, 2^-9 of a value at
    # most, on either way)
    assert (got - want).norm() <= 2 * (8 * m.cfg.num_layers) ** 0.5 * 2.0 ** -9 * want.norm()


def test_query_graphs_on_the_callers_streams(hip):
    """Replays enqueued from several streams and threads at once: the graphs share buffers, every vector is its own text's, and later work of
    a caller's stream finds it there."""
    import threading

    from llm_kubernetes_minikube_sharp4dev_amd.engine.embed_engine import EmbeddingEngine
    from llm_kubernetes_minikube_sharp4dev_amd.models import build_encoder

    m = build_encoder("bert-tiny", device="cuda").random_init(3)
    eager, g = EmbeddingEngine(m, None, "e"), torch.Generator().manual_seed(2)
    texts = [torch.randint(1000, 30000, (n,), generator=g).tolist() for n in (3, 9, 9, 14, 20)]
    want = [eager.embed_ids([t]) for t in texts]
    eng = EmbeddingEngine(m, None, "g")
    assert eng.capture_queries(max_len=16, dtypes=(torch.float32,)) == 16
    got = {}

    def caller(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for r in range(20):
                for k, t in enumerate(texts):
                    got[i, r, k] = eng.embed_ids([t]).clone()
            torch.cuda.current_stream().synchronize()

    threads = [threading.Thread(target=caller, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for r in range(20):
        for k, t in enumerate(texts):
            got["main", r, k] = eng.embed_ids([t]) * 1.0
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert len(got) == 4 * 20 * len(texts)
    for (_, _, k), v in got.items():
        assert torch.equal(v, want[k])


@pytest.mark.parametrize("n", [1, 63, 64, 65])
def test_host_ids(hip, n):
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    buf, host = torch.full((n + 1,), -7, dtype=torch.int32, device="cuda"), torch.arange(n, dtype=torch.int32) * 3 - 5
    ops.set_ids(buf[:n], host)
    keep = host.clone()
    host.zero_()   # (the values have been taken)
    assert torch.equal(buf[:n].cpu(), keep) and int(buf[n]) == -7


@pytest.mark.parametrize("M", [8, 9, 10, 31, 32])
def test_two_row_tiles(hip, M):
    """Both sides of the lines where a workgroup takes half the rows, even and odd numbers of them, and widths that the wider column tile does not divide."""
    for K, N, gelu in ((768, 3072, True), (384, 1152, False), (64, 32, True), (320, 48, False)):
        test_ln_linear(hip, M, K, N, gelu)
    for nh, N in ((12, 768), (7, 448), (1, 16)):
        test_attn_linear(hip, M, nh, N)
