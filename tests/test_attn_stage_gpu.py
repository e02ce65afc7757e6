"""Prompt attention with keys and values staged in LDS (csrc/attn_stage.h): sigmoid and masked softmax against the f32 reference of the
same bf16 operands, at the edges of its tiles (16 queries, 32 keys, head sizes 64 / 96 / 128, blocks of 16, 32 and 48)."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops

pytestmark = pytest.mark.gpu


def _step(H, G, dim, vdim, BS, lens, seed, pool=False):
    """(q, k cache, v cache, block tables, cu, ctx) of chunks [(new rows, context)] whose blocks lie scattered in the pool."""
    g = torch.Generator().manual_seed(seed)
    need = [-(-c // BS) for _, c in lens]
    perm, at, NB = torch.randperm(sum(need) + 1, generator=g).to(torch.int32), 0, sum(need) + 1
    bt = torch.zeros(len(lens), max(need) + 1, dtype=torch.int32)
    for b, n in enumerate(need):
        bt[b, :n] = perm[at:at + n]
        at += n
    r = lambda *s: torch.randn(*s, generator=g).to(torch.bfloat16)  # noqa: E731
    q, kc, vc = r(sum(n for n, _ in lens), H * dim + 8), r(NB, G, BS, dim), r(NB, G, vdim, BS)
    pooled = (r(NB, G, BS, dim), r(NB, G, vdim, BS)) if pool else None
    cu = torch.tensor([0] + [n for n, _ in lens]).cumsum(0).to(torch.int32)
    return q, kc, vc, bt, cu, torch.tensor([c for _, c in lens], dtype=torch.int32), pooled


def _both(fn, q, kc, vc, bt, cu, ctx, H, vdim, extra, **kw):
    """The result on the GPU, and the CPU's reference in f32."""
    out = torch.zeros(q.shape[0], H * vdim, dtype=torch.bfloat16, device="cuda")
    dev = lambda t: t.cuda() if torch.is_tensor(t) else tuple(dev(x) for x in t) if isinstance(t, tuple) else t  # noqa: E731
    fn(dev(q), dev(kc), dev(vc), dev(bt), dev(cu), dev(ctx), *[dev(a) for a in extra], out, **{k: dev(v) for k, v in kw.items()})
    ref = torch.zeros(q.shape[0], H * vdim)
    flt = lambda t: t.float() if torch.is_tensor(t) and t.dtype == torch.bfloat16 else tuple(flt(x) for x in t) if isinstance(t, tuple) else t  # noqa: E731
    fn(flt(q), flt(kc), flt(vc), bt, cu, ctx, *[flt(a) for a in extra], ref, **{k: flt(v) for k, v in kw.items()})
    return out.float().cpu(), ref


LENS = [[(1, 1)], [(15, 15), (16, 16), (17, 17)], [(31, 31), (33, 70), (1, 129)], [(64, 64), (65, 200), (100, 100)]]
SHAPES = [(8, 2, 128, 128, 16), (4, 4, 64, 64, 32), (6, 3, 96, 80, 16), (12, 4, 72, 96, 48), (5, 5, 40, 128, 16)]


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("H,G,dim,vdim,BS", SHAPES)
def test_sigmoid(hip, H, G, dim, vdim, BS, lens):
    q, kc, vc, bt, cu, ctx, _ = _step(H, G, dim, vdim, BS, lens, 1)
    g = torch.Generator().manual_seed(2)
    r1, r2, pb = torch.rand(H, generator=g), torch.rand(H, generator=g), torch.randn(H, generator=g) * 0.1
    got, ref = _both(ops.sigmoid_attention_prefill, q, kc, vc, bt, cu, ctx, H, vdim, (H, G, dim, vdim, dim ** -0.5, r1, r2, pb))
    # weights of at most 1 rounded to bf16 (2^-9), times values of size ~1: sqrt(keys) of those errors, six times; and the result's rounding
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 6 * 2.0 ** -9 * float(ctx.max()) ** 0.5).all()
    assert (got - ref).norm() <= 2.0 ** -7 * ref.norm()


@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("mode", ["causal", "chunk", "window", "pooled", "kept", "cap", "sink", "gate", "gates"])
@pytest.mark.parametrize("H,G,dim,vdim,BS", SHAPES[:4])
def test_softmax(hip, H, G, dim, vdim, BS, lens, mode):
    q, kc, vc, bt, cu, ctx, pooled = _step(H, G, dim, vdim, BS, lens, 3, pool=mode == "pooled")
    kind = {"causal": ops.MASK_CAUSAL, "cap": ops.MASK_CAUSAL, "chunk": ops.MASK_CHUNK}.get(mode, ops.MASK_WINDOW)
    g = torch.Generator().manual_seed(4)
    gate = torch.randn(q.shape[0], H * vdim + 3, generator=g).to(torch.bfloat16) if mode.startswith("gate") else None
    kw = {"pooled": dict(pool=pooled + (8,) if pooled else None), "kept": dict(keep_first=3), "cap": dict(softcap=2.0),
          "gates": dict(gate_elem=True)}.get(mode, {})
    size = 24 if mode in ("pooled", "kept") else 37
    got, ref = _both(ops.sink_attention_prefill, q, kc, vc, bt, cu, ctx, H, vdim,
                     (H, G, dim, vdim, torch.rand(H, generator=g) * dim ** -0.5, kind, size, mode == "sink", gate, 3), **kw)
    # weights rounded to bf16 (2^-9 of each) against their f32 sum: 2^-9 of the largest value (below 5), and the result's rounding
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 5 * 2.0 ** -9).all()


@pytest.mark.parametrize("what", ["sigmoid", "window"])
def test_a_later_token_reaches_no_earlier_tile(hip, what):
    """NaN keys and values of token 40 of one chunk: queries of earlier 16-token tiles, and the other chunk, are as without them."""
    H, G, dim, BS = 8, 2, 64, 16
    q, kc, vc, bt, cu, ctx, _ = _step(H, G, dim, dim, BS, [(70, 70), (20, 20)], 5)

    def run(kc, vc):
        out = torch.zeros(90, H * dim, dtype=torch.bfloat16, device="cuda")
        if what == "sigmoid":
            one = torch.ones(H, device="cuda")
            ops.sigmoid_attention_prefill(q.cuda(), kc, vc, bt.cuda(), cu.cuda(), ctx.cuda(), H, G, dim, dim, 0.125, one, one, one, out)
        else:
            ops.sink_attention_prefill(q.cuda(), kc, vc, bt.cuda(), cu.cuda(), ctx.cuda(), H, G, dim, dim, torch.ones(H, device="cuda"),
                                       ops.MASK_WINDOW, 24, False, None, 0, out)
        return out

    clean = run(kc.cuda(), vc.cuda())
    blk = int(bt[0, 40 // BS])
    kc[blk, :, 40 % BS] = float("nan")
    vc[blk, :, :, 40 % BS] = float("nan")
    bad = run(kc.cuda(), vc.cuda())
    assert torch.equal(bad[:32], clean[:32]) and torch.equal(bad[70:], clean[70:]) and bad[40:64].isnan().all()


@pytest.mark.parametrize("dim", [40, 72, 80])
@pytest.mark.parametrize("what", ["sigmoid", "window"])
@pytest.mark.parametrize("decode", [False, True])
def test_infinite_last_columns(hip, what, dim, decode):
    """Infinities in the last columns of a key, of heads that do not fill their fragments: the sigmoid saturates and the softmax gives
    minus infinity no weight, as for every other head size."""
    H, G, BS = 8, 2, 16
    lens = [(1, 30 + b) for b in range(20)] if decode else [(17, 17)] * 130   # (prompts: enough tiles for the staged form)
    q, kc, vc, bt, cu, ctx, _ = _step(H, G, dim, dim, BS, lens, 7)
    q = q.abs()   # (infinity's sign is then the score's)
    kc[:, :, 3, -8:] = float("inf") if what == "sigmoid" else float("-inf")
    kc[:, :, 5, -1] = float("-inf")
    if what == "sigmoid":
        one = torch.ones(H)
        fn, extra = (ops.sigmoid_attention_decode if decode else ops.sigmoid_attention_prefill), (H, G, dim, dim, dim ** -0.5, one, one, one)
    else:
        fn, extra = (ops.sink_attention_decode if decode else ops.sink_attention_prefill), (
            H, G, dim, dim, torch.full((H,), dim ** -0.5), ops.MASK_WINDOW, 24, True, None, 0)
    if decode:
        got, ref = _both(lambda q, kc, vc, bt, cu, ctx, *a: fn(q, kc, vc, bt, ctx, *a), q, kc, vc, bt, cu, ctx, H, dim, extra)
    else:
        got, ref = _both(fn, q, kc, vc, bt, cu, ctx, H, dim, extra)
    assert ref.isfinite().all()
    # as test_sigmoid and test_softmax (weights of at most 1, rounded to bf16)
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 6 * 2.0 ** -9 * float(ctx.max()) ** 0.5).all()


def test_more_tiles_than_a_grid_takes(hip):
    """65,536 tiles of a window: more than one grid dimension holds of the staged kernel's, and a quarter of the other kernel's limit."""
    H, G, dim, BS, long_, short = 1, 1, 64, 16, 65535 * 16, 40
    g = torch.Generator("cuda").manual_seed(9)
    r = lambda *s: torch.randn(*s, generator=g, device="cuda").to(torch.bfloat16)  # noqa: E731
    nb = [long_ // BS, 3]
    kc, vc, q = r(sum(nb), G, BS, dim), r(sum(nb), G, dim, BS), r(long_ + short, H * dim)
    bt = torch.zeros(2, nb[0], dtype=torch.int32, device="cuda")
    bt[0], bt[1, :3] = torch.arange(nb[0]), torch.arange(nb[0], sum(nb))
    scale = torch.full((H,), dim ** -0.5, device="cuda")

    def run(q, bt, lens):
        out = torch.zeros(q.shape[0], H * dim, dtype=torch.bfloat16, device="cuda")
        n = torch.tensor(lens, dtype=torch.int32, device="cuda")
        cu = torch.tensor([0] + lens).cumsum(0).to(torch.int32).cuda()
        return ops.sink_attention_prefill(q, kc, vc, bt, cu, n, H, G, dim, dim, scale, ops.MASK_WINDOW, 16, False, None, 0, out, q_lens_cpu=lens)

    got = run(q, bt, [long_, short])
    tail, alone = run(q[:1600], bt, [1600]), run(q[long_:], bt[1:], [short])
    # the two kernels round the same weights (2^-9 of each) against their f32 sum: as test_softmax
    for a, b in ((got[:1600], tail), (got[long_:], alone)):
        assert ((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs() + 5 * 2.0 ** -8).all()
    last = got[long_ - 16:long_].float()   # the long sequence's last rows, with their keys alone
    k = kc[nb[0] - 2:nb[0], 0].reshape(32, dim).float()
    v = vc[nb[0] - 2:nb[0], 0].transpose(1, 2).reshape(32, dim).float()
    s = q[long_ - 16:long_].float() @ k.T * dim ** -0.5
    d = torch.arange(16, 32, device="cuda")[:, None] - torch.arange(32, device="cuda")[None]
    want = torch.softmax(s.masked_fill((d < 0) | (d >= 16), float("-inf")), 1) @ v
    assert ((last - want).abs() <= 2.0 ** -8 * want.abs() + 5 * 2.0 ** -9).all()


@pytest.mark.parametrize("lens", [[(17, 17)] * 130, [(16, 40), (33, 33), (1, 70)] * 40, [(2100, 2300)]])
@pytest.mark.parametrize("what", ["sigmoid", "causal", "chunk", "kept"])
@pytest.mark.parametrize("H,G,dim,vdim,BS", SHAPES[:4])
def test_many_tiles(hip, H, G, dim, vdim, BS, lens, what):
    """Steps with tiles enough for the staged kernel at every mask (the few of the tests above take it for short windows alone)."""
    rows = sum(n for n, _ in lens)
    if rows == 2100 and (dim, what) != (128, "sigmoid"):
        pytest.skip("one long prompt: one head size (the reference is slow)")
    q, kc, vc, bt, cu, ctx, _ = _step(H, G, dim, vdim, BS, lens, 11)
    g = torch.Generator().manual_seed(12)
    tiles = sum(-(-n // 16) for n, _ in lens)
    if what == "sigmoid":
        assert hip.sigattn_staged(tiles, H, dim, vdim) == (tiles * H >= (1024 if max(dim, vdim) > 96 else 2048))
        r1, r2, pb = torch.rand(H, generator=g), torch.rand(H, generator=g), torch.randn(H, generator=g) * 0.1
        got, ref = _both(ops.sigmoid_attention_prefill, q, kc, vc, bt, cu, ctx, H, vdim, (H, G, dim, vdim, dim ** -0.5, r1, r2, pb))
        assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 6 * 2.0 ** -9 * float(ctx.max()) ** 0.5).all()   # as test_sigmoid
    else:
        kind, kw = {"causal": (ops.MASK_CAUSAL, {}), "chunk": (ops.MASK_CHUNK, {}), "kept": (ops.MASK_WINDOW, dict(keep_first=3))}[what]
        size = 600 if what == "chunk" else 24
        got, ref = _both(ops.sink_attention_prefill, q, kc, vc, bt, cu, ctx, H, vdim,
                         (H, G, dim, vdim, torch.rand(H, generator=g) * dim ** -0.5, kind, size, False, None, 0), **kw)
        assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 5 * 2.0 ** -9).all()   # as test_softmax


@pytest.mark.parametrize("tiles,H,dim,window,staged", [
    (1, 16, 128, 0, False), (32, 16, 128, 0, False), (64, 16, 128, 0, True), (63, 16, 128, 600, False), (1, 16, 128, 512, True), (65535, 1, 64, 512, True),
    (65536, 16, 128, 512, False), (64, 16, 64, 0, False), (128, 16, 64, 0, True), (170, 12, 96, 513, False), (171, 12, 96, 513, True), (4096, 16, 192, 512, False)])
def test_line_between_the_kernels(hip, tiles, H, dim, window, staged):
    """Portions of few tiles over many keys keep the kernel that splits a tile's keys over four waves, on both sides of the measured line."""
    assert hip.sinkattn_staged(tiles, H, dim, dim, window) == staged
    if window == 0:
        assert hip.sigattn_staged(tiles, H, dim, dim) == staged
