"""Model parity vs HuggingFace transformers (same random weights, fp32, CPU) and
engine consistency (paged KV, chunked prefill, prefix caching, preemption)."""
import pytest
import torch

transformers = pytest.importorskip("transformers")

from llm_kubernetes_minikube_sharp4dev_amd.engine.llm_engine import LLMEngine
from llm_kubernetes_minikube_sharp4dev_amd.engine.sampling import SamplingParams
from llm_kubernetes_minikube_sharp4dev_amd.models import build_decoder, build_encoder
from llm_kubernetes_minikube_sharp4dev_amd.models.configs import DecoderConfig, EncoderConfig


def _hf_llama():
    cfg = transformers.LlamaConfig(vocab_size=512, hidden_size=128, intermediate_size=256, num_hidden_layers=2,
                                   num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=1024,
                                   rope_theta=10000.0, rms_norm_eps=1e-5, tie_word_embeddings=False)
    torch.manual_seed(0)
    m = transformers.LlamaForCausalLM(cfg).eval()
    ours = DecoderConfig("t", "llama", 2, 128, 4, 2, 32, 256, 512, max_position=1024, rope_theta=10000.0)
    return m, ours


def _engine(model, **kw):
    kw.setdefault("num_blocks", 128)
    kw.setdefault("eos_ids", set())
    return LLMEngine(model, None, block_size=16, max_model_len=512, max_num_seqs=8, **kw)


def test_llama_matches_hf():
    hf, cfg = _hf_llama()
    m = build_decoder(cfg, dtype=torch.float32)
    m.load_hf_state_dict(hf.state_dict())
    prompt = [5, 17, 99, 3, 250, 7, 7, 1, 400, 33, 21, 8, 2, 9, 11, 60, 61, 62, 63]
    with torch.no_grad():
        ref = hf.generate(torch.tensor([prompt]), max_new_tokens=12, do_sample=False)[0, len(prompt):].tolist()
        hf_logits = hf(torch.tensor([prompt])).logits[0, -1]
    eng = _engine(m)
    seq = eng.generate([prompt], SamplingParams.greedy(12))[0]
    assert seq.output_ids == ref
    # logits of the first step
    eng2 = _engine(m)
    s2 = eng2.add_request(prompt, SamplingParams.greedy(1))
    eng2._drain_inbox()
    batch = eng2.scheduler.schedule()
    rows, lg = eng2.runner.forward_logits(batch.items)
    assert torch.allclose(lg[0], hf_logits, atol=1e-4, rtol=1e-4)


def test_opt_matches_hf():
    cfg = transformers.OPTConfig(vocab_size=512, hidden_size=64, ffn_dim=128, num_hidden_layers=2,
                                 num_attention_heads=2, max_position_embeddings=256, word_embed_proj_dim=64,
                                 do_layer_norm_before=True, enable_bias=True)
    torch.manual_seed(1)
    hf = transformers.OPTForCausalLM(cfg).eval()
    ours = DecoderConfig("t", "opt", 2, 64, 2, 2, 32, 128, 512, max_position=256, tie_word_embeddings=True,
                         activation="relu", bias=True)
    m = build_decoder(ours, dtype=torch.float32)
    m.load_hf_state_dict(hf.state_dict())
    prompt = [2, 45, 100, 7, 8, 300, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22]
    with torch.no_grad():
        ref = hf.generate(torch.tensor([prompt]), max_new_tokens=10, do_sample=False)[0, len(prompt):].tolist()
    seq = _engine(m).generate([prompt], SamplingParams.greedy(10))[0]
    assert seq.output_ids == ref


@pytest.mark.parametrize("pooling", ["cls", "mean"])
def test_bert_matches_hf(pooling):
    cfg = transformers.BertConfig(vocab_size=300, hidden_size=64, num_hidden_layers=2, num_attention_heads=2,
                                  intermediate_size=128, max_position_embeddings=128, hidden_act="gelu")
    torch.manual_seed(2)
    hf = transformers.BertModel(cfg, add_pooling_layer=False).eval()
    ours = EncoderConfig("t", "bert", 2, 64, 2, 128, 300, max_position=128, pooling=pooling)
    m = build_encoder(ours, dtype=torch.float32)
    m.load_hf_state_dict(hf.state_dict())
    seqs = [[1, 5, 9, 22, 2], [1, 7, 2], [1, 100, 101, 102, 103, 104, 105, 2]]
    ids = torch.tensor(sum(seqs, []), dtype=torch.int32)
    cu = torch.tensor([0, 5, 8, 16], dtype=torch.int32)
    pos = torch.tensor(sum([list(range(len(s))) for s in seqs], []), dtype=torch.int32)
    emb = m(ids, cu, pos, [len(s) for s in seqs])
    for i, s in enumerate(seqs):
        with torch.no_grad():
            h = hf(torch.tensor([s])).last_hidden_state[0]
        v = h[0] if pooling == "cls" else h.mean(0)
        v = v / v.norm()
        assert torch.allclose(emb[i], v, atol=1e-4), (i, (emb[i] - v).abs().max())


def test_chunked_prefill_prefix_cache_and_preemption_consistent():
    m = build_decoder("llama-tiny", dtype=torch.float32)
    prompts = [list(range(3, 3 + n)) for n in (70, 33, 5, 100)]
    ref = [s.output_ids for s in _engine(m).generate(prompts, SamplingParams.greedy(10))]
    # tiny token budget -> chunked prefill interleaved with decode
    chunked = _engine(m, max_num_batched_tokens=24)
    assert [s.output_ids for s in chunked.generate(prompts, SamplingParams.greedy(10))] == ref
    # prefix cache: a second request sharing 64 tokens reuses 4 blocks
    eng = _engine(m)
    eng.generate([prompts[0]], SamplingParams.greedy(10))
    s = eng.generate([prompts[0][:64] + [7, 8, 9]], SamplingParams.greedy(4))[0]
    assert s.num_cached_prefix == 64
    fresh = _engine(m, max_num_batched_tokens=4096).generate([prompts[0][:64] + [7, 8, 9]],
                                                              SamplingParams.greedy(4))[0]
    assert s.output_ids == fresh.output_ids
    # KV pool too small for all sequences at once -> preemption + recompute, same answers
    ref30 = [s.output_ids for s in _engine(m).generate(prompts, SamplingParams.greedy(30))]
    small = _engine(m, num_blocks=10)
    out = small.generate(prompts, SamplingParams.greedy(30))
    assert [x.output_ids for x in out] == ref30
    assert sum(x.num_preemptions for x in out) > 0


def test_unified_mixed_attention_matches_split(monkeypatch):
    """LK_UNIFIED_ATTN: a mixed step's decode rows join the prompt chunks as one-token sequences
    of ONE flash-attention call (combined cu / ctx / block tables built by ModelRunner._meta);
    tokens equal the split path (flash for the chunks + paged decode for the rows), with
    chunked prefill interleaved with decode and jump-forward-free greedy decoding."""
    from llm_kubernetes_minikube_sharp4dev_amd.models import attention

    m = build_decoder("llama-tiny", dtype=torch.float32)
    prompts = [list(range(3, 3 + n)) for n in (70, 33, 5, 100, 17)]
    ref = [s.output_ids for s in _engine(m, max_num_batched_tokens=24).generate(prompts, SamplingParams.greedy(12))]
    seen = []
    real = attention.ops.flash_prefill

    def spy(q, *a, **kw):
        seen.append(q.shape[0])
        return real(q, *a, **kw)

    monkeypatch.setattr(attention, "UNIFIED_ATTN", True)
    monkeypatch.setattr(attention.ops, "flash_prefill", spy)
    eng = _engine(m, max_num_batched_tokens=24)
    out = [s.output_ids for s in eng.generate(prompts, SamplingParams.greedy(12))]
    assert out == ref
    # some steps were mixed and ran as one launch covering prompt and decode rows
    assert getattr(eng.runner, "unified_attn_steps", 0) > 0 and seen and max(seen) <= 24


def _run_pipelined(eng, prompts, params_fn, stagger: int = 0):
    """Drive eng with step_pipelined (requests i >= 2 admitted `stagger` iterations apart)."""
    seqs, pending, it = [], list(enumerate(prompts)), 0
    while pending or eng.has_work():
        while pending and (not stagger or it >= stagger * pending[0][0] or pending[0][0] < 2):
            i, p = pending.pop(0)
            seqs.append((i, eng.add_request(p, params_fn())))
        if eng.has_work():
            eng.step_pipelined()
        else:
            eng.flush()
        it += 1
    eng.flush()
    return [s.output_ids for _, s in sorted(seqs, key=lambda x: x[0])]


def test_pipelined_steps_match_synchronous():
    """step_pipelined (step N+1 launched before step N's ids reach the host, decode
    inputs gathered on the device) gives exactly the synchronous engine's tokens:
    chunked prefill, staggered admission, EOS stops mid-flight, a history-dependent
    logits processor, and preemption under a tiny KV pool."""
    m = build_decoder("llama-tiny", dtype=torch.float32)
    prompts = [list(range(3, 3 + n)) for n in (70, 33, 5, 100, 17)]

    def proc(hist):  # history-dependent constraint (like the tool-call grammar)
        return list(range(1 + (len(hist) % 5), m.cfg.vocab_size, 3))

    cases = [
        (lambda: SamplingParams.greedy(12), {}),
        (lambda: SamplingParams.greedy(12, logits_processor=proc), {"max_num_batched_tokens": 24}),
        (lambda: SamplingParams.greedy(30), {"num_blocks": 10}),
    ]
    for params_fn, kw in cases:
        ref = [s.output_ids for s in _engine(m, **kw).generate(prompts, params_fn())]
        assert _run_pipelined(_engine(m, **kw), prompts, params_fn) == ref
        assert _run_pipelined(_engine(m, **kw), prompts, params_fn, stagger=3) == ref
    # EOS stop: pick a token the reference emits mid-sequence
    base = [s.output_ids for s in _engine(m).generate(prompts, SamplingParams.greedy(12))]
    eos = base[0][4]
    ref = [s.output_ids for s in _engine(m, eos_ids={eos}).generate(prompts, SamplingParams.greedy(12))]
    assert any(len(r) < 12 for r in ref)
    eng = LLMEngine(m, None, block_size=16, max_model_len=512, max_num_seqs=8, eos_ids={eos}, num_blocks=128)
    assert _run_pipelined(eng, prompts, lambda: SamplingParams.greedy(12)) == ref
    assert eng.allocator.usage() == 0.0 or not eng.scheduler.running


@pytest.mark.parametrize("ext_as_decode", [16, 0])
def test_jump_forward_matches_step_by_step(monkeypatch, ext_as_decode):
    """Grammar jump-forward (tokens with a one-id mask appended by the host and run as an
    extend chunk -- as causal decode rows, or as a prefill chunk) gives exactly the
    step-by-step tokens, synchronous and pipelined, under chunked prefill and preemption,
    with fewer engine steps per request; the last token of every request is still sampled."""
    from llm_kubernetes_minikube_sharp4dev_amd.engine import llm_engine, model_runner

    monkeypatch.setattr(model_runner, "EXTEND_AS_DECODE", ext_as_decode)

    m = build_decoder("llama-tiny", dtype=torch.float32)
    V = m.cfg.vocab_size
    prompts = [list(range(3, 3 + n)) for n in (70, 33, 5, 100, 17)]

    def proc(hist):  # runs of forced tokens (a literal) between free choices
        n = len(hist)
        if n % 7 in (2, 3, 4) or (n % 11 == 5):
            return [(n * 37 + 11) % V]
        return list(range(1 + (n % 5), V, 3))

    cases = [
        (lambda: SamplingParams.greedy(20, logits_processor=proc), {}),
        (lambda: SamplingParams.greedy(20, logits_processor=proc), {"max_num_batched_tokens": 24}),
        (lambda: SamplingParams.greedy(30, logits_processor=proc), {"num_blocks": 10}),
    ]
    for params_fn, kw in cases:
        monkeypatch.setattr(llm_engine, "JUMP_FORWARD", False)
        off = _engine(m, **kw).generate(prompts, params_fn())
        ref = [s.output_ids for s in off]
        assert all(s.jumped == 0 for s in off)
        monkeypatch.setattr(llm_engine, "JUMP_FORWARD", True)
        on = _engine(m, **kw).generate(prompts, params_fn())
        assert [s.output_ids for s in on] == ref
        assert all(s.jumped > 0 for s in on)
        assert sum(s.steps_run for s in on) < sum(s.steps_run for s in off)
        assert _run_pipelined(_engine(m, **kw), prompts, params_fn) == ref
        assert _run_pipelined(_engine(m, **kw), prompts, params_fn, stagger=3) == ref
    # a forced final token is not appended by the host: with every token forced the request
    # still takes its last token from the sampler (no forward pass of the step-by-step run skipped)
    eng = _engine(m)
    s = eng.generate([prompts[2]], SamplingParams.greedy(6, logits_processor=lambda h: [9]))[0]
    assert s.output_ids == [9] * 6 and s.jumped == 4  # first sampled, 4 jumped, last sampled
    assert eng.allocator.usage() == 0.0 or not eng.scheduler.running


def test_prefill_hold_back_same_tokens_fuller_steps(monkeypatch):
    """Prefill hold-back (LK_PREFILL_HOLD): with enough decode rows running, new prompts wait
    until they fill the step's token budget (or the hold limit expires): same greedy tokens
    as the eager scheduler, and every step that carries prefill is full unless the hold
    expired or nothing else was running."""
    m = build_decoder("llama-tiny", dtype=torch.float32)
    monkeypatch.setenv("LK_HOLD_MIN_DECODE", "2")
    prompts = [list(range(3, 3 + n)) for n in (40, 33, 25, 30, 17, 22, 35, 28)]

    def run(hold):
        eng = _engine(m, max_num_batched_tokens=64, prefill_hold=hold, token_align=0)
        eng.step_trace = []
        seqs = [eng.add_request(p, SamplingParams.greedy(12)) for p in prompts[:3]]
        it = 0
        while eng.has_work() or len(seqs) < len(prompts):
            if it % 3 == 2 and len(seqs) < len(prompts):  # arrivals while others decode
                seqs.append(eng.add_request(prompts[len(seqs)], SamplingParams.greedy(12)))
            eng.step()
            it += 1
        return [s.output_ids for s in seqs], eng.step_trace

    ref, tr0 = run(0)
    got, tr1 = run(4)
    assert got == ref
    part0 = sum(1 for t in tr0 if 0 < t[0] and t[0] + t[1] < 64)
    part1 = sum(1 for t in tr1 if 0 < t[0] and t[0] + t[1] < 64)
    assert part1 < part0, (part0, part1)


def test_prefill_hold_small_fill_same_tokens(monkeypatch):
    """LK_HOLD_SMALL: a held step still takes prompt tokens up to hold_small rows in total -- same
    greedy tokens as the eager scheduler, no held step past hold_small rows, and prompt tokens do
    ride in steps the plain hold-back leaves decode-only."""
    m = build_decoder("llama-tiny", dtype=torch.float32)
    monkeypatch.setenv("LK_HOLD_MIN_DECODE", "2")
    prompts = [list(range(3, 3 + n)) for n in (40, 33, 25, 30, 17, 22, 35, 28)]

    def run(hold, small):
        monkeypatch.setenv("LK_HOLD_SMALL", str(small))
        eng = _engine(m, max_num_batched_tokens=64, prefill_hold=hold, token_align=0)
        eng.step_trace = []
        seqs = [eng.add_request(p, SamplingParams.greedy(12)) for p in prompts[:3]]
        it, held_sizes = 0, []
        while eng.has_work() or len(seqs) < len(prompts):
            if it % 3 == 2 and len(seqs) < len(prompts):
                seqs.append(eng.add_request(prompts[len(seqs)], SamplingParams.greedy(12)))
            held_before = eng.scheduler._held
            eng.step()
            if eng.scheduler._held > held_before:  # this step held prefill back
                held_sizes.append(eng.step_trace[-1][0] + eng.step_trace[-1][1])
            it += 1
        return [s.output_ids for s in seqs], eng.step_trace, held_sizes

    ref, _, _ = run(0, 0)
    got0, tr0, held0 = run(4, 0)
    got1, tr1, held1 = run(4, 8)
    assert got0 == ref and got1 == ref
    assert held1 and max(held1) <= 8, held1
    small0 = sum(t[0] for t in tr0 if t[0] + t[1] <= 8)
    small1 = sum(t[0] for t in tr1 if t[0] + t[1] <= 8)
    assert small1 > small0, (small0, small1)


def test_small_step_bucket_alignment_same_tokens(monkeypatch):
    """LK_SMALL_STEP_ALIGN: a weight-streaming step (<= the largest bucket in rows) with decode
    rows trims prompt prefill to the row bucket its decode rows need (the trimmed tokens lead the
    next step): same greedy tokens as without it, and no step mixes decode rows with prefill
    past that bucket."""
    m = build_decoder("llama-tiny", dtype=torch.float32)
    prompts = [list(range(3, 3 + n)) for n in (40, 33, 25, 30, 17, 22, 35, 28)]

    def run(buckets):
        monkeypatch.setenv("LK_SMALL_STEP_ALIGN", buckets)
        eng = _engine(m, max_num_batched_tokens=64, token_align=0)
        eng.step_trace = []
        seqs = [eng.add_request(p, SamplingParams.greedy(12)) for p in prompts[:3]]
        it = 0
        while eng.has_work() or len(seqs) < len(prompts):
            if it % 3 == 2 and len(seqs) < len(prompts):
                seqs.append(eng.add_request(prompts[len(seqs)], SamplingParams.greedy(12)))
            eng.step()
            it += 1
        return [s.output_ids for s in seqs], eng.step_trace

    ref, _ = run("0")
    got, tr = run("4,8,16")
    assert got == ref
    trimmed = 0
    for npre, ndec, *_ in tr:  # (prefill tokens, decode rows, ...)
        if npre and ndec and npre + ndec <= 16:  # a step the alignment applies to
            cap = next(b for b in (4, 8, 16) if b >= ndec)
            assert npre + ndec <= cap, (npre, ndec)
            trimmed += npre + ndec == cap
    assert trimmed  # the policy engaged


def test_fused_decode_ops_cpu_fallback():
    """ops.linear_add_rmsnorm / ops.linear_rope_kv on CPU tensors are the unfused
    reference ops (the HIP fusions only exist for split-K decode shapes on the GPU)."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    torch.manual_seed(0)
    x, w = torch.randn(5, 64), torch.randn(32, 64) * 0.1
    g, res = torch.rand(32) + 0.5, torch.randn(5, 32)
    r1, r2 = res.clone(), res.clone()
    y = ops.linear_add_rmsnorm(x, w, r1, g, 1e-5)
    y2 = ops.rmsnorm(ops.linear(x, w), g, 1e-5, residual=r2)
    assert torch.equal(y, y2) and torch.equal(r1, r2)

    Hq, Hkv, D, BS, NB = 4, 2, 16, 4, 8
    wq = torch.randn((Hq + 2 * Hkv) * D, 64) * 0.1
    pos = torch.arange(5, dtype=torch.int32)
    cs = ops.rope_cos_sin(64, D, 10000.0)
    kc, vc = torch.zeros(NB, Hkv, BS, D), torch.zeros(NB, Hkv, BS, D)
    kc2, vc2 = kc.clone(), vc.clone()
    slots = torch.tensor([0, 1, 2, 5, 9], dtype=torch.int32)
    q1 = ops.linear_rope_kv(x, wq, pos, cs, Hq, Hkv, D, kc, vc, slots)
    q2 = ops.linear(x, wq)
    ops.rope_kv_(q2, pos, cs, Hq, Hkv, D, kc2, vc2, slots)
    assert torch.equal(q1, q2) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


def test_gemm_split_k_policy():
    """Prefill-GEMM dispatch (pure host logic): split-K only where the 256-row tile grid covers
    at most half of the 256 CUs, never for SwiGLU, at most 4 splits of >= 8 K-tiles each
    (profiles/r2_gemm_splitk.md)."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    assert ops._gemm_default(1024, 4096, 4096, 0) == (ops._gemm_sched(4096), 256, 4)
    if ops.GEMM_SCHED is None:  # default schedule policy: static-priority 4-phase for the decoder's K
        assert ops._gemm_sched(4096) == 2 and ops._gemm_sched(14336) == 2 and ops._gemm_sched(768) == 0
    assert ops._gemm_default(2048, 4096, 14336, 0)[2] == 2
    assert ops._gemm_default(1024, 6144, 4096, 0)[1:] == (192, 2)
    assert ops._gemm_default(4096, 1280, 8192, 0)[2] == 3
    assert ops._gemm_default(8192, 4096, 4096, 0)[2] == 1
    assert ops._gemm_default(2560, 4096, 4096, 2)[2] == 1
    assert ops._gemm_default(2560, 4096, 14336, 0)[2] == 3  # 160 tiles, long K
    assert ops._gemm_default(2816, 4096, 14336, 0)[2] == 1  # 176 tiles
    assert ops._gemm_default(512, 28672, 4096, 1)[2] == 1  # SwiGLU: single pass
    assert ops._gemm_default(256, 768, 768, 2)[2] == 1  # 12 K-tiles: < 8 per split at S 2


@pytest.mark.parametrize("prefix_caching", [True, False])
def test_decode_reads_past_the_caches_only_without_prefix_reuse(monkeypatch, prefix_caching):
    """Decode attention is told that no cache block belongs to two sequences exactly where prefixes are not reused."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    hf, cfg = _hf_llama()
    m = build_decoder(cfg, dtype=torch.float32)
    m.load_hf_state_dict(hf.state_dict())
    eng, told, fn = _engine(m, enable_prefix_caching=prefix_caching), [], ops.paged_decode
    monkeypatch.setattr(ops, "paged_decode", lambda *a, own_blocks=None, **k: told.append(own_blocks) or fn(*a, own_blocks=own_blocks, **k))
    eng.generate([[5, 17, 99, 3] * 5, [5, 17, 99, 3] * 5 + [7]], SamplingParams(max_tokens=3, temperature=0.0))
    assert told and all(t is (not prefix_caching) for t in told)


def test_gemm1w_default_policy(monkeypatch):
    """Fallback policy (shapes without a measured entry): 256-wide prefill tiles go to the
    one-wave-per-SIMD kernel (variant 3, csrc/gemm1w.hip) once they fill a wave of 256 CUs, its
    192-row tiles (variant 4) where 256-row tiles would leave over a third of one wave idle; QKV
    at M 4096 keeps gemm.hip's 192-wide tiles (2 whole waves), split-K shapes stay on gemm.hip;
    LK_GEMM1W=0 turns it off."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "GEMM1W", True)
    assert ops._gemm_default(4096, 4096, 4096, 0) == (3, 256, 1)      # O
    assert ops._gemm_default(4096, 4096, 14336, 6) == (3, 256, 1)     # down, RESID
    assert ops._gemm_default(4096, 28672, 4096, 1) == (3, 256, 1)     # gate_up + SwiGLU
    assert ops._gemm_default(4096, 6144, 4096, 7)[:2] == (ops._gemm_sched(4096), 192)  # QKV: 2 whole waves
    assert ops._gemm_default(8192, 6144, 4096, 0) == (3, 256, 1)      # tie on waves -> 256
    assert ops._gemm_default(2664, 4096, 4096, 0) == (4, 256, 1)      # 176 tiles -> 224 of 192 rows
    assert ops._gemm_default(1024, 4096, 4096, 0)[0] not in ops.GEMM1W_BM  # 64 tiles: split-K on gemm.hip
    assert {(3, 256), (4, 256), (5, 256)} <= set(ops._gemm_configs(4096, 0))
    assert (3, 256) in ops._gemm_configs(28672, 1)
    assert all(c[0] not in ops.GEMM1W_BM for c in ops._gemm_configs(1152, 0))  # no 256-wide tile
    monkeypatch.setattr(ops, "GEMM1W", False)
    assert ops._gemm_default(4096, 4096, 4096, 0)[0] == ops._gemm_sched(4096)
    assert all(c[0] not in ops.GEMM1W_BM for c in ops._gemm_configs(4096, 0))


@pytest.mark.parametrize("M,N,K,epi,pick", [
    (1500, 1536, 4096, 0, None), (2048, 1536, 4096, 0, None), (2048, 768, 3072, 2, None), (2900, 768, 3072, 2, None), (1500, 2048, 5632, 0, None),
    (2900, 1536, 4096, 0, 5), (949, 3072, 2048, 0, 5), (2048, 3072, 768, 3, 5), (2900, 2304, 768, 2, 5), (2900, 3072, 2048, 0, 4), (2048, 11264, 2048, 1, 4),
    (4096, 3072, 2048, 0, 3), (4096, 11264, 2048, 1, None), (5500, 3072, 2048, 0, None), (640, 8192, 14336, 0, None), (640, 7168, 6144, 0, None)])
def test_tile_rule_takes_what_measured_fastest(monkeypatch, M, N, K, epi, pick):
    """Tiles of shapes without a measured entry, on both sides of the lines between split-K, the fallback and the three row tiles (None: the
    fallback's own choice)."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "GEMM1W", True)
    monkeypatch.setattr(ops, "_CUS", 256)
    monkeypatch.setattr(ops, "_TILE_RULE", {})
    assert ops._tile_rule(M, N, K, epi) == (ops._gemm_default(M, N, K, epi) if pick is None else (pick, 256, 1))


@pytest.mark.parametrize("M,N,cfg,pick", [
    (257, 28672, 3, 4), (384, 28672, 3, 4), (385, 28672, 3, 3), (512, 28672, 3, 3), (949, 28672, 3, 7), (961, 28672, 3, 3), (1100, 28672, 6, 4),
    (1100, 28672, 3, 4), (1194, 28672, 6, 6), (256, 28672, 3, 3), (4609, 28672, 3, 3), (4095, 10496, 3, 7), (2589, 14336, 3, 6), (2600, 4096, 4, 4),
    (300, 2048, 3, 4)])
def test_fill_rule_takes_what_measured_fastest(monkeypatch, M, N, cfg, pick):
    """Tiles of 256 and 192 rows and column splits by the rounds of this number of rows; other variants and ranges of K are left."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    for name, value in (("GEMM1W", True), ("SPLIT_ON", True), ("_CUS", 256)):
        monkeypatch.setattr(ops, name, value)
    assert ops._fill_rule(M, N, 1, (cfg, 256, 1)) == (pick, 256, 1)
    for kept in ((5, 256, 1), (2, 256, 4), (3, 256, 2), (0, 192, 1), None):
        assert ops._fill_rule(M, N, 1, kept) == kept
    monkeypatch.setattr(ops, "SPLIT_ON", False)
    assert ops._fill_rule(M, N, 1, (3, 256, 1))[0] in (3, 4)


@pytest.mark.parametrize("M,N,K,epi,cfg,pick", [
    (300, 4096, 4096, 0, (2, 256, 4), (5, 256, 4)), (1152, 4096, 4096, 0, (5, 256, 1), (5, 256, 1)), (1536, 4096, 14336, 0, (2, 256, 2), (4, 256, 2)),
    (300, 2048, 5632, 0, (2, 256, 4), (5, 256, 8)), (3072, 2048, 5632, 0, (2, 256, 2), (5, 256, 1)), (512, 2048, 2048, 0, (5, 256, 1), (5, 256, 4)),
    (1024, 2048, 1024, 3, (5, 256, 1), (5, 256, 1)), (4608, 4096, 4096, 0, (3, 256, 1), (3, 256, 1)),
    (256, 4096, 4096, 0, (2, 256, 4), None), (4609, 2048, 5632, 0, (2, 256, 2), None), (300, 2112, 4096, 0, (2, 192, 4), None),
    (300, 4096, 4096, 1, (0, 256, 1), None), (2664, 6144, 4096, 0, (6, 256, 1), None), (300, 256, 128, 0, (0, 256, 1), None), (300, 2048, 2048, 0, None, None)])
def test_split_rule_takes_what_measured_fastest(monkeypatch, M, N, K, epi, cfg, pick):
    """Ranges of K on gemm1w.hip's tiles, on both sides of the line (None: the rule does not take the product, whatever its pick)."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    for name, value in (("GEMM1W", True), ("GEMM_SPLITK", True), ("_CUS", 256), ("_SPLIT_RULE", {})):
        monkeypatch.setattr(ops, name, value)
    assert ops._split_rule(M, N, K, epi, cfg, K) == (pick or cfg)
    got = ops._split_rule(M, N, K, epi, cfg, (1 << 26) // (M + 256) + 1)   # rows too far apart for 32-bit offsets
    assert got == cfg
    for name in ("GEMM1W", "GEMM_SPLITK"):
        monkeypatch.setattr(ops, name, False)
        assert ops._split_rule(M, N, K, epi, cfg, K) == cfg
        monkeypatch.setattr(ops, name, True)


@pytest.mark.parametrize("M,N,K,epi,cfg,pick", [
    (4258, 6144, 192, 0, 3, 3), (4099, 6144, 192, 3, 3, 3), (3754, 10496, 256, 0, 3, 3), (4139, 10496, 512, 0, 3, 3), (3821, 11264, 768, 3, 3, 3),
    (3733, 11264, 1024, 3, 3, 3), (1148, 28672, 1024, 0, 3, 4), (2413, 16384, 4096, 1, 3, 6), (2589, 14336, 4096, 1, 3, 6)])
def test_fill_rule_weighs_a_second_launch(monkeypatch, M, N, K, epi, cfg, pick):
    """What a column split saves grows with K, what its second launch costs does not: a short K stays in one launch."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    for name, value in (("GEMM1W", True), ("SPLIT_ON", True), ("_CUS", 256)):
        monkeypatch.setattr(ops, name, value)
    assert ops._fill_rule(M, N, epi, (cfg, 256, 1), K) == (pick, 256, 1)


@pytest.mark.parametrize("M,N,K,epi,fastest", [
    (949, 28672, 256, 1, (3, 256, 1)), (1100, 28672, 256, 1, (6, 256, 1)), (512, 512, 4096, 0, (2, 256, 4)), (300, 512, 4096, 3, (0, 256, 2)),
    (512, 512, 4096, 2, (5, 256, 8)), (768, 768, 2048, 0, (4, 256, 1)), (512, 512, 1024, 0, None)])
def test_measured_products_run_as_measured(monkeypatch, M, N, K, epi, fastest):
    """``tune_gemm`` on a clock that lets one candidate win: that one runs at the measured rows and at all that make as many tiles, and the
    rules, which know estimates only, are not asked there."""
    from types import SimpleNamespace

    from llm_kubernetes_minikube_sharp4dev_amd import ops

    ran = []

    class Event:
        def __init__(self, **kw):
            self.record = self.synchronize = lambda: None

        def elapsed_time(self, other):
            return 1.0 if ran[-1] == fastest else 2.0 + 0.001 * len(set(ran[:ran.index(ran[-1])]))

    lib = SimpleNamespace(gemm_supported=lambda M, N, K, epi, bn, ks, v: True, gemm=lambda x, w, b, epi, bn, out, v, ks: ran.append((v, bn, ks)))
    for name, value in (("GEMM1W", True), ("GEMM_SPLITK", True), ("SPLIT_ON", True), ("_CUS", 256), ("lib", lambda: lib), ("_GEMM_TABLE", {}),
                        ("_GEMM_MEASURED", {}), ("_gemm_splits", lambda M, N, K, epi, bn: fastest[2] if fastest and fastest[0] < 3 else 1)):
        monkeypatch.setattr(ops, name, value, raising=False)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    ops.tune_gemm([(torch.zeros(N, K, dtype=torch.bfloat16), epi)], 0, iters=1, cold_bytes=0, ms=[M])

    def runs(m):
        cfg = ops._cfg_of(m, N, K, epi)
        return ops._split_rule(m, N, K, epi, cfg, K)

    pick = fastest or ran[0]   # (None: the first of the candidates)
    assert pick in ran and runs(M) == pick
    tiles = lambda m: [-(-m // bm) for bm in (128, 192, 256)]  # noqa: E731
    for m in range(max(257, M - 256), M + 256):
        if tiles(m) == tiles(M):
            assert runs(m) == pick
    if fastest and fastest[0] >= 3 and fastest[2] > 1:   # unsplit where a split cannot run: fused QKV, rows further apart
        assert ops._cfg_of(M, N, K, epi)[2] == 1
        assert ops._split_rule(M, N, K, epi, ops._cfg_of(M, N, K, epi), 1 << 20) == ops._cfg_of(M, N, K, epi)


@pytest.mark.parametrize("S,heads,P,N,max_len,rows,piped", [
    (4, 32, 64, 64, 8, 32, 1), (16, 32, 64, 64, 8, 128, 0), (64, 32, 64, 64, 64, 4096, 0), (256, 8, 64, 64, 16, 4096, 0), (64, 16, 128, 64, 128, 8192, 0),
    (8, 32, 64, 64, 512, 4096, 1), (4, 128, 64, 64, 1024, 4096, 1), (1, 128, 64, 64, 8, 8, 1), (65, 32, 64, 64, 8, 72, 0), (65, 32, 64, 64, 512, 576, 1),
    (65, 128, 64, 64, 512, 576, 0), (257, 24, 64, 40, 8, 264, 0), (16, 16, 32, 48, 64, 1024, 1), (64, 80, 64, 72, 8, 512, 1), (256, 64, 64, 128, 8, 2048, 1)])
def test_state_space_pipeline_takes_what_it_is_faster_at(S, heads, P, N, max_len, rows, piped):
    """33 - 64 state columns: many short portions stay with the kernel of two workgroups to a CU."""
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    assert _ext.lib().ssm_piped(S, heads, P, N, max_len, rows, 256) == piped


@pytest.mark.parametrize("ntiles,groups,workgroups", [(1, 1, 16), (796, 12, 9600), ((1 << 20) - 16, 16, (1 << 24) - 256),
                                                      ((1 << 20) - 15, 16, 0), (1 << 20, 16, 0), (8 << 20, 2, 0)])
def test_encoder_attention_grid_stays_in_a_launch(ntiles, groups, workgroups):
    """One dimension of a launch holds fewer than 2^32 threads: past that the attention over many short texts keeps its two-dimensional grid."""
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    assert _ext.lib().prefill_pairs(ntiles, groups, 256) == workgroups


@pytest.mark.parametrize("texts,rows,heads,D,order", [
    (4096, 10, 12, 64, 0), (2500, 10, 12, 32, 0), (260, 96, 12, 64, 0), (384, 65, 16, 64, 0), (500, 128, 12, 64, 1), (260, 96, 12, 32, 1), (260, 96, 16, 128, 1),
    (496, 129, 12, 64, 1), (69, 129, 16, 128, 1), (128, 450, 12, 64, 1), (64, 1024, 12, 64, 1), (43, 1500, 16, 64, 1), (32, 2048, 12, 64, 0),
    (8, 8192, 12, 64, 0), (16, 4096, 16, 128, 0)])
def test_encoder_attention_order_by_its_texts(texts, rows, heads, D, order):
    """Pairs of tiles with all of their heads where that measured faster: not for many texts of a few rows, nor for long ones."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    tiles = len(ops.prefill_tiles([rows] * texts, [rows] * texts, 1, False, D)[0])
    assert _ext.lib().prefill_order(tiles, texts, rows * texts, heads, D) == order


def test_reference_switch_follows_the_environment(monkeypatch):
    """Set, changed and taken away while the process runs, and in a mapping put in the environment's place."""
    import os

    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    monkeypatch.delenv("LK_FORCE_REFERENCE", raising=False)
    assert not _ext.force_reference()
    for value, on in (("1", True), ("0", False), ("", False), ("false", False), ("yes", True)):
        monkeypatch.setenv("LK_FORCE_REFERENCE", value)
        assert _ext.force_reference() == on
    monkeypatch.delenv("LK_FORCE_REFERENCE")
    assert not _ext.force_reference()
    monkeypatch.setattr(os, "environ", {"LK_FORCE_REFERENCE": "1"})
    assert _ext.force_reference()


def test_reference_switch_asks_no_library(monkeypatch):
    """What chooses a kernel asks the library only where kernels run: with the switch on it need not be there."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops
    from llm_kubernetes_minikube_sharp4dev_amd.ops import window

    def absent():
        raise RuntimeError("no library")

    monkeypatch.setattr(window, "lib", absent)
    monkeypatch.setenv("LK_FORCE_REFERENCE", "1")
    assert not ops.moe_skips_rows(4, 2, 8, 256, 128)


@pytest.mark.parametrize("T,W,N2,E,ff,top,beside", [(1, 2048, 2048, 16, 2816, 2, 1), (64, 2048, 2048, 16, 2816, 2, 1), (40, 4096, 4096, 16, 1536, 2, 0), (16, 4096, 4096, 16, 1536, 2, 1),
                                                    (40, 7168, 7168, 16, 2048, 2, 0), (80, 2048, 4096, 16, 2816, 2, 0), (80, 1024, 1024, 16, 1408, 2, 1), (96, 2048, 256, 16, 2816, 2, 1),
                                                    (97, 1024, 1024, 16, 1408, 2, 0), (0, 1024, 1024, 16, 1408, 2, 0), (8, 1000, 1024, 16, 1408, 2, 0), (8, 1024, 1000, 16, 1408, 2, 0)])
def test_gate_beside_the_experts_by_its_bytes(T, W, N2, E, ff, top, beside):
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    assert _ext.lib().moe_beside_ok(T, top, E, 2 * ff, W, N2) == bool(beside)


@pytest.mark.parametrize("M,N,I,K,bn", [(64, 3072, 5632, 2048, 64), (64, 10496, 5632, 2048, 128), (4, 3072, 5632, 2048, 64), (64, 4096, 8192, 4096, 128), (16, 4096, 8192, 4096, 0),
                                       (1, 384, 512, 8192, 0), (64, 384, 512, 8192, 0), (128, 384, 512, 8192, 0), (128, 2048, 2048, 2048, 0), (1, 2048, 2048, 2048, 0),
                                       (48, 2048, 2048, 2048, 64), (128, 128, 128, 2560, 0), (64, 3072, 512, 12288, 0), (129, 3072, 5632, 2048, 0), (64, 3072, 5632, 2000, 0),
                                       (0, 3072, 5632, 2048, 0), (4, 0, 5632, 2048, 0)])
def test_products_beside_by_their_chain(monkeypatch, M, N, I, K, bn):
    """Long K on few workgroups stays apart; where start-up measured the products alone, that is what the chain is held against."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    if not ops.available():
        pytest.skip("the kernel library is not built")
    monkeypatch.setattr(ops, "_DECODE_US", {})
    monkeypatch.setattr(ops, "_CUS", 256)
    assert ops._beside_rule(M, N, I, K) == bn
    if bn and M > ops.LM_HEAD_SKINNY_MAX_M:
        b = ops._decode_bucket(M)
        ops._DECODE_US.update({(b, N, K, False): 0.5, (b, 2 * I, K, True): 0.5})
        assert ops._beside_rule(M, N, I, K) == 0


@pytest.mark.parametrize("M,N,K,swiglu,plan", [(64, 10496, 2048, False, (64, 1)), (256, 11264, 2048, True, (64, 1)), (128, 8960, 4096, False, (64, 1)), (129, 8960, 4096, False, (128, 2)),
                                              (16, 9472, 7168, False, (128, 2)), (16, 9472, 7168, True, (128, 2)), (192, 5120, 5120, False, (128, 4)), (8, 2560, 14336, False, (128, 8)),
                                              (120, 4096, 14336, False, (128, 8)), (120, 28672, 4096, True, (128, 1)), (120, 6144, 4096, False, (96, 4))])
def test_streaming_plans_by_k_and_rows(M, N, K, swiglu, plan):
    """Whole K on 64-column tiles only where it is short; otherwise as many parts of 128 columns."""
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    assert tuple(_ext.lib().ws_plan(M, N, K, swiglu)) == plan


@pytest.mark.parametrize("M,N,K,swiglu,few", [(56, 1280, 6400, True, True), (64, 1152, 5888, False, True), (56, 768, 7168, True, True), (64, 512, 5120, True, True),
                                             (40, 3456, 6656, False, False), (80, 14080, 4352, True, False), (160, 6144, 6400, True, False), (120, 28672, 4096, True, False)])
def test_narrow_products_of_long_k_take_the_few_row_kernel(monkeypatch, M, N, K, swiglu, few):
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    if not ops.available():
        pytest.skip("the kernel library is not built")
    monkeypatch.setattr(ops, "_ROWS_TABLE", {})
    monkeypatch.setattr(ops, "_ROWS_RULE", {})
    assert (ops._rows_choice(M, N, K, int(swiglu)) is not None) == few


@pytest.mark.parametrize("lens,Hq,Hkv,two", [([159], 32, 8, 0), ([160], 32, 8, 1), ([100] * 8, 32, 8, 0), ([1024], 32, 8, 1), ([2048], 32, 8, 1), ([2049], 32, 8, 0),
                                             ([400] * 3, 32, 8, 0), ([600] * 2, 32, 8, 1), ([500] * 4, 32, 8, 0), ([1500], 32, 32, 1)])
def test_prompt_attention_splits_keys_where_few_chains_are_long(lens, Hq, Hkv, two):
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    G = Hq // Hkv
    rows = 32 if G >= 4 else 32 * (4 // G)
    groups = sum(-(-n // rows) for n in lens) * Hq // min(G, 4)
    assert _ext.lib().prefill_split_keys(groups, sum(lens), len(lens), 256) == two


@pytest.mark.parametrize("S,cblocks,max_len,rows", [(1, 3, 60, 4), (1, 3, 400, 4), (1, 3, 401, 8), (1, 3, 1600, 8), (1, 3, 1601, 16), (4, 3, 1024, 16), (300, 1, 1, 4),
                                                    (600, 1, 2, 8), (601, 1, 8, 16)])
def test_convolution_tiles_count_the_devices_cus(S, cblocks, max_len, rows):
    """The convolution's tiles fill the CUs of the device: a partition of 32 picks what the whole chip does at eight times the workgroups."""
    from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext

    if not _ext.available():
        pytest.skip("the kernel library is not built")
    pick = _ext.lib().conv_rows
    assert pick(S, cblocks, max_len, 256) == rows
    assert pick(S, 8 * cblocks, max_len, 2048) == rows
    assert pick(S, cblocks, max_len, 32) >= rows and pick(S, cblocks, max_len, 32) == pick(S, 8 * cblocks, max_len, 256)


@pytest.mark.parametrize("rule", ["_TILE_RULE", "_FILL_RULE", "_SPLIT_RULE"])
def test_rules_of_tiles_survive_a_full_table(monkeypatch, rule):
    """A rule's table of picks is shared by threads and emptied when it is full: a pick does not need its entry to be there still."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    class Emptied(dict):   # another thread empties the table right behind every entry
        def __setitem__(self, key, value):
            super().__setitem__(key, value)
            self.clear()

    for name, value in (("GEMM1W", True), ("GEMM_SPLITK", True), ("SPLIT_ON", True), ("_CUS", 256)):
        monkeypatch.setattr(ops, name, value)
    picks = {"_TILE_RULE": lambda M: ops._tile_rule(M, 2048, 5632, 0), "_FILL_RULE": lambda M: ops._fill_rule(M, 28672, 1, (3, 256, 1)),
             "_SPLIT_RULE": lambda M: ops._split_rule(M, 4096, 4096, 0, (3, 256, 1), 4096)}[rule]
    monkeypatch.setattr(ops, rule, {})
    want = [picks(M) for M in range(300, 1500, 100)]
    assert [picks(M) for M in range(300, 1500, 100)] == want   # (from the table)
    monkeypatch.setattr(ops, rule, Emptied())
    assert [picks(M) for M in range(300, 1500, 100)] == want


@pytest.mark.parametrize("M,N,K,epi,pick", [
    (58963, 2304, 768, 2, 3), (35218, 1536, 768, 2, 3), (44104, 768, 768, 2, 4), (17401, 768, 768, 2, 3), (8925, 2304, 1536, 0, 4), (5500, 3072, 2048, 0, 4),
    (62947, 6144, 2048, 0, 3), (14488, 1536, 4096, 0, 4), (4609, 768, 3072, 2, None), (4608, 2304, 768, 2, None), (9000, 192, 768, 0, None),
    (200000, 6144, 2048, 0, None)])
def test_rounds_rule_takes_what_measured_fastest(monkeypatch, M, N, K, epi, pick):
    """Row tiles past 4,608 rows by their rounds over the CUs; split-K, fewer rows and widths without 256-column tiles keep their rules."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "GEMM1W", True)
    monkeypatch.setattr(ops, "_CUS", 256)
    assert ops._rounds_rule(M, N, K, epi) == (None if pick is None else (pick, 256, 1))
    monkeypatch.setattr(ops, "GEMM1W", False)
    assert ops._rounds_rule(M, N, K, epi) is None


def test_few_row_rule_counts_the_devices_cus(monkeypatch):
    """The few-row kernel's rounds are of the device's CUs: what it wins on a whole chip (128 workgroups in half a round) it loses on a
    partition of 32 CUs, where they are four rounds."""
    from types import SimpleNamespace

    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "lib", lambda: SimpleNamespace(rows_supported=lambda *a: True))
    for cus, pick in ((256, False), (32, None)):
        monkeypatch.setattr(ops, "_CUS", cus)
        monkeypatch.setattr(ops, "_ROWS_RULE", {})
        assert ops._rows_rule(64, 2048, 2048, 0) is pick


@pytest.mark.parametrize("M,N,K,epi,rows", [(512, 48, 8192, 0, False), (128, 96, 8192, 2, False), (400, 2064, 1024, 0, False),
                                            (400, 2064, 1024, 3, False), (512, 96, 8192, 1, False), (64, 2064, 1024, 0, True),
                                            (64, 400, 1024, 0, True), (192, 48, 256, 2, True), (512, 48, 256, 3, True)])
def test_few_row_rule_where_no_tile_takes_the_width(monkeypatch, M, N, K, epi, rows):
    """Widths that go to the vendor's kernels otherwise: those are the other side of the comparison, not the tiles."""
    from types import SimpleNamespace

    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "lib", lambda: SimpleNamespace(rows_supported=lambda *a: True))
    monkeypatch.setattr(ops, "_CUS", 256)
    monkeypatch.setattr(ops, "_ROWS_RULE", {})
    assert (ops._rows_rule(M, N, K, epi) is not None) == rows


def test_static_gemm_table_is_well_formed(monkeypatch):
    """The shipped measured dispatch table (benchmarks/gemm_table.py on an MI355X): every entry a
    kernel / tile / split the dispatch knows, looked up by _cfg_of before the fallback policy,
    and ignored under LK_GEMM1W=0 where it names a gemm1w variant."""
    import json
    import os

    from llm_kubernetes_minikube_sharp4dev_amd import ops

    if not os.path.exists(ops.GEMM_TABLE_FILE):
        pytest.skip("no measured table shipped")
    doc = json.load(open(ops.GEMM_TABLE_FILE))
    assert doc["arch"] == "gfx950" and doc["entries"]
    for mb, n, k, epi, v, bn, ks in doc["entries"]:
        assert v in (0, 1, 2, 3, 4, 5, 6, 7) and bn in (192, 256) and 1 <= ks <= 4 and epi in (0, 1, 2, 3, 4)
        assert bn == 256 or v not in ops.GEMM1W_BM
        assert ks == 1 or v not in ops.GEMM1W_BM
        assert k % 64 == 0 and n % bn == 0
    mb, n, k, epi, v, bn, ks = doc["entries"][0]
    monkeypatch.setattr(ops, "_GEMM_TABLE", {})
    monkeypatch.setattr(ops, "GEMM1W", True)
    assert ops._cfg_of(mb * 256, n, k, epi) == (v, bn, ks)
    monkeypatch.setattr(ops, "GEMM1W", False)
    assert ops._cfg_of(mb * 256, n, k, epi)[0] not in ops.GEMM1W_BM


def test_lib_path_ab_knob_loads_the_named_build():
    """LK_LIB_PATH (same-box A/B of two builds of the kernel library) loads the extension from
    the given file instead of the in-tree one."""
    import glob
    import os
    import subprocess
    import sys

    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    so = glob.glob(os.path.join(root, "llm_kubernetes_minikube_sharp4dev_amd", "_C.*.so"))
    if not so:
        pytest.skip("kernel library not built")
    code = ("from llm_kubernetes_minikube_sharp4dev_amd.ops import _ext; m = _ext.try_lib(); "
            "print(m.__file__ if m is not None else 'ERR ' + repr(_ext._err))")
    env = {**os.environ, "LK_LIB_PATH": so[0]}
    out = subprocess.run([sys.executable, "-c", code], cwd=root, env=env, capture_output=True, text=True,
                         timeout=300).stdout.strip().splitlines()[-1]
    assert out == so[0], out


def _first_step_logits(m, prompts):
    eng = _engine(m)
    for p in prompts:
        eng.add_request(p, SamplingParams.greedy(1))
    eng._drain_inbox()
    rows, lg = eng.runner.forward_logits(eng.scheduler.schedule().items)
    return lg


def test_folded_norms_and_fused_chain_match_hf(monkeypatch):
    """fold_norms (norm weights into qkv / gate_up, q / k rows to adjacent RoPE pairs) is the same
    model, and the fused prefill chain (_forward_chain: scale-in-epilogue GEMMs, RESID partial
    sums of squares, RoPE + KV write in the QKV epilogue) computes the same logits and greedy
    tokens as HF -- fp32 reference ops on the CPU (the GPU test runs the HIP epilogues)."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    hcfg = transformers.LlamaConfig(vocab_size=512, hidden_size=256, intermediate_size=512, num_hidden_layers=2,
                                    num_attention_heads=4, num_key_value_heads=2, max_position_embeddings=1024,
                                    rope_theta=10000.0, rms_norm_eps=1e-5, tie_word_embeddings=False)
    torch.manual_seed(0)
    hf = transformers.LlamaForCausalLM(hcfg).eval()
    cfg = DecoderConfig("t", "llama", 2, 256, 4, 2, 64, 512, 512, max_position=1024, rope_theta=10000.0)
    sd = hf.state_dict()
    for k in list(sd):  # non-trivial norm weights, so the fold is exercised
        if k.endswith("norm.weight"):
            sd[k] = 1 + 0.1 * torch.randn_like(sd[k])
    hf.load_state_dict(sd)
    prompts = [[5, 17, 99, 3, 250, 7, 7, 1, 400, 33, 21, 8, 2, 9, 11, 60, 61, 62, 63], list(range(30, 70))]
    m = build_decoder(cfg, dtype=torch.float32)
    m.load_hf_state_dict(sd)
    assert not m.folded  # CPU: checkpoint layout
    with torch.no_grad():
        want = torch.stack([hf(torch.tensor([p])).logits[0, -1] for p in prompts])
    plain = _first_step_logits(m, prompts)
    m.fold_norms()
    assert m.folded and not m.rope_neox and torch.all(m.layers[0].input_norm == 1)
    folded = _first_step_logits(m, prompts)
    calls = []
    real = m._forward_chain

    def spy(*a, **k):
        calls.append(1)
        return real(*a, **k)

    monkeypatch.setattr(ops, "prefill_chain_ok", lambda *a: True)
    monkeypatch.setattr(m, "_forward_chain", spy)
    chained = _first_step_logits(m, prompts)
    assert calls, "the fused chain did not run"
    for got in (plain, folded, chained):
        assert torch.allclose(got, want, atol=2e-4, rtol=2e-4), (got - want).abs().max()
    seqs = _engine(m).generate(prompts, SamplingParams.greedy(8))
    with torch.no_grad():
        for p, s in zip(prompts, seqs):
            ref = hf.generate(torch.tensor([p]), max_new_tokens=8, do_sample=False)[0, len(p):].tolist()
            assert s.output_ids == ref


def test_fused_chain_reference_ops():
    """The CPU oracles of the fused epilogues: RESID partial sums of squares per 256 columns and
    the consumer's row scale reproduce RMSNorm; the QKV oracle is GEMM -> interleaved rope_kv_."""
    from llm_kubernetes_minikube_sharp4dev_amd.ops import reference as R

    torch.manual_seed(1)
    M, H = 37, 512
    r = torch.randn(M, H)
    x = torch.randn(M, 256)
    w = torch.randn(H, 256) * 0.05
    ss = torch.zeros(H // 256, 64)
    r2 = r.clone()
    R.linear_resid(x, w, r2, ss)
    assert torch.allclose(r2, r + x @ w.t(), atol=1e-5)
    s = R.row_scale(ss, H, 1e-5)[:M]
    assert torch.allclose(s, torch.rsqrt(r2.pow(2).mean(-1) + 1e-5), rtol=1e-5)
    wg = torch.randn(64, H) * 0.05
    y = R.gemm_scaled(r2, wg, ss, H, 1e-5)
    normed = r2 * torch.rsqrt(r2.pow(2).mean(-1, keepdim=True) + 1e-5)
    assert torch.allclose(y, normed @ wg.t(), atol=1e-4)


def test_gemm1w_column_split_plan():
    """Variants 6 / 7 split the column tiles: whole waves of 256-row tiles first (mirrors
    lk_gemm1w_split_cols in csrc/gemm1w.hip)."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    assert ops.gemm1w_split_cols(4096, 6144, 0) == 16  # 16 x 24 = 1.5 waves -> 16 x 16, then 8 columns
    assert ops._split_applies(4096, 6144, 0)
    assert not ops._split_applies(4096, 4096, 0)  # 16 x 16: exactly one wave
    assert not ops._split_applies(8192, 6144, 0)  # 32 x 24: three waves
    assert not ops._split_applies(1024, 4096, 0)  # under a wave: nothing to split
    assert ops.gemm1w_split_cols(600, 28672, 1) == 85  # SwiGLU: 3 x 112 tiles


@pytest.mark.parametrize("M,N,K,epi,form", [
    (768, 3072, 768, 0, None), (1000, 3072, 768, 3, None), (400, 6144, 768, 1, None), (128, 16384, 1024, 0, None), (192, 16384, 1024, 0, None),
    (96, 32768, 1024, 1, None), (640, 6272, 1024, 1, None), (65, 8192, 8192, 0, None), (400, 1152, 384, 0, True), (400, 576, 1152, 0, True),
    (192, 4096, 5632, 1, 2), (64, 10496, 2048, 0, 2), (33, 12288, 4096, 1, 2), (64, 2048, 2048, 0, False)])
def test_few_row_rule_on_measured_shapes(monkeypatch, M, N, K, epi, form):
    """Rounds of workgroups, weights read again by further row tiles, and what the weight-streaming and tiled kernels take: the measured faster side."""
    from types import SimpleNamespace

    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "lib", lambda: SimpleNamespace(rows_supported=lambda *a: True))
    monkeypatch.setattr(ops, "_CUS", 256)
    monkeypatch.setattr(ops, "_ROWS_RULE", {})
    assert ops._rows_rule(M, N, K, epi) == form


@pytest.mark.parametrize("M,N,K1,K2,pay", [
    (1, 2048, 4096, 5632, True), (64, 2048, 4096, 5632, True), (64, 8192, 512, 960, True), (1, 4096, 4096, 8192, False), (4, 4096, 4096, 8192, True),
    (64, 5120, 5120, 5120, True), (64, 8192, 8192, 28672, False), (64, 6144, 6144, 16384, False), (64, 8192, 2048, 8192, False),
    (2, 8192, 8192, 8192, False), (64, 8192, 8192, 8192, True)])
def test_sums_of_two_products_where_they_pay(monkeypatch, M, N, K1, K2, pay):
    """Ranges of K of different length leave CUs waiting: measured on both sides."""
    from llm_kubernetes_minikube_sharp4dev_amd import ops

    monkeypatch.setattr(ops, "_CUS", 256)
    assert ops.sums_pay(M, N, K1, K2) == pay


def _query_replay(monkeypatch, current, priority, last=None):
    """EmbeddingEngine._replay_query on a device that is only written down: what it did, in order, each with the device and stream it was
    done on (``last``: the stream of the replay before, or "own", the engine's)."""
    import threading
    from types import SimpleNamespace

    import numpy as np

    from llm_kubernetes_minikube_sharp4dev_amd import ops
    from llm_kubernetes_minikube_sharp4dev_amd.engine.embed_engine import EmbeddingEngine

    done, device, on = [], [0], [current]

    class Within:
        def __init__(self, cell, value):
            self.cell, self.value = cell, value

        def __enter__(self):
            self.before, self.cell[0] = self.cell[0], self.value

        def __exit__(self, *a):
            self.cell[0] = self.before

    def did(what):
        return lambda *a: done.append((what, device[0], on[0]))

    monkeypatch.setattr(torch.cuda, "device", lambda d: Within(device, torch.device(d).index))
    monkeypatch.setattr(torch.cuda, "stream", lambda s: Within(on, s))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda d=None: current)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(ops, "set_ids", did("ids"))
    eng = object.__new__(EmbeddingEngine)
    eng.device = torch.device("cuda", 1)
    own = SimpleNamespace(priority=priority, wait_stream=did("wait"), wait_event=did("event"))
    eng._gstream, eng._gpriority, eng._glock, eng._glast = own, priority, threading.Lock(), own if last == "own" else last
    eng._gdone = SimpleNamespace(record=did("done"))
    eng._qgraphs = {(3, torch.float32): (SimpleNamespace(replay=did("replay")), None, None)}
    dst = SimpleNamespace(dtype=torch.float32, copy_=did("out"), record_stream=did("kept"))
    assert eng._replay_query(np.array([1, 2, 3]), dst)
    assert device == [0] and on == [current]
    return done, own


def test_query_replay_switches_to_its_device(monkeypatch):
    """A caller whose current device is another one: ids, graph and result are enqueued on the engine's."""
    from types import SimpleNamespace

    cur = SimpleNamespace(priority=0, wait_stream=lambda s: None)
    done, _ = _query_replay(monkeypatch, cur, 0)
    assert done == [(w, 1, cur) for w in ("ids", "replay", "out", "done")]


@pytest.mark.parametrize("current,priority,mine", [(0, 0, True), (-1, 0, True), (-1, -1, True), (0, -1, False)])
def test_query_replay_stream(monkeypatch, current, priority, mine):
    """Replays run on the caller's stream, or on the engine's where that has a priority that the caller's has not; behind a replay on another stream."""
    from types import SimpleNamespace

    joined, events = [], []
    cur = SimpleNamespace(priority=current, wait_stream=joined.append, wait_event=events.append)
    for last in (None, "own", cur, SimpleNamespace()):
        done, own = _query_replay(monkeypatch, cur, priority, last)
        on = cur if mine else own
        other = last is not None and (own if last == "own" else last) is not on
        work = [(w, 1, on) for w in ("ids", "replay", "out", "done")]
        if mine:
            assert done == work and len(events) == other and not joined
        else:   # (waits for the caller's work before, and the caller for it behind; the result is kept for this stream)
            assert done == [("wait", 1, cur)] + [("event", 1, own)] * other + work + [("kept", 0, cur)] and joined == [own]
        joined.clear(), events.clear()
