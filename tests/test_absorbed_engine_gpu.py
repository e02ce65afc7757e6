"""The Fusasun decoder on the cached latent (``LatentAttnSpec.absorb``) through the engine, against the float64 oracle: whole prompts,
portions, single tokens, captured decode steps with padding rows, requests that share steps, pages and slots that are used again, and the
cache's size."""
import pytest
import torch

from llm_kubernetes_minikube_sharp4dev_amd import ops
from llm_kubernetes_minikube_sharp4dev_amd.engine.sampling import SamplingParams
import fusasun_oracle as O
import test_fusasun_engine as E

pytestmark = pytest.mark.gpu
BF = torch.bfloat16
# a window shorter than a prompt and no page's size; a convolution, a windowed softmax layer and experts beside the latent layers
E.CONFIGS["absorbed"] = E.config([E.moe(E.lat(16, 128, 64, 128, 96, 512, 0.07, 37, 1000.0, (4.0, 64, 4.0, 1.0)), 64, 4, 2),
                                  E.moe(E.att(4, 2, 32, 32, 0.2, 20, None, 16, 50.0), 0),
                                  E.moe(E.lat(16, 64, 32, 64, 64, 128, 0.1, 24, 500.0), 0)], 64)


@pytest.fixture(scope="module")
def model():
    m, sd = E.model_and_weights("absorbed", "cuda", BF)
    specs = [L.mix.spec for L in m.layers if L.type == "latent_attention"]
    assert len(specs) == 2 and all(s.absorbed for s in specs)      # the rule takes these sizes: what follows runs on the cached latent
    return m, sd


def test_portions_and_single_tokens(model):
    E.test_prefill_equals_token_by_token_and_portions("absorbed", "cuda", BF)
    E.test_whole_prompt_streams_and_logits("absorbed", "cuda", BF)


def test_mixed_steps(model):
    """Portions of some requests beside single tokens of others (two and three decode rows: captured steps pad them to four); every request
    as alone, and the pages and slots come back."""
    m, sd = model
    V = m.cfg.vocab_size
    T = {"a": E.toks(60, V, 10), "b": E.toks(24, V, 11), "c": E.toks(12, V, 12), "d": E.toks(41, V, 13)}
    plan = [[("a", 17)], [("a", 15), ("b", 20), ("c", 1)], [("a", 1), ("b", 1), ("c", 1)], [("a", 1), ("b", 1), ("c", 1)], [("a", 1), ("b", 1), ("c", 2), ("d", 31)],
            [("a", 1), ("b", 1), ("d", 1)], [("a", 24), ("c", 7), ("d", 1)], [("d", 8)]]
    eng = E.engine(m, tokens=160, seqs=4)
    at, got = {k: 0 for k in T}, {k: [] for k in T}
    for step in plan:
        entries, end = [], []
        for k, n in step:
            entries.append((k, T[k][at[k]:at[k] + n], list(range(n))))
            at[k] += n
            if at[k] == len(T[k]):
                end.append(k)
        lg, r = eng.replay_step(entries, end), 0
        for k, n in step:
            got[k].append(lg[r:r + n])
            r += n
    assert at == {k: len(v) for k, v in T.items()}
    assert eng.allocator.num_free == eng.runner.num_blocks and eng.state_pool.num_free == 4
    for k in T:
        want = O.forward(E.CONFIGS["absorbed"], sd, T[k])
        ok, err = E.close(torch.cat(got[k]), want, BF)
        assert ok, (k, err)
        alone = E.replay(eng, k + "-alone", T[k], [n for step in plan for kk, n in step if kk == k])
        assert float((alone.double() - torch.cat(got[k]).double()).abs().max() / want.abs().max()) < 6e-2


def test_pages_and_slots_are_used_again(model):
    m, sd = model
    a, b = E.toks(64, m.cfg.vocab_size, 20), E.toks(50, m.cfg.vocab_size, 21)
    eng = E.engine(m, tokens=64, seqs=1)
    first, other, again = E.replay(eng, "a", a, [30, 5]), E.replay(eng, "b", b, [3, 40]), E.replay(eng, "a2", a, [30, 5])
    assert torch.equal(first, again)
    assert E.close(first, O.forward(E.CONFIGS["absorbed"], sd, a), BF)[0] and E.close(other, O.forward(E.CONFIGS["absorbed"], sd, b), BF)[0]


def test_generation_and_cache_size(model):
    """Greedy decoding of three prompts by the scheduler; a block's bytes are those of its latent rows and of the softmax layer."""
    m, sd = model
    V = m.cfg.vocab_size
    eng = E.LLMEngine(m, None, block_size=16, max_model_len=256, max_num_seqs=3, num_blocks=16, eos_ids=set(), max_num_batched_tokens=24)
    prompts = [E.toks(50, V, 40), E.toks(7, V, 41), E.toks(1, V, 42)]
    for seq, p in zip(eng.generate(prompts, SamplingParams.greedy(12)), prompts):
        lg = O.forward(E.CONFIGS["absorbed"], sd, p + seq.output_ids)
        for i, t in enumerate(seq.output_ids):
            row = lg[len(p) - 1 + i]
            assert float(row.max() - row[t]) <= 0.05 * float(row.abs().max())   # the oracle's argmax, or a tie within bf16 logits
    rows = sum(sum(ops.latent_row(r, d)) for r, d in ((512, 64), (128, 32)))
    assert m.cache_block_bytes(16) == 16 * 2 * (rows + 2 * (32 + 32))
    assert sum(c.numel() * c.element_size() for cs in eng.runner.kv_caches for c in cs if c.shape[0] == 16) == 16 * m.cache_block_bytes(16)
