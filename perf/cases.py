"""What a user of this framework has it do, as cases to be timed and checked.

The stack answers questions over a corpus: an encoder embeds queries and documents, a cosine search
ranks the corpus, and a decoder behind a continuous-batching engine reads prompts and writes tokens.
The cases take these in turn, each through the call that a serving process makes, from one query
alone on the device to full batches; two further decoder designs stand for those the engine serves
beside Llama (a hybrid of sigmoid attention and state-space layers, and windowed / latent attention
with routed experts).  Everything is bf16 as served; weights are random under the checkpoints' names
and shapes.

``exact`` is each result in float64 from the same weights and inputs, in plain torch.
"""
import math
import random

import numpy as np
import torch

from llm_kubernetes_minikube_sharp4dev_amd.engine.embed_engine import EmbeddingEngine
from llm_kubernetes_minikube_sharp4dev_amd.engine.llm_engine import LLMEngine
from llm_kubernetes_minikube_sharp4dev_amd.engine.sampling import SamplingParams
from llm_kubernetes_minikube_sharp4dev_amd.engine.sequence import Sequence
from llm_kubernetes_minikube_sharp4dev_amd.models.bert import EncoderModel
from llm_kubernetes_minikube_sharp4dev_amd.models.configs import (FusasunConfig, LebepelConfig, decoder_config, encoder_config,
                                                                  fusasun_layers, lebepel_layers)
from llm_kubernetes_minikube_sharp4dev_amd.models.fusasun import FusasunModel
from llm_kubernetes_minikube_sharp4dev_amd.models.lebepel import LebepelModel
from llm_kubernetes_minikube_sharp4dev_amd.models.llama import LlamaModel
from llm_kubernetes_minikube_sharp4dev_amd.rag.index import RagChunk, RagIndex

DEV = "cuda"
BF, F32, F64 = torch.bfloat16, torch.float32, torch.float64
VOCAB = 32768            # the built-in tokenizer's
BLOCK = 16               # cache block of the engine
STEPS = 4                # decode steps of one pass


def listed():
    return [
        # one question's embedding: the first thing a request waits for
        {"name": "embed_query", "kind": "embed", "n": 1, "lo": 19, "hi": 19},
        # documents of an index build, ragged chunks of the corpus's average length
        {"name": "embed_chunks", "kind": "embed", "n": 1024, "lo": 20, "hi": 224},
        # one question against a knowledge base just large enough for the device search
        {"name": "search_one", "kind": "search", "rows": 20011, "n": 1, "k": 5},
        # an admission's questions against the 100k-document corpus (485,620 chunks)
        {"name": "search_corpus", "kind": "search", "rows": 485620, "n": 16, "k": 6},
        # a single request's prompt: the time to its first token
        {"name": "llama_prompt", "kind": "llama", "phase": "prefill", "n": 1, "lo": 949, "hi": 949},
        # a full engine step of several prompts under load
        {"name": "llama_prompts", "kind": "llama", "phase": "prefill", "n": 5, "lo": 640, "hi": 998},
        # one session writing tokens alone
        {"name": "llama_decode_one", "kind": "llama", "phase": "decode", "n": 1, "lo": 961, "hi": 961},
        # the continuous batch of the serving benchmark
        {"name": "llama_decode_batch", "kind": "llama", "phase": "decode", "n": 120, "lo": 700, "hi": 1200},
        # the state-space hybrid: prompts, and a batch of sessions
        {"name": "lebepel_prompts", "kind": "lebepel", "phase": "prefill", "n": 4, "lo": 900, "hi": 1148},
        {"name": "lebepel_decode", "kind": "lebepel", "phase": "decode", "n": 64, "lo": 700, "hi": 1200},
        # the routed-expert design: prompts, and a batch of sessions
        {"name": "fusasun_prompts", "kind": "fusasun", "phase": "prefill", "n": 4, "lo": 900, "hi": 1148},
        {"name": "fusasun_decode", "kind": "fusasun", "phase": "decode", "n": 64, "lo": 700, "hi": 1200},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["embed", "search", "llama", "lebepel", "fusasun"])
    if kind == "embed":
        lo = rng.randint(8, 100)
        return {"kind": kind, "n": _log(rng, 1, 1000), "lo": lo, "hi": lo + rng.randint(0, 100)}
    if kind == "search":
        return {"kind": kind, "rows": _log(rng, 20001, 480000), "n": _log(rng, 1, 16), "k": rng.randint(1, 8)}
    if rng.random() < 0.5:
        n = _log(rng, 1, 8)
        mean = _log(rng, 40, 4096 // n)
        return {"kind": kind, "phase": "prefill", "n": n, "lo": mean - mean // 5, "hi": mean + (mean // 6 if n > 1 else 0)}
    mean = _log(rng, 100, 950)
    return {"kind": kind, "phase": "decode", "n": _log(rng, 1, 120 if kind == "llama" else 64), "lo": mean - mean // 4, "hi": mean + mean // 4}


def _lens(case):
    """The lengths of a case's sequences: spread over lo..hi, in mixed order."""
    n, lo, hi = case["n"], case["lo"], case["hi"]
    out = [lo + (hi - lo) * i // max(n - 1, 1) for i in range(n)]
    random.Random(n).shuffle(out)
    return out


# ---------------------------------------------------------------------------------------------- weights
class _Rand:
    """Normal tensors on the device from one seed."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def __call__(self, *shape, scale=1.0, shift=0.0, dtype=F32):
        return torch.randn(*shape, generator=self.g, device=DEV, dtype=F32).mul_(scale).add_(shift).to(dtype)

    def lin(self, out, inp):
        return self(out, inp, scale=1 / math.sqrt(inp), dtype=BF)


def _encoder_weights(cfg, seed):
    r, H, I = _Rand(seed), cfg.hidden, cfg.intermediate
    sd = {"embeddings.word_embeddings.weight": r(cfg.vocab_size, H, scale=0.5, dtype=BF),
          "embeddings.position_embeddings.weight": r(cfg.max_position, H, scale=0.2, dtype=BF),
          "embeddings.token_type_embeddings.weight": r(cfg.type_vocab_size, H, scale=0.1, dtype=BF)}

    def norm(p):
        sd.update({p + ".weight": r(H, scale=0.1, shift=1.0, dtype=BF), p + ".bias": r(H, scale=0.1, dtype=BF)})

    norm("embeddings.LayerNorm")
    for i in range(cfg.num_layers):
        p = f"encoder.layer.{i}."
        for n, o, k in (("attention.self.query", H, H), ("attention.self.key", H, H), ("attention.self.value", H, H),
                        ("attention.output.dense", H, H), ("intermediate.dense", I, H), ("output.dense", H, I)):
            sd[p + n + ".weight"] = r.lin(o, k)
            sd[p + n + ".bias"] = r(o, scale=0.1, dtype=BF)
        norm(p + "attention.output.LayerNorm")
        norm(p + "output.LayerNorm")
    return sd


def _llama_config():
    """The 8B's layer (width 4096, 32 / 8 heads of 128, feed-forward 14336), four of them."""
    return decoder_config("llama-3-8b", num_layers=4, vocab_size=VOCAB, max_position=8192)


def _llama_weights(cfg, seed):
    r, W, D, I = _Rand(seed), cfg.hidden, cfg.head_dim, cfg.intermediate
    sd = {"model.embed_tokens.weight": r(cfg.vocab_size, W, dtype=BF), "lm_head.weight": r.lin(cfg.vocab_size, W),
          "model.norm.weight": r(W, scale=0.1, shift=1.0, dtype=BF)}
    for i in range(cfg.num_layers):
        p = f"model.layers.{i}."
        for n, o, k in (("self_attn.q_proj", cfg.num_heads * D, W), ("self_attn.k_proj", cfg.num_kv_heads * D, W),
                        ("self_attn.v_proj", cfg.num_kv_heads * D, W), ("self_attn.o_proj", W, cfg.num_heads * D),
                        ("mlp.gate_proj", I, W), ("mlp.up_proj", I, W), ("mlp.down_proj", W, I)):
            sd[p + n + ".weight"] = r.lin(o, k)
        sd[p + "input_layernorm.weight"] = r(W, scale=0.1, shift=1.0, dtype=BF)
        sd[p + "post_attention_layernorm.weight"] = r(W, scale=0.1, shift=1.0, dtype=BF)
    return sd


def _lebepel_config():
    """The decoder benchmark's sizes at width 2048."""
    return LebepelConfig("lebepel-w2048", VOCAB, 2048, lebepel_layers(8, 2048, 16, 4, 128, 5632, 64, 64, 128, 8, 4, 8),
                         max_position=8192, residual_mult=0.5, logit_softcap=30.0)


def _lebepel_weights(cfg, seed):
    r, W = _Rand(seed), cfg.hidden
    sd = {"embed": r(cfg.vocab_size, W, scale=0.5, dtype=BF), "pos": r(cfg.max_position, W, scale=0.5, dtype=BF),
          "final.norm": r(W, scale=0.05), "head": r.lin(cfg.vocab_size, W)}
    for i, l in enumerate(cfg.layers):
        b, p, m = f"l{i}.", f"l{i}.mix.", l.mixer
        sd[b + "norm1"] = r(W, scale=0.05)
        if l.type == "attention":
            H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            for n, o in (("q", H * D), ("k", G * D), ("v", G * V)):
                sd[p + n], sd[p + n + ".b"] = r.lin(o, W), r(o, scale=0.1, dtype=BF)
            sd[p + "o"], sd[p + "o.b"] = r.lin(W, H * V), r(W, scale=0.1)
            sd[p + "r1"], sd[p + "r2"] = r(H, scale=0.1, shift=0.5), r(H).abs_().mul_(0.2).add_(0.05)
            sd[p + "pb"] = r(H, scale=0.1)
        else:
            H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
            inner, ch = H * P, H * P + 2 * G * N
            sd[p + "in"] = r.lin(inner + ch + H, W)
            sd[p + "conv"], sd[p + "conv.b"] = r(ch, m["conv"], scale=0.3), r(ch, scale=0.1)
            sd[p + "dt_bias"], sd[p + "A_log"], sd[p + "D"] = r(H, scale=0.5, shift=-1.0), r(H, scale=0.3), r(H, scale=0.2, shift=1.0)
            sd[p + "norm"], sd[p + "o"] = r(inner, scale=0.05, shift=1.0), r.lin(W, inner)
        ff = l.mlp["ff"]
        sd[b + "mlp.gate"], sd[b + "mlp.up"], sd[b + "mlp.down"] = r.lin(ff, W), r.lin(ff, W), r.lin(W, ff)
    return sd


def _fusasun_config():
    """The decoder benchmark's sizes at width 2048."""
    return FusasunConfig("fusasun-w2048", VOCAB, 2048,
                         fusasun_layers(8, 16, 128, 2816, 16, 2, kv_heads=4, window=512, pool=64, rot_dim=64, q_rank=1024, kv_rank=512),
                         embed_scale=1.0, canon_taps=4)


def _fusasun_weights(cfg, seed):
    r, W = _Rand(seed), cfg.hidden
    one = dict(scale=0.1, shift=1.0)
    sd = {"embed": r(cfg.vocab_size, W, dtype=BF), "final.norm": r(W, **one), "head": r.lin(cfg.vocab_size, W)}
    for i, l in enumerate(cfg.layers):
        b, p, m = f"l{i}.", f"l{i}.mix.", l.mixer
        sd.update({b + "norm1": r(W, **one), b + "norm1b": r(W, **one), b + "rg1": r.lin(W, W), b + "rg1.b": r(W, scale=0.5),
                   b + "canon1": r(W, cfg.canon_taps, scale=0.3)})
        H, D, V = m["heads"], m["dim"], m["vdim"]
        if l.type == "attention":
            G = m["kv_heads"]
            sd.update({p + "q": r.lin(H * D, W), p + "k": r.lin(G * D, W), p + "v": r.lin(G * V, W), p + "o": r.lin(W, H * V)})
        else:
            R, Q, rd = m["kv_rank"], m["q_rank"], m["rot_dim"]
            sd.update({p + "dq": r.lin(Q, W), p + "dq.norm": r(Q, **one), p + "uq": r.lin(H * (D + rd), Q),
                       p + "dkv": r.lin(R + rd, W), p + "dkv.norm": r(R, **one), p + "uk": r.lin(H * D, R),
                       p + "uv": r.lin(H * V, R), p + "g": r.lin(H, W), p + "o": r.lin(W, H * V)})
        E, top, ff = l.mlp["router"]["experts"], l.mlp["router"]["top"], l.mlp["expert"]["ff"]
        for j in range(E):
            e = f"{b}mlp.e{j}."
            sd.update({e + "gate": r.lin(ff, W), e + "up": r.lin(ff, W), e + "down": r.lin(W, ff)})
        sd[b + "mlp.table"] = torch.rand(cfg.vocab_size, E, generator=r.g, device=DEV).argsort(1)[:, :top].to(torch.int32)
        sd.update({b + "norm2": r(W, **one), b + "norm2b": r(W, **one), b + "rg2": r.lin(W, W), b + "rg2.b": r(W, scale=0.5)})
    return sd


_DECODERS = {"llama": (_llama_config, _llama_weights, LlamaModel, "load_hf_state_dict"),
             "lebepel": (_lebepel_config, _lebepel_weights, LebepelModel, "load_state_dict_native"),
             "fusasun": (_fusasun_config, _fusasun_weights, FusasunModel, "load_state_dict_native")}


# ---------------------------------------------------------------------------------------------- inputs
def _encoder_inputs(case, seed):
    rng, V = random.Random(seed), encoder_config("bge-base").vocab_size
    return [[101] + [rng.randrange(1000, V) for _ in range(n - 2)] + [102] for n in _lens(case)]


def _search_inputs(case, seed):
    """Unit vectors around the topics of a corpus, and questions near some of them."""
    r, D = _Rand(seed), 768
    topics = r(2000, D)
    at = torch.randint(0, 2000, (case["rows"],), generator=r.g, device=DEV)
    corpus = torch.empty(case["rows"], D, device=DEV, dtype=BF)
    for a in range(0, case["rows"], 65536):
        x = topics[at[a:a + 65536]]
        corpus[a:a + 65536] = torch.nn.functional.normalize(x + r(*x.shape, scale=0.7), dim=1)
    q = topics[torch.randint(0, 2000, (case["n"],), generator=r.g, device=DEV)]
    return corpus, torch.nn.functional.normalize(q + r(*q.shape, scale=0.7), dim=1).to(BF)


def _token_inputs(case, seed):
    """(prompts, for a decode pass the tokens that its steps are given)"""
    rng = random.Random(seed)
    prompts = [[rng.randrange(VOCAB) for _ in range(n)] for n in _lens(case)]
    return prompts, [[rng.randrange(VOCAB) for _ in range(STEPS)] for _ in prompts]


# ---------------------------------------------------------------------------------------------- passes
@torch.no_grad()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "embed":
        cfg = encoder_config("bge-base")
        model = EncoderModel(cfg, BF, DEV).load_hf_state_dict(_encoder_weights(cfg, seed)).eval()
        eng = EmbeddingEngine(model, None, cfg.name)
        seqs = _encoder_inputs(case, seed)
        if len(seqs) == 1:  # as a server does at its start
            eng.capture_queries(max_len=min(64, len(seqs[0])), dtypes=(F32,))
        return {"case": case, "engine": eng, "seqs": seqs}
    if kind == "search":
        corpus, q = _search_inputs(case, seed)
        index = RagIndex(None, backend="gpu", device=DEV)
        index.chunks = [RagChunk("doc#0", "doc", "")] * case["rows"]
        index.set_gpu_corpus(corpus)
        return {"case": case, "index": index, "q": q}
    make_cfg, make_weights, cls, load = _DECODERS[kind]
    cfg = make_cfg()
    model = getattr(cls(cfg, dtype=BF, device=DEV), load)(make_weights(cfg, seed)).eval()
    prompts, given = _token_inputs(case, seed)
    n = len(prompts)
    blocks = sum(-(-(len(p) + STEPS) // BLOCK) for p in prompts) + 16
    eng = LLMEngine(model, None, block_size=BLOCK, max_model_len=2048 if case["phase"] == "decode" else 8192, max_num_seqs=max(n, 8),
                    num_blocks=blocks, eos_ids=set(), enable_prefix_caching=False)
    if case["phase"] == "prefill":
        return {"case": case, "engine": eng, "entries": [(f"r{i}", p, [len(p) - 1]) for i, p in enumerate(prompts)],
                "end": [f"r{i}" for i in range(n)]}
    run_ = eng.runner
    with torch.inference_mode():  # as a server does at its start
        run_.capture(min(b for b in run_.graph_sizes if b >= n))
    seqs = [Sequence(p, SamplingParams(max_tokens=STEPS + 1)) for p in prompts]
    group, rows = [], 0
    for s in seqs:
        if not eng.scheduler.admit_forced(s, s.length + STEPS):
            raise RuntimeError("the cache pool does not hold the contexts")
        group.append((s, 0, s.length))
        rows += s.length
        if rows >= 8192 or s is seqs[-1]:
            run_.forward_logits(group, want={})
            group, rows = [], 0
    return {"case": case, "engine": eng, "seqs": seqs, "given": given}


def run(state):
    kind = state["case"]["kind"]
    if kind == "embed":
        return state["engine"].embed_ids(state["seqs"])
    if kind == "search":
        k = state["case"]["k"]
        hits = state["index"].search_vectors(state["q"], k)
        return {"ids": np.array([[i for i, _ in h] for h in hits], dtype=np.int64),
                "scores": np.array([[s for _, s in h] for h in hits], dtype=np.float64)}
    if state["case"]["phase"] == "prefill":
        return state["engine"].replay_step(state["entries"], state["end"])
    # consecutive decode steps over given tokens; every pass starts from the prompts' ends again
    out, runner = [], state["engine"].runner
    for k in range(STEPS):
        items = []
        for s, t in zip(state["seqs"], state["given"]):
            s.output_ids = t[:k + 1]
            s.num_computed = len(s.prompt_ids) + k
            items.append((s, s.num_computed, 1))
        out.append(runner.forward_logits(items)[1].to(F32, copy=True))
    return out


# ---------------------------------------------------------------------------------------------- what a pass cannot do without
def _decoder_sizes(kind):
    """(weights of every row's products, weights of one expert, experts, experts per row, cache bytes per key, state bytes per
    sequence, flops per row and key) over all layers; embedding and head apart."""
    cfg = _DECODERS[kind][0]()
    W = cfg.hidden
    if kind == "llama":
        D, L = cfg.head_dim, cfg.num_layers
        per = W * (cfg.num_heads + 2 * cfg.num_kv_heads) * D + cfg.num_heads * D * W + 3 * W * cfg.intermediate
        return L * per, 0, 0, 0, L * 4 * cfg.num_kv_heads * D, 0, L * 4 * cfg.num_heads * D
    dense = kv = st = fl = ew = 0
    for l in cfg.layers:
        m = l.mixer
        if kind == "lebepel":
            dense += 3 * W * l.mlp["ff"]
            if l.type == "attention":
                dense += W * ((m["heads"] + 2 * m["kv_heads"]) * m["dim"] + m["heads"] * m["dim"])
                kv += 4 * m["kv_heads"] * m["dim"]
                fl += 4 * m["heads"] * m["dim"]
            else:
                inner, gn = m["heads"] * m["vdim"], m["groups"] * m["state"]
                dense += W * (3 * inner + 2 * gn + m["heads"])
                st += 2 * 4 * inner * m["state"]
        else:
            dense += 2 * W * W
            ew += 3 * W * l.mlp["expert"]["ff"]
            H, D = m["heads"], m["dim"]
            if l.type == "attention":
                dense += W * (2 * H + 2 * m["kv_heads"]) * D
                kv += 4 * m["kv_heads"] * D
                fl += 4 * H * D
            else:
                R, Q, rd = m["kv_rank"], m["q_rank"], m["rot_dim"]
                dense += W * (Q + R + rd + H) + Q * H * (D + rd) + R * 2 * H * D + W * H * D
                kv += 2 * (R + rd)
                fl += 2 * H * (2 * D + rd)
    if kind == "lebepel":
        return dense, 0, 0, 0, kv, st, fl
    return dense, ew, 16, 2, kv, 0, fl


def work(case):
    kind = case["kind"]
    if kind == "embed":
        c, lens = encoder_config("bge-base"), _lens(case)
        T, per = sum(lens), c.num_layers * (4 * c.hidden ** 2 + 2 * c.hidden * c.intermediate)
        return {"bytes": 2 * per + 2 * T * c.hidden + 4 * len(lens) * c.hidden,
                "flops": 2 * T * per + 4 * c.num_layers * c.hidden * sum(n * n for n in lens)}
    if kind == "search":
        return {"bytes": 2 * 768 * (case["rows"] + case["n"]) + 4 * case["rows"], "flops": 2 * 768 * case["rows"] * case["n"]}
    cfg, lens = _DECODERS[kind][0](), _lens(case)
    dense, ew, E, top, kv, st, fl = _decoder_sizes(kind)
    window = 512 if kind == "fusasun" else 1 << 30
    head = cfg.vocab_size * cfg.hidden
    if case["phase"] == "prefill":
        T, n = sum(lens), len(lens)
        keys = sum(min(i + 1, window) for x in lens for i in range(x))
        touched = E * (1 - (1 - top / E) ** T) if E else 0
        return {"bytes": 2 * (dense + ew * touched + head) + 2 * T * cfg.hidden + T * kv + n * (st + 4 * cfg.vocab_size),
                "flops": 2 * T * (dense + ew * top) + 2 * n * head + keys * fl + 2 * T * st / 4}
    n = len(lens)
    keys = sum(min(x + 1 + k, window) for x in lens for k in range(STEPS))
    touched = E * (1 - (1 - top / E) ** n) if E else 0
    return {"bytes": STEPS * (2 * (dense + ew * touched + head) + n * (2 * cfg.hidden + 4 * cfg.vocab_size + st)) + keys * kv,
            "flops": 2 * STEPS * n * (dense + ew * top + head + st / 4) + keys * fl}


def tolerance(case):
    """About four times what was measured against ``exact``: scores are f32 sums of products of bf16 values, the
    other results bf16 activations through 4 to 12 layers."""
    if case["kind"] == "search":
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.02}
    if case["kind"] == "embed":
        return {"rel": 0.03, "max": 0.15}
    return {"rel": 0.04, "max": 0.2}


# ---------------------------------------------------------------------------------------------- the same in float64
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _sig(x):
    return torch.sigmoid(x)


def _lnorm(x, w, b, eps):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + eps) * w + b


def _double(sd, prefix):
    """The tensors under ``prefix`` without it, floating ones in f64."""
    return {k[len(prefix):]: v.double() if v.is_floating_point() else v.long() for k, v in sd.items() if k.startswith(prefix)}


def _batches(seqs, most):
    """[(indices, ids [b, T])] of sequences of similar length, padded behind their ends."""
    order = sorted(range(len(seqs)), key=lambda i: len(seqs[i]))
    out, at = [], 0
    while at < len(order):
        b = 1
        while at + b < len(order) and (b + 1) * len(seqs[order[at + b]]) <= most:
            b += 1
        idx = order[at:at + b]
        ids = torch.zeros(b, max(len(seqs[i]) for i in idx), dtype=torch.long)
        for r, i in enumerate(idx):
            ids[r, :len(seqs[i])] = torch.tensor(seqs[i])
        out.append((idx, ids.to(DEV)))
        at += b
    return out


def _attend(s, v):
    """softmax over the last axis of s [b, h, i, j] times v [b, j, h, d]"""
    return torch.matmul(torch.softmax(s, -1), v.transpose(1, 2)).transpose(1, 2)


def _exact_encoder(case, seed):
    cfg, sd, seqs = encoder_config("bge-base"), None, _encoder_inputs(case, seed)
    sd = {k: v.double() for k, v in _encoder_weights(cfg, seed).items()}
    H, nh = cfg.hidden, cfg.num_heads
    out = torch.empty(len(seqs), H, device=DEV, dtype=F64)
    for idx, ids in _batches(seqs, 8192):
        b, T = ids.shape
        lens = torch.tensor([len(seqs[i]) for i in idx], device=DEV)
        hide = (torch.arange(T, device=DEV)[None, :] >= lens[:, None])[:, None, None, :]
        e = "embeddings."
        h = sd[e + "word_embeddings.weight"][ids] + sd[e + "position_embeddings.weight"][:T] + sd[e + "token_type_embeddings.weight"][0]
        h = _lnorm(h, sd[e + "LayerNorm.weight"], sd[e + "LayerNorm.bias"], cfg.norm_eps)
        for i in range(cfg.num_layers):
            p = f"encoder.layer.{i}."

            def lin(x, n):
                return x @ sd[p + n + ".weight"].T + sd[p + n + ".bias"]

            def norm(x, n):
                return _lnorm(x, sd[p + n + ".LayerNorm.weight"], sd[p + n + ".LayerNorm.bias"], cfg.norm_eps)

            q, k, v = (lin(h, "attention.self." + n).view(b, T, nh, H // nh) for n in ("query", "key", "value"))
            s = torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1).contiguous()) / math.sqrt(H // nh)
            a = _attend(s.masked_fill(hide, -math.inf), v).reshape(b, T, H)
            h = norm(lin(a, "attention.output.dense") + h, "attention.output")
            f = lin(h, "intermediate.dense")
            h = norm(lin(0.5 * f * (1 + torch.erf(f / math.sqrt(2))), "output.dense") + h, "output")
        out[idx] = torch.nn.functional.normalize(h[:, 0], dim=1)
    return out


def _exact_search(case, seed):
    corpus, q = _search_inputs(case, seed)
    q = q.double()
    s = torch.empty(case["n"], case["rows"], device=DEV, dtype=F64)
    for a in range(0, case["rows"], 65536):
        c = corpus[a:a + 65536].double()
        s[:, a:a + 65536] = (q @ c.T) / (q.norm(dim=1)[:, None] * c.norm(dim=1)[None, :] + 1e-9)
    top, at = s.sort(dim=1, descending=True, stable=True)
    return {"ids": at[:, :case["k"]].cpu().numpy(), "scores": top[:, :case["k"]].cpu().numpy()}


def _turn(x, f, mag, pairs):
    """x [b, T, h, d] rotated by the angles position * f: halves (i, i + d/2) or adjacent ``pairs`` (2i, 2i + 1)."""
    a = torch.arange(x.shape[1], device=DEV, dtype=F64)[:, None] * f
    c, s = (a.cos() * mag)[None, :, None], (a.sin() * mag)[None, :, None]
    n = f.numel()
    u, v = (x[..., 0::2], x[..., 1::2]) if pairs else (x[..., :n], x[..., n:])
    y = (u * c - v * s, v * c + u * s)
    return torch.stack(y, -1).flatten(-2) if pairs else torch.cat(y, -1)


def _wave_freqs(dims, base, factor, low, high, orig):
    f = base ** (-torch.arange(0, dims, 2, device=DEV, dtype=F64) / dims)
    turns = orig * f / (2 * math.pi)
    mix = ((turns - low) / (high - low)).clamp(0, 1)
    return (1 - mix) * f / factor + mix * f


def _ramp_freqs(dims, base, sc):
    f = base ** (-torch.arange(0, dims, 2, device=DEV, dtype=F64) / dims)
    at = lambda t: dims * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(base))  # noqa: E731
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, device=DEV, dtype=F64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / sc["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def _scores(q, k, scale):
    """q [b, T, h, d], k [b, T, g, d] -> [b, h, T, T]"""
    k = k.repeat_interleave(q.shape[2] // k.shape[2], 2)
    return torch.matmul(q.transpose(1, 2), k.permute(0, 2, 3, 1).contiguous()) * scale


def _gap(T):
    i = torch.arange(T, device=DEV)
    return i[:, None] - i[None, :]


def _llama_layers(cfg, sd, ids):
    b, T = ids.shape
    H, G, D, eps = cfg.num_heads, cfg.num_kv_heads, cfg.head_dim, cfg.norm_eps
    sc = cfg.rope_scaling
    f = _wave_freqs(D, cfg.rope_theta, sc["factor"], sc["low_freq_factor"], sc["high_freq_factor"], sc["original_max_position_embeddings"])
    x = sd["model.embed_tokens.weight"][ids].double()
    for i in range(cfg.num_layers):
        w = _double(sd, f"model.layers.{i}.")
        h = _rms(x, eps) * w["input_layernorm.weight"]
        q = _turn((h @ w["self_attn.q_proj.weight"].T).view(b, T, H, D), f, 1.0, False)
        k = _turn((h @ w["self_attn.k_proj.weight"].T).view(b, T, G, D), f, 1.0, False)
        v = (h @ w["self_attn.v_proj.weight"].T).view(b, T, G, D).repeat_interleave(H // G, 2)
        a = _attend(_scores(q, k, D ** -0.5).masked_fill_(_gap(T) < 0, -math.inf), v)
        x = x + a.reshape(b, T, H * D) @ w["self_attn.o_proj.weight"].T
        h = _rms(x, eps) * w["post_attention_layernorm.weight"]
        g = h @ w["mlp.gate_proj.weight"].T
        x = x + (g * _sig(g) * (h @ w["mlp.up_proj.weight"].T)) @ w["mlp.down_proj.weight"].T
    return _rms(x, eps) * sd["model.norm.weight"].double(), sd["lm_head.weight"].double(), 0.0


def _conv(x, w):
    """x [b, T, C], w [C, taps], the last tap on the current token"""
    taps, T = w.shape[1], x.shape[1]
    p = torch.nn.functional.pad(x, (0, 0, taps - 1, 0))
    return sum(p[:, j:j + T] * w[:, j] for j in range(taps))


def _state_space(h, w, m, eps):
    b, T, _ = h.shape
    H, P, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    inner = H * P
    u = h @ w["in"].T
    z, xbc, dt = u[..., :inner], u[..., inner:-H], u[..., -H:]
    xbc = _conv(xbc, w["conv"]) + w["conv.b"]
    xbc = xbc * _sig(xbc)
    x = xbc[..., :inner].view(b, T, H, P)
    B, C = (t.view(b, T, G, N).repeat_interleave(H // G, 2) for t in (xbc[..., inner:inner + G * N], xbc[..., inner + G * N:]))
    dt = torch.nn.functional.softplus(dt + w["dt_bias"])
    keep = torch.exp(-torch.exp(w["A_log"]) * dt)
    S = torch.zeros(b, H, N, P, device=DEV, dtype=F64)
    y = torch.empty(b, T, H, P, device=DEV, dtype=F64)
    add = B * dt[..., None]
    for t in range(T):
        S.mul_(keep[:, t, :, None, None]).add_(add[:, t, :, :, None] * x[:, t, :, None, :])
        y[:, t] = torch.matmul(C[:, t, :, None, :], S)[:, :, 0]
    y = (y + x * w["D"][:, None]).reshape(b, T, inner) * (z * _sig(z))
    return (_rms(y.view(b, T, m["norm_groups"], -1), eps).reshape(b, T, inner) * w["norm"]) @ w["o"].T


def _lebepel_layers(cfg, sd, ids):
    b, T = ids.shape
    eps = cfg.norm_eps
    x = sd["embed"][ids].double() + sd["pos"][:T].double()
    for i, l in enumerate(cfg.layers):
        w, m = _double(sd, f"l{i}.mix."), l.mixer
        h = _rms(x, eps) * (1 + sd[f"l{i}.norm1"].double())
        if l.type == "attention":
            H, G, D = m["heads"], m["kv_heads"], m["dim"]
            q = _rms((h @ w["q"].T + w["q.b"]).view(b, T, H, D), eps)
            k = _rms((h @ w["k"].T + w["k.b"]).view(b, T, G, D), eps)
            v = (h @ w["v"].T + w["v.b"]).view(b, T, G, m["vdim"]).repeat_interleave(H // G, 2)
            d = _gap(T)
            far = w["r1"][:, None, None] * torch.log1p(w["r2"][:, None, None] * d.clamp(min=0))
            p = _sig(_scores(q, k, m["scale"]) - far + w["pb"][:, None, None]) * (d >= 0)
            y = torch.matmul(p, v.transpose(1, 2)).transpose(1, 2).reshape(b, T, -1) @ w["o"].T + w["o.b"]
        else:
            y = _state_space(h, w, m, eps)
        f = _double(sd, f"l{i}.mlp.")
        g = h @ f["gate"].T
        x = x + cfg.residual_mult * (y + (g * _sig(g) * (h @ f["up"].T)) @ f["down"].T)
    return _rms(x, eps) * (1 + sd["final.norm"].double()), sd["head"].double(), cfg.logit_softcap


def _pooled_attention(h, w, m):
    b, T, _ = h.shape
    H, G, D, size, P = m["heads"], m["kv_heads"], m["dim"], m["mask"]["size"], m["mask"]["pool"]
    r = m["rot"]
    sc = r["scaling"]
    f = _wave_freqs(r["dims"], r["base"], sc["factor"], sc["low"], sc["high"], sc["original"])
    q = _turn((h @ w["q"].T).view(b, T, H, D), f, 1.0, True)
    k = _turn((h @ w["k"].T).view(b, T, G, D), f, 1.0, True)
    v = (h @ w["v"].T).view(b, T, G, -1)
    n = T // P
    mean = lambda t: t[:, :n * P].reshape(b, n, P, G, -1).mean(2)  # noqa: E731
    d = _gap(T)
    s = _scores(q, k, m["scale"]).masked_fill_((d < 0) | (d >= size), -math.inf)
    i, e = torch.arange(T, device=DEV)[:, None], torch.arange(n, device=DEV)[None, :] * P + P - 1
    sp = _scores(q, mean(k), m["scale"]).masked_fill_(e > i - size, -math.inf)
    return _attend(torch.cat([sp, s], -1), torch.cat([mean(v), v], 1).repeat_interleave(H // G, 2)).reshape(b, T, -1) @ w["o"].T


def _latent_attention(h, w, m, eps):
    b, T, _ = h.shape
    H, D, rd, V, R = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
    f, mag = _ramp_freqs(rd, m["rot"]["base"], m["rot"]["scaling"])
    q = ((_rms(h @ w["dq"].T, eps) * w["dq.norm"]) @ w["uq"].T).view(b, T, H, D + rd)
    q = torch.cat([q[..., :D], _turn(q[..., D:], f, mag, True)], -1)
    c = h @ w["dkv"].T
    kr = _turn(c[..., None, R:], f, mag, True).expand(b, T, H, rd)
    c = _rms(c[..., :R], eps) * w["dkv.norm"]
    k = torch.cat([(c @ w["uk"].T).view(b, T, H, D), kr], -1)
    d = _gap(T)
    s = _scores(q, k, m["scale"]).masked_fill_((d < 0) | (d >= m["mask"]["size"]), -math.inf)
    a = _attend(s, (c @ w["uv"].T).view(b, T, H, V)) * _sig(h @ w["g"].T)[..., None]
    return a.reshape(b, T, -1) @ w["o"].T


def _fusasun_layers(cfg, sd, ids):
    b, T = ids.shape
    eps = cfg.norm_eps
    x = sd["embed"][ids].double() * cfg.embed_scale
    for i, l in enumerate(cfg.layers):
        w, m = _double(sd, f"l{i}.mix."), l.mixer
        p = {k: sd[f"l{i}." + k].double() for k in ("norm1", "norm1b", "rg1", "rg1.b", "canon1", "norm2", "norm2b", "rg2", "rg2.b")}
        h = _rms(x, eps) * p["norm1"]
        hc = h + _conv(h, p["canon1"])
        y = _pooled_attention(hc, w, m) if l.type == "attention" else _latent_attention(hc, w, m, eps)
        x = x + _rms(_sig(h @ p["rg1"].T + p["rg1.b"]) * y, eps) * p["norm1b"]
        h = _rms(x, eps) * p["norm2"]
        flat, table = h.reshape(b * T, -1), sd[f"l{i}.mlp.table"].long()[ids.reshape(-1)]
        y = torch.zeros_like(flat)
        for j in range(l.mlp["router"]["experts"]):
            e = _double(sd, f"l{i}.mlp.e{j}.")
            at = (table == j).any(1).nonzero()[:, 0]
            g = flat[at] @ e["gate"].T
            y[at] += ((g * _sig(g) * (flat[at] @ e["up"].T)) @ e["down"].T) / table.shape[1]
        x = x + _rms(_sig(h @ p["rg2"].T + p["rg2.b"]) * y.view(b, T, -1), eps) * p["norm2b"]
    return _rms(x, eps) * sd["final.norm"].double(), sd["head"].double(), 0.0


_LAYERS = {"llama": _llama_layers, "lebepel": _lebepel_layers, "fusasun": _fusasun_layers}


def _exact_decoder(case, seed):
    kind = case["kind"]
    make_cfg, make_weights = _DECODERS[kind][:2]
    cfg = make_cfg()
    sd = make_weights(cfg, seed)
    prompts, given = _token_inputs(case, seed)
    decode = case["phase"] == "decode"
    seqs = [p + g for p, g in zip(prompts, given)] if decode else prompts
    steps = STEPS if decode else 1
    out = torch.empty(steps, len(seqs), cfg.vocab_size, device=DEV, dtype=F64)
    for idx, ids in _batches(seqs, 16384):
        h, head, cap = _LAYERS[kind](cfg, sd, ids)
        for r, i in enumerate(idx):
            z = h[r, len(seqs[i]) - steps:len(seqs[i])] @ head.T
            out[:, i] = cap * torch.tanh(z / cap) if cap else z
    return list(out) if decode else out[0]


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "embed":
        return _exact_encoder(case, seed)
    if case["kind"] == "search":
        return _exact_search(case, seed)
    return _exact_decoder(case, seed)
