"""What is timed: the work a user of this framework has its engines do, through the engine's public calls.

A case is one member model with an engine around it. Weights are random bf16 tensors of the named architecture (drawn
on the GPU from the seed), tokens are random. Three kinds of pass:

* ``generate``: requests are submitted and the engine runs until all are answered (prompt steps, then recorded decode
  steps). Returned: every chain's tokens and its decision log-probs, which is what the vote and the judge read.
* ``score``: prompts whose last position is scored against listed targets (a judge reading candidates).
* ``replay``: given tokens go through ``Engine.replay_step``, as ``bin/trace_run`` drives it; returned: logits.

The language model head is the embedding table shifted by a few rows, scaled so that the next token has most of the
probability, as a trained model's has: what is sampled then does not hang on the last bit of a logit, and tokens can be
compared. Transformers have the published width of the named model, the larger ones and the drawn ones fewer of its equal
layers, so that a pass stays short; the hybrid decoders have the sizes of ``bench.py --hybrid``.
"""
from __future__ import annotations

import math
import zlib

import numpy as np
import torch

from llm_consensus_amd import bench_hybrid
from llm_consensus_amd._native import core
from llm_consensus_amd.engine.engine import Engine
from llm_consensus_amd.models.config import get_preset
from llm_consensus_amd.models.hybrid import HybridModel, config_to_dict, param_shapes
from llm_consensus_amd.models.transformer import TransformerModel, hf_param_shape

DEV = "cuda:0"
SHIFT = 17              # the token that follows token t is t + SHIFT
BLOCK = 64
HYBRID = {"nidozen": bench_hybrid.hybrid_config, "telurax": bench_hybrid.telurax_config,
          "gizilorn": bench_hybrid.gizilorn_config, "rizurax": bench_hybrid.rizurax_config}


# ------------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one person's question to one 8B member: every step is a single row
        dict(name="ask_one", kind="generate", model="llama-3-8b", layers=32, questions=1, chains=1, prompt=96, new=16,
             temperature=0.0),
        # a batch of the vote ensemble's questions (512-token prompts) through one 7B member
        dict(name="vote_batch", kind="generate", model="qwen2.5-7b", layers=28, questions=16, chains=1, prompt=512, new=24,
             temperature=0.8),
        # self-consistency: sixteen sampled chains per question over one shared prompt
        dict(name="self_consistency", kind="generate", model="llama-3-8b", layers=16, questions=8, chains=16, prompt=480, new=24,
             temperature=0.8),
        # the judge reads questions with candidates (ragged lengths) and scores two verdicts; prompts over several steps
        dict(name="judge_score", kind="score", model="llama-3-70b", layers=4, questions=19, prompt=733),
        # the routed proposer: four samples per question
        dict(name="moe_generate", kind="generate", model="mixtral-8x7b", layers=6, questions=12, chains=4, prompt=200, new=16,
             temperature=0.8),
        # one long document, in portions of the step's token budget, under a sliding window
        dict(name="long_score", kind="score", model="mistral-7b", layers=8, questions=1, prompt=11003),
        # one prompt through a hybrid decoder, three designs at the middle size
        dict(name="nidozen_prompt", kind="replay", model="nidozen", size="2k", dtype="bf16", prompts=1, prompt=2048, steps=0),
        dict(name="telurax_prompt", kind="replay", model="telurax", size="2k", dtype="bf16", prompts=1, prompt=1500, steps=0),
        dict(name="rizurax_prompt", kind="replay", model="rizurax", size="2k", dtype="bf16", prompts=1, prompt=3001, steps=0),
        # several short prompts in one step, then given tokens one by one beside each other
        dict(name="gizilorn_trace", kind="replay", model="gizilorn", size="2k", dtype="bf16", prompts=4, prompt=700, steps=6),
        # the number format of reference traces: 32 bits throughout, small model, portions and single tokens
        dict(name="nidozen_trace_f32", kind="replay", model="nidozen", size="1k", dtype="f32", prompts=3, prompt=333, steps=8),
        # a batch of chats on a hybrid decoder: short prompts, recorded decode steps of 32 rows
        dict(name="rizurax_chats", kind="generate", model="rizurax", size="2k", questions=32, chains=1, prompt=64, new=32,
             temperature=0.8),
    ]


def _between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    k = rng.choice(["generate", "generate", "score", "replay", "replay", "replay", "chats"])
    temp = rng.choice([0.0, 0.8])
    if k == "generate":
        model = rng.choice(["llama-3-8b", "qwen2.5-7b", "mistral-7b", "mixtral-8x7b"])
        chains = rng.choice([1, 1, 4, 16])
        return dict(kind="generate", model=model, layers=4 if model == "mixtral-8x7b" else 8,
                    questions=_between(rng, 1, 128 // chains if chains > 1 else 24), chains=chains,
                    prompt=_between(rng, 24, 512), new=rng.randint(8, 24), temperature=temp)
    if k == "score":
        return dict(kind="score", model=rng.choice(["llama-3-8b", "qwen2.5-7b", "mistral-7b", "llama-3-70b"]), layers=4,
                    questions=_between(rng, 1, 19), prompt=_between(rng, 60, 733))
    model, size = rng.choice(sorted(HYBRID)), rng.choice(["1k", "2k"])
    if k == "chats":
        return dict(kind="generate", model=model, size=size, questions=_between(rng, 1, 48), chains=1,
                    prompt=_between(rng, 16, 200), new=rng.randint(8, 32), temperature=temp)
    f32 = rng.random() < 0.25
    return dict(kind="replay", model=model, size="1k" if f32 else size, dtype="f32" if f32 else "bf16", prompts=rng.randint(1, 4),
                prompt=_between(rng, 40, 400 if f32 else 750), steps=rng.choice([0, 0, rng.randint(1, 8)]))


# ------------------------------------------------------------------------------------------------ weights
def _is_hybrid(case):
    return case["model"] in HYBRID


def _config(case):
    if _is_hybrid(case):
        return HYBRID[case["model"]](bench_hybrid.SIZES[case["size"]])
    return get_preset(case["model"], num_layers=case["layers"])


# Head scale per family, such that the next token has a probability between about one half and one: the cosine between
# the final stream and the embedding row falls with depth, and a design that norms its sublayers' results falls fastest.
HEAD_GAIN = {"nidozen": 1.55, "telurax": 0.8, "rizurax": 0.95, "gizilorn": 1.0}


def _head_gain(case, cfg):
    if _is_hybrid(case):
        return HEAD_GAIN[case["model"]]
    cos = (1.0 + 0.45 * cfg.num_layers) ** -0.5
    return (math.log(cfg.vocab_size) + 3.0) / (cos * cfg.hidden_size ** 0.5)


class Weights:
    """Checkpoint tensors by name, drawn on the GPU, one stream per name."""

    def __init__(self, case, seed):
        self.case, self.seed, self.cfg = case, seed, _config(case)
        self.hybrid = _is_hybrid(case)
        self.shapes = param_shapes(self.cfg) if self.hybrid else None
        self.gen = torch.Generator(device=DEV)
        self.gain = _head_gain(case, self.cfg)

    # (routers' rows are larger than the others, so that their choices are clear-cut, as a trained router's are)
    def _randn(self, shape, name):
        self.gen.manual_seed((self.seed * 1000003 + zlib.crc32(name.encode())) & 0x7FFFFFFFFFFFFFFF)
        return torch.randn(shape, generator=self.gen, device=DEV)

    def __call__(self, name):
        return self.hybrid_tensor(name) if self.hybrid else self.transformer_tensor(name)

    def _shifted_head(self, embed_name):
        e = self(embed_name).float()
        return (torch.roll(e, SHIFT, 0) * (self.gain * e.shape[1] ** -0.5)).to(torch.bfloat16)

    def transformer_tensor(self, name):
        shape = hf_param_shape(self.cfg, name)
        if name == "lm_head.weight":
            return self._shifted_head("model.embed_tokens.weight")
        t = self._randn(shape, name)
        if name.endswith("norm.weight"):
            t = 1.0 + 0.1 * t
        elif len(shape) == 1:
            t = 0.1 * t
        elif name != "model.embed_tokens.weight":
            t = t * ((6.0 if name.endswith(".gate.weight") else 1.0) * shape[1] ** -0.5)
        return t.to(torch.bfloat16)

    def hybrid_tensor(self, name):
        shape, leaf = tuple(self.shapes[name]), name.split(".")[-1]
        if name == "head":
            return self._shifted_head("embed")
        t = self._randn(shape, name)
        offset = self.cfg.design.norm_offset != 0.0
        if ".hc" in name:               # streams that neither die out nor blow up
            n = self.cfg.streams
            t = 0.05 * t + {"in": 1.0 / n, "out": 1.0, "mix": torch.eye(n, device=DEV)}[leaf]
        elif leaf == "talk":
            t = 0.1 * t + torch.eye(shape[0], device=DEV)
        elif name == "embed":
            pass
        elif name == "bigram":
            t = 0.3 * t
        elif leaf == "conv":
            t = 0.5 * t
        elif len(shape) == 2:
            t = t * ((8.0 if leaf == "router" else 1.0) * shape[1] ** -0.5)
        elif offset and (leaf in ("norm1", "norm2") or name == "final.norm"):
            t = 0.1 * t
        elif leaf in ("norm", "norm1", "norm2"):
            t = 1.0 + 0.1 * t
        elif leaf == "dt_bias":
            t = -3.0 + t
        elif name.endswith("a2.b") or name.endswith("mix.f.b"):
            t = 2.0 + t
        elif leaf == "correction":
            t = 0.02 * t
        else:
            t = 0.1 * t
        return t.to(torch.bfloat16)


# ------------------------------------------------------------------------------------------------ inputs
def _lengths(case):
    """Prompt lengths: the stated one, and shorter ones beside it (questions are not all as long)."""
    n = case["prompts"] if case["kind"] == "replay" else case["questions"]
    return [max(4, case["prompt"] - (7 * i * i + 5 * i) % max(1, case["prompt"] // 3)) for i in range(n)]


def _tokens(case, seed, vocab):
    rng = np.random.default_rng([seed, 7])
    extra = case["steps"] if case["kind"] == "replay" else 0
    toks = [rng.integers(0, vocab, n + extra).tolist() for n in _lengths(case)]
    return toks, sorted(rng.choice(vocab, 8, replace=False).tolist())


def _wants(n):
    """Places of a prompt whose logits are asked for."""
    return sorted({n // 3, n - 1})


def prepare(case, seed):
    cfg = _config(case)
    w = Weights(case, seed)
    toks, targets = _tokens(case, seed, cfg.vocab_size)
    if _is_hybrid(case):
        model = HybridModel(cfg, DEV, torch.float32 if case.get("dtype") == "f32" else torch.bfloat16)
        model.set_weights(w)
    else:
        model = TransformerModel(cfg, DEV)
        model.set_weights_from_hf(w)
    longest = max(len(t) for t in toks) + case.get("new", 0)
    rows = len(toks) * case.get("chains", 1)
    per_seq = -(-longest // BLOCK) + 1
    kw = dict(num_kv_blocks=rows * per_seq + 8, block_size=BLOCK, max_model_len=longest + BLOCK, enable_prefix_cache=False,
              name=case["model"])
    if case["kind"] == "replay":        # as bin/trace_run makes its engine
        eng = Engine(model, max_batch_seqs=4, state_slots=4, use_graphs=False, pipeline_decode=False, **kw)
    else:
        eng = Engine(model, max_batch_seqs=max(rows, 4), **kw)
    state = dict(case=case, engine=eng, tokens=toks, targets=targets)
    if case["kind"] == "generate":
        params = []
        for i in range(len(toks)):
            p = core.SamplingParams()
            # (a nucleus that the likeliest token fills alone: the sampler does all its work, and what it returns is certain)
            p.temperature, p.top_p, p.max_new_tokens, p.ignore_eos, p.seed = case["temperature"], 0.3, case["new"], True, 1000 * i
            params.append(p)
        state["params"] = params
    return state


def run(s):
    case, eng, toks = s["case"], s["engine"], s["tokens"]
    if case["kind"] == "replay":
        return _replay(eng, toks, case["steps"])
    if case["kind"] == "generate":
        ids = [eng.submit(t, n=case["chains"], params=p, decision_ids=s["targets"]) for t, p in zip(toks, s["params"])]
    else:
        ids = [eng.submit(t, kind=core.RequestKind.Score, score_ids=s["targets"]) for t in toks]
    eng.run_until_done()
    outs = [eng.pop_result(i) for i in ids]
    if case["kind"] == "score":
        return np.array([o.scores for o in outs], np.float32)
    return {"tokens": np.array([o.token_ids for o in outs], np.int32),
            "decisions": np.array([o.decision_logprobs for o in outs], np.float32)}


def _replay(eng, toks, steps):
    ids = [eng.replay_open() for _ in toks]
    ns = [len(t) - steps for t in toks]
    if steps and len(toks) > 1:         # the last request comes in two portions, the second beside the others' single tokens
        cut = max(1, ns[-1] // 2)
    else:
        cut = ns[-1]
    first = [(r, t[:n], _wants(n)) for r, t, n in zip(ids[:-1], toks, ns)]
    first.append((ids[-1], toks[-1][:cut], _wants(cut)))
    out = [eng.replay_step(first)]
    for k in range(steps):
        e = [(r, [t[n + k]], [0]) for r, t, n in zip(ids, toks, ns)]
        if k == 0 and cut < ns[-1]:
            e[-1] = (ids[-1], toks[-1][cut:ns[-1] + 1], [ns[-1] - cut])
        out.append(eng.replay_step(e))
    for r in ids:
        eng.replay_close(r)
    return out


# ------------------------------------------------------------------------------------------------ least work
def _per_row(case, cfg):
    """(weights a row multiplies, weights a step of many rows reads, without the head and the tables), in numbers."""
    if not _is_hybrid(case):
        d, kv = cfg.hidden_size, cfg.kv_size
        attn = d * (cfg.q_size + 2 * kv) + cfg.q_size * d
        ff = 3 * d * cfg.intermediate_size
        return (cfg.num_layers * (attn + ff * max(1, cfg.experts_per_tok)), cfg.num_layers * (attn + ff * max(1, cfg.num_experts)))
    mult = read = 0
    shapes = param_shapes(cfg)
    for i, l in enumerate(cfg.layers):
        times = cfg.loop[2] if cfg.loop[0] <= i < cfg.loop[1] else 1
        for n, s in shapes.items():
            if n.startswith(f"l{i}.") and len(s) == 2:
                size = s[0] * s[1]
                share = l.moe.top / l.moe.outputs if l.moe is not None and n.split(".")[2][:1] == "e" else 1.0
                mult += times * share * size
                read += times * size
    return mult, read


def _pairs(case, cfg, n):
    """Flops of attention (scores and weighted values) over a prompt of n rows, all layers."""
    if not _is_hybrid(case):
        w = cfg.sliding_window or n
        seen = n * (n + 1) / 2 if n <= w else w * (w + 1) / 2 + (n - w) * w
        return cfg.num_layers * seen * 4 * cfg.q_size
    total = 0.0
    for i, _ in cfg.runs:
        l = cfg.layers[i]
        if l.type not in ("attention", "latent_attention"):
            continue
        w = min(n, l.window or n)
        seen = n * (n + 1) / 2 if w == n else w * (w + 1) / 2 + (n - w) * w
        if l.chunk:
            seen = (n // l.chunk) * l.chunk * (l.chunk + 1) / 2 + (n % l.chunk) * (n % l.chunk + 1) / 2
        width = 2 * (l.dim + l.vdim) if l.type == "attention" else 4 * l.kv_rank
        total += seen * l.heads * l.maps * width
    return total


def work(case):
    cfg = _config(case)
    mult, read = _per_row(case, cfg)
    head = cfg.vocab_size * cfg.hidden_size
    es = 4 if case.get("dtype") == "f32" else 2
    lens = _lengths(case)
    flops = sum(2.0 * mult * n + _pairs(case, cfg, n) for n in lens)
    steps = max(1, -(-sum(lens) // 8192))
    nbytes = es * (steps * read + head) + sum(lens) * cfg.hidden_size * es
    kv = cfg.kv_bytes_per_token(es)
    nbytes += sum(lens) * kv
    if case["kind"] == "replay":
        flops += 2.0 * head * len(lens) * (2 + case["steps"]) + case["steps"] * len(lens) * 2.0 * mult
        nbytes += case["steps"] * (es * (read + head) + sum(lens) * kv)
    elif case["kind"] == "generate":
        rows, more = len(lens) * case["chains"], case["new"] - 1
        flops += 2.0 * head * (rows * more + len(lens)) + more * rows * 2.0 * mult
        nbytes += more * (es * (min(read, rows * mult) + head) + sum(lens) * kv)
    else:
        flops += 2.0 * head * len(lens)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """About four times the distance from ``exact`` that the cases show. A logit is a sum over rounded activations of ten
    and more layers; a routed layer's near ties add to that (a row may take another expert)."""
    if case.get("dtype") == "f32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["kind"] == "replay":
        return {"rel": 3e-2, "max": 0.5}
    if case["model"] in ("mixtral-8x7b", "telurax"):
        return {"rel": 2e-2, "max": 0.1, "differ": 0.005}
    return {"rel": 4e-3, "max": 2e-2, "differ": 0.005}


# ------------------------------------------------------------------------------------------------ plain 64-bit forms
def exact(case, seed):
    """The same values in 64 bits with plain torch: whole sequences at once, no cache."""
    cfg = _config(case)
    toks, targets = _tokens(case, seed, cfg.vocab_size)
    full = toks
    if case["kind"] == "generate":      # the chain that the head leads to, without the last token
        full = [t + [(t[-1] + SHIFT * (k + 1)) % cfg.vocab_size for k in range(case["new"] - 1)] for t in toks]
    n = max(len(t) for t in full)
    ids = torch.zeros(len(full), n, dtype=torch.long, device=DEV)
    for b, t in enumerate(full):        # (padded behind: no mechanism looks ahead)
        ids[b, :len(t)] = torch.tensor(t, device=DEV)
    raw = Weights(case, seed)

    def W(name):
        return raw(name).double()

    if _is_hybrid(case):
        x, norm, head = Hybrid64(config_to_dict(cfg), W).stream(ids)
    else:
        x, norm, head = _transformer64(cfg, W, ids)
    if case["kind"] == "replay":
        steps, lens = case["steps"], [len(t) - case["steps"] for t in toks]
        cut = max(1, lens[-1] // 2) if steps and len(toks) > 1 else lens[-1]
        where = [[(b, p) for b, m in enumerate(lens[:-1] + [cut]) for p in _wants(m)]]
        where += [[(b, m + k) for b, m in enumerate(lens)] for k in range(steps)]
        h = head()
        return [norm(torch.stack([x[b, p] for b, p in step])) @ h.T for step in where]
    last = norm(torch.stack([x[b, len(t) - 1] for b, t in enumerate(full)])) @ head().T
    lp = torch.log_softmax(last, -1)[:, targets]
    if case["kind"] == "score":
        return lp
    return {"tokens": None, "decisions": lp[:, None].expand(-1, case["chains"], -1).contiguous()}


def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, low, cap=0.0, sink=False, talk=None):
    """q [B, H, T, D], k / v [B, G, T, *]; row i sees the keys low[i] .. i. ``cap``: scores are capped; ``sink``: a silent entry
    of score zero in the softmax; ``talk``: the heads' weights are mixed before they meet the values."""
    B, H, T, _ = q.shape
    G = k.shape[1]
    i = torch.arange(T, device=q.device)
    hidden = (i[None, :] > i[:, None]) | (i[None, :] < low[:, None])
    out = torch.empty(B, H, T, v.shape[-1], dtype=q.dtype, device=q.device)
    for b in range(B):
        mixed = 0.0
        for h in range(H):
            g = h // (H // G)
            s = (q[b, h] @ k[b, g].T).mul_(scale)
            s = (cap * torch.tanh(s / cap) if cap else s).masked_fill_(hidden, float("-inf"))
            w = torch.softmax(torch.cat([s, torch.zeros_like(s[:, :1])], 1), -1)[:, :-1] if sink else torch.softmax(s, -1)
            if talk is None:
                out[b, h] = w @ v[b, g]
            else:
                mixed = mixed + talk[:, h, None, None] * w
        if talk is not None:
            for h in range(H):
                out[b, h] = mixed[h] @ v[b, h // (H // G)]
    return out


def _turn(x, f, pairs, mag=1.0):
    """x [B, H, T, D]: the first 2 len(f) coordinates turn by the position (neighbours, or i with i + half)."""
    a = torch.arange(x.shape[2], dtype=torch.float64, device=x.device)[:, None] * torch.tensor(f, dtype=torch.float64, device=x.device)
    c, s, n = mag * torch.cos(a), mag * torch.sin(a), len(f)
    out = x.clone()
    u, v = (x[..., 0:2 * n:2], x[..., 1:2 * n:2]) if pairs else (x[..., :n], x[..., n:2 * n])
    if pairs:
        out[..., 0:2 * n:2], out[..., 1:2 * n:2] = u * c - v * s, v * c + u * s
    else:
        out[..., :n], out[..., n:2 * n] = u * c - v * s, v * c + u * s
    return out


def _heads(x, H):
    return x.view(x.shape[0], x.shape[1], H, -1).transpose(1, 2).contiguous()


def _join(x):
    return x.transpose(1, 2).flatten(2)


def _transformer64(cfg, W, ids):
    emb = "model.embed_tokens.weight"
    x = W(emb)[ids]
    T = ids.shape[1]
    f = [cfg.rope_theta ** (-2.0 * j / cfg.head_dim) for j in range(cfg.head_dim // 2)]
    i = torch.arange(T, device=DEV)
    low = (i - cfg.sliding_window + 1).clamp(min=0) if cfg.sliding_window else torch.zeros_like(i)
    for n in range(cfg.num_layers):
        p = f"model.layers.{n}."
        h = _rms(x, cfg.rms_eps) * W(p + "input_layernorm.weight")
        q, k, v = (h @ W(p + f"self_attn.{c}_proj.weight").T + (W(p + f"self_attn.{c}_proj.bias") if cfg.qkv_bias else 0.0) for c in "qkv")
        q, k, v = _heads(q, cfg.num_heads), _heads(k, cfg.num_kv_heads), _heads(v, cfg.num_kv_heads)
        a = _attend(_turn(q, f, False), _turn(k, f, False), v, cfg.head_dim ** -0.5, low)
        x = x + _join(a) @ W(p + "self_attn.o_proj.weight").T
        h = _rms(x, cfg.rms_eps) * W(p + "post_attention_layernorm.weight")
        if not cfg.is_moe:
            g = torch.nn.functional.silu(h @ W(p + "mlp.gate_proj.weight").T) * (h @ W(p + "mlp.up_proj.weight").T)
            x = x + g @ W(p + "mlp.down_proj.weight").T
            continue
        m = p + "block_sparse_moe."
        w, e = torch.topk(torch.softmax(h @ W(m + "gate.weight").T, -1), cfg.experts_per_tok, -1)
        w = w / w.sum(-1, keepdim=True)
        y = torch.zeros_like(x)
        for j in range(cfg.num_experts):
            share = (w * (e == j)).sum(-1)
            at = share > 0
            z = h[at]
            z = torch.nn.functional.silu(z @ W(m + f"experts.{j}.w1.weight").T) * (z @ W(m + f"experts.{j}.w3.weight").T)
            y[at] += share[at][:, None] * (z @ W(m + f"experts.{j}.w2.weight").T)
        x = x + y
    return x, lambda r: _rms(r, cfg.rms_eps) * W("model.norm.weight"), lambda: W(emb if cfg.tie_embeddings else "lm_head.weight")


class Hybrid64:
    """The hybrid designs' equations on whole padded batches [B, T, d]."""

    def __init__(self, c, W):
        self.c, self.W, self.eps = c, W, c["norm"]["eps"]

    def norm(self, x, name):
        return _rms(x, self.eps) * (self.W(name) + (0.0 if self.c["architecture"] in ("Nidozen", "Gizilorn") else 1.0))

    def stream(self, ids):
        c, W, arch = self.c, self.W, self.c["architecture"]
        e = c.get("embedding") or {}
        x = W("embed")[ids] * e.get("scale", 1.0)
        if e.get("bigram"):
            b = e["bigram"]
            rows = torch.full_like(ids, b["buckets"])
            rows[:, 1:] = (ids[:, :-1] * b["mul_prev"] + ids[:, 1:] * b["mul_cur"]) % b["buckets"]
            x = x + W("bigram")[rows]
        if arch == "Telurax":
            d = c["width"]
            a = torch.arange(ids.shape[1], dtype=torch.float64, device=DEV)[:, None] * \
                torch.tensor([10000.0 ** (-2.0 * j / d) for j in range(d // 2)], dtype=torch.float64, device=DEV)
            x = x + torch.stack([torch.sin(a), torch.cos(a)], -1).flatten(1)
        loop = c.get("loop") or {"start": 0, "stop": 0, "times": 1}
        n = len(c["layers"])
        order = list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], n))
        kv = {}
        if arch == "Gizilorn":          # the residual: parallel streams [S, B, T, d]
            x = self.norm(x, "embed.norm").expand(c["streams"], -1, -1, -1)
        for i in order:
            L, p = c["layers"][i], f"l{i}."
            mix, ff = getattr(self, L["type"]), L.get("mlp")
            if arch == "Gizilorn":
                for q, f in (("1", lambda h: mix(h, p + "mix.", L["mixer"], i, kv)), ("2", lambda h: self.ff(h, p + "mlp.", ff))):
                    y = f(self.norm(torch.tensordot(W(p + f"hc{q}.in"), x, 1), p + "norm" + q))
                    x = torch.tensordot(W(p + f"hc{q}.mix").T, x, 1) + W(p + f"hc{q}.out")[:, None, None, None] * y
            elif arch == "Nidozen":
                x = x + self.norm(mix(x, p + "mix.", L["mixer"], i, kv), p + "norm1")
                x = x + self.norm(self.ff(x, p + "mlp.", ff), p + "norm2")
            elif arch == "Rizurax":
                x = x + mix(self.norm(x, p + "norm1"), p + "mix.", L["mixer"], i, kv) + self.ff(self.norm(x, p + "norm2"), p + "mlp.", ff)
            else:
                x = x + mix(self.norm(x, p + "norm1"), p + "mix.", L["mixer"], i, kv)
                x = x + self.ff(self.norm(x, p + "norm2"), p + "mlp.", ff)
        x = x.sum(0) if arch == "Gizilorn" else x
        return x, lambda r: self.norm(r, "final.norm") * c.get("logit_scale", 1.0), lambda: W("head")

    # -------------------------------------------------------------------------------- feed-forwards
    def ff(self, h, p, mlp):
        W, arch = self.W, self.c["architecture"]
        if mlp["kind"] == "dense":
            up = h @ W(p + "up").T
            if arch == "Gizilorn":
                up, sp = up + W(p + "up.b"), torch.nn.functional.softplus(W(p + "act"))
                act = torch.where(up > 0, sp[0] * up * up, (0.5 + sp[1]) * (torch.expm1(up.clamp(max=0.0)) - up)) + up / 2
                return act @ W(p + "down").T + W(p + "down.b")
            if arch == "Nidozen":
                return torch.relu(up) ** 2 @ W(p + "down").T
            g = h @ W(p + "gate").T
            g = torch.relu(g) if arch == "Telurax" else torch.nn.functional.gelu(g, approximate="tanh")
            return (g * up) @ W(p + "down").T
        r = mlp["router"]
        s = torch.softmax(h @ W(p + "router").T, -1)
        choice, g = s + W(p + "correction"), r["groups"]
        best = choice.view(*choice.shape[:-1], g["count"], -1).amax(-1).topk(g["keep"], -1).indices
        keep = torch.zeros(*choice.shape[:-1], g["count"], dtype=torch.bool, device=h.device).scatter_(-1, best, True)
        choice = choice.masked_fill(~keep.repeat_interleave(choice.shape[-1] // g["count"], -1), float("-inf"))
        e = choice.topk(r["top"], -1).indices
        w = s.gather(-1, e) * r.get("scale", 1.0)
        y = torch.zeros_like(h)
        for j in range(s.shape[-1]):
            share = (w * (e == j)).sum(-1)
            at = share > 0
            if not bool(at.any()):
                continue
            k, t = share[at][:, None], h[at]
            if j >= r["experts"]:
                y[at] += k * t
            else:
                y[at] += k * (torch.relu(t @ W(p + f"e{j}.up").T) ** 2 @ W(p + f"e{j}.down").T)
        return y + torch.relu(h @ W(p + "shared.up").T) ** 2 @ W(p + "shared.down").T

    # -------------------------------------------------------------------------------- mixers
    def attention(self, h, p, m, i, kv):
        W, arch, eps = self.W, self.c["architecture"], self.eps
        H, G, D = m["heads"], m["kv_heads"], m["dim"]
        at = torch.arange(h.shape[1], device=h.device)
        rot, size = m["rot"], (m.get("mask") or {}).get("size", 0)
        f = [rot["base"] ** (-2.0 * j / rot["dims"]) for j in range(rot["dims"] // 2)]
        if arch == "Nidozen":
            q = _turn(_heads(_rms(h @ W(p + "q").T + W(p + "q.b"), eps) * W(p + "q.norm"), H), f, False)
            if "kv_from" not in m:
                k = _turn(_heads(_rms(h @ W(p + "k").T + W(p + "k.b"), eps) * W(p + "k.norm"), G), f, False)
                kv[i] = k, _rms(_heads(h @ W(p + "v").T + W(p + "v.b"), G), eps)
            k, v = kv[m.get("kv_from", i)]
            return _join(_attend(q, k, v, m["scale"], at // size * size)) @ W(p + "o").T + W(p + "o.b")
        if arch == "Gizilorn":
            q, k, v = (_heads(h @ W(p + n).T + W(p + n + ".b"), n_h) for n, n_h in (("q", H), ("k", G), ("v", G)))
            fv = [rot["base"] ** (-2.0 * j / m["vdim"]) for j in range(m["vdim"] // 2)]
            a = _attend(_turn(q, f, False), _turn(k, f, False), _turn(v, fv, False), m["scale"], (at - size + 1).clamp(min=0),
                        m["softcap"], True, W(p + "talk"))
            return _join(_turn(a, [-x for x in fv], False)) @ W(p + "o").T
        sc, mag = rot["scaling"], 0.1 * math.log(rot["scaling"]["factor"]) + 1.0

        def pair_at(turns):
            return rot["dims"] * math.log(sc["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
        lo, hi = max(math.floor(pair_at(sc["fast"])), 0), min(math.ceil(pair_at(sc["slow"])), rot["dims"] - 1)
        ramp = [min(max((j - lo) / max(hi - lo, 0.001), 0.0), 1.0) for j in range(len(f))]
        f = [x / sc["factor"] * r + x * (1 - r) for x, r in zip(f, ramp)]
        q, k = _turn(_heads(h @ W(p + "q").T, 2 * H), f, True, mag), _turn(_heads(h @ W(p + "k").T, 2 * G), f, True, mag)
        v, low = _heads(h @ W(p + "v").T, G), torch.zeros_like(at)
        one, two = (_attend(q[:, j::2].contiguous(), k[:, j::2].contiguous(), v, m["scale"], low) for j in (0, 1))
        lam = torch.exp((W(p + "lq1") * W(p + "lk1")).sum()) - torch.exp((W(p + "lq2") * W(p + "lk2")).sum()) + m["diff"]
        return _join(_rms(one - lam * two, eps) * (1.0 - m["diff"])) @ W(p + "o").T

    def latent_attention(self, h, p, m, i, kv):
        W, H, D, R, rd = self.W, m["heads"], m["dim"], m["kv_rank"], m.get("rot_dim", 0)
        q = _heads(h @ W(p + "q").T, H)
        f = [m["rot"]["base"] ** (-2.0 * j / rd) for j in range(rd // 2)] if rd else []
        if "kv_from" not in m:
            down = h @ W(p + "dkv").T
            turned = _turn(down[:, None, :, R:], f, True) if rd else None       # one key part for all heads
            kv[i] = _rms(down[..., :R], self.eps) * W(p + "dkv.norm"), turned
        c, turned = kv[m.get("kv_from", i)]
        k, v = _heads(c @ W(p + "uk").T, H), _heads(c @ W(p + "uv").T, H)
        if rd:
            q = torch.cat([q[..., :D], _turn(q[..., D:], f, True)], -1)
            k = torch.cat([k, turned.expand(-1, H, -1, -1)], -1)
        at, size = torch.arange(h.shape[1], device=h.device), (m.get("mask") or {}).get("size", 0) or h.shape[1]
        a = _attend(q, k, v, m["scale"], (at - size + 1).clamp(min=0))
        g = torch.sigmoid(h @ W(p + "g").T)
        a = _join(a) * g if rd else _join(a * g.transpose(1, 2)[..., None])
        return a @ W(p + "o").T

    def mingru(self, h, p, m, i, kv):
        W = self.W
        z = torch.sigmoid(h @ W(p + "z").T + W(p + "z.b"))
        u = h @ W(p + "x").T + W(p + "x.b")
        u = torch.where(u >= 0, u + 0.5, torch.sigmoid(u))
        S, rows = torch.zeros_like(z[:, 0]), []
        for t in range(h.shape[1]):
            S = (1 - z[:, t]) * S + z[:, t] * u[:, t]
            rows.append(S)
        return (torch.stack(rows, 1) * torch.nn.functional.silu(h @ W(p + "g").T)) @ W(p + "o").T

    def gla(self, h, p, m, i, kv):
        W, H = self.W, m["heads"]
        q, k, v = (_heads(h @ W(p + n).T, H) for n in "qkv")
        a = _heads(torch.sigmoid((h @ W(p + "a1").T) @ W(p + "a2").T + W(p + "a2.b")) ** (1.0 / m["tau"]), H)
        S, rows = 0.0, []
        for t in range(h.shape[1]):
            S = a[:, :, t, :, None] * S + k[:, :, t, :, None] * v[:, :, t, None, :]
            rows.append((q[:, :, t, None, :] @ S)[:, :, 0] * m["dim"] ** -0.5)
        o = _rms(torch.stack(rows, 2), self.eps) * W(p + "norm")
        return (_join(o) * torch.nn.functional.silu(h @ W(p + "g").T)) @ W(p + "o").T

    def mlstm(self, h, p, m, i, kv):
        W, H, cap = self.W, m["heads"], m["gate_cap"]
        q, k, v = (_heads(h @ W(p + n).T, H) for n in "qkv")
        q = q * m["dim"] ** -0.5
        li, lf = (cap * torch.tanh((h @ W(p + n).T + W(p + n + ".b")) / cap) for n in "if")
        lf = torch.nn.functional.logsigmoid(lf)
        v = torch.cat([v, torch.ones_like(v[..., :1])], -1)      # (the normaliser is a value column of ones)
        S, mx, rows = 0.0, torch.zeros_like(li[:, 0]), []
        for t in range(h.shape[1]):
            new = torch.maximum(lf[:, t] + mx, li[:, t])
            S = torch.exp(lf[:, t] + mx - new)[..., None, None] * S + torch.exp(li[:, t] - new)[..., None, None] * \
                k[:, :, t, :, None] * v[:, :, t, None, :]
            mx = new
            o = (q[:, :, t, None, :] @ S)[:, :, 0]
            den = torch.maximum(o[..., -1].abs(), torch.exp(-mx)) + 1e-6
            rows.append(_rms(o[..., :-1] / den[..., None], self.eps))
        o = _join(torch.stack(rows, 2)) * W(p + "norm")
        return (o * torch.sigmoid(h @ W(p + "g").T)) @ W(p + "o").T

    def delta(self, h, p, m, i, kv):
        W, H, G = self.W, m["heads"], m["kv_heads"]
        silu, sp = torch.nn.functional.silu, torch.nn.functional.softplus

        def conv(n):
            u, w = h @ W(p + n).T, W(p + n + ".conv")
            taps = w.shape[1]
            u = torch.nn.functional.pad(u, (0, 0, taps - 1, 0))
            return silu(sum(w[:, j] * u[:, j:j + h.shape[1]] for j in range(taps)))
        q, k = (_heads(conv(n), G) for n in "qk")
        v = _heads(conv("v"), H)
        q, k = (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        q, k = (q * m["dim"] ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
        beta = torch.sigmoid(h @ W(p + "b").T)
        g = torch.exp(-torch.exp(W(p + "A_log")) * sp(h @ W(p + "a").T + W(p + "dt_bias")))
        S = torch.zeros(h.shape[0], H, m["dim"], m["vdim"], dtype=torch.float64, device=h.device)
        rows = []
        for t in range(h.shape[1]):
            S = S * g[:, t, :, None, None]
            u = beta[:, t, :, None] * (v[:, :, t] - (k[:, :, t, None, :] @ S)[:, :, 0])
            S = S + k[:, :, t, :, None] * u[:, :, None, :]
            rows.append((q[:, :, t, None, :] @ S)[:, :, 0])
        o = _rms(torch.stack(rows, 2), self.eps) * W(p + "norm") * _heads(silu(h @ W(p + "g").T), H)
        return _join(o) @ W(p + "o").T
