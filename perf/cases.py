"""The work that this engine is used for, as cases that can be timed and checked.

A case is one step of a serving loop (``ModelRunner.step``, the call under ``LLMEngine.step`` and the
trace replayer), a short replay of whole requests, or the choice of the next tokens (``Sampler``):

* ``step``: ``requests`` requests that hold up to ``keys`` tokens each and get one more, and/or one
  request's portion of ``tokens`` prompt tokens behind ``cached`` tokens that it holds already. With
  ``tokens`` 0 it is a decode step, with ``requests`` 0 a prefill step, with both a mixed one. The
  output is the logits that the step was asked for: one row for each request.
* ``replay``: ``requests`` new requests with prompts of ``tokens`` tokens, then ``steps`` steps of one
  given token for each: pages are taken and given back inside. Used where a step changes a state that
  is not addressed by position (a recurrence), and for float32. The output is every step's logits.
* ``sample``: tokens for ``rows`` rows of logits.

The model is what a server holds for as long as it runs: its weights do not depend on the seed and it
is built once for all states that use it. The requests and their tokens are the state, made from the seed.
Model sizes are the benchmark's (``bench.py``: ``--shape``, ``--design fuvavik``).

Routed experts are left out: two correct implementations in bfloat16 send a few tokens in a hundred to
other experts, and the outputs then differ by more than any tolerance that would still find a mistake.
"""

from __future__ import annotations

import gc
import itertools
import math
import zlib
from types import SimpleNamespace

import torch

from clockwork_amd.config.engine import EngineConfig
from clockwork_amd.engine.batch import StepEntry
from clockwork_amd.engine.model_runner import ModelRunner
from clockwork_amd.engine.sequence import SamplingParams, Sequence
from clockwork_amd.sampling.sampler import Sampler

BLOCK = 16       # tokens a page
BUDGET = 2048    # tokens a step may run
MAX_REQUESTS = 64


def _qwen2(layers, hidden, heads, kv_heads, inner, vocab=151936, tied=True):
    return dict(model_type="qwen2", architectures=["Qwen2ForCausalLM"], vocab_size=vocab, hidden_size=hidden,
                num_hidden_layers=layers, num_attention_heads=heads, num_key_value_heads=kv_heads,
                intermediate_size=inner, rms_norm_eps=1e-6, rope_theta=1000000.0, tie_word_embeddings=tied,
                hidden_act="silu", use_sliding_window=False, max_position_embeddings=32768)


def _fuvavik(width, heads, dim, r_heads, r_vdim, rank, inner):
    left = {"heads": heads, "kv_heads": 2, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "mask": {"size": 1024}}
    right = {"heads": r_heads, "dim": 64, "vdim": r_vdim, "tau": 16.0, "rank": rank}
    layer = {"type": "parallel", "mixer": {"left": left, "right": right}, "mlp": {"kind": "dense", "ff": inner}}
    return {"architecture": "Fuvavik", "vocab": 32768, "width": width, "max_positions": 4096, "embedding": {"scale": 1.0},
            "norm": {"eps": 1e-6}, "logit_softcap": 30.0, "layers": [layer] * 4}


MODELS = {
    "qwen2.5-0.5b": _qwen2(24, 896, 14, 2, 4864),
    "qwen2.5-1.5b": _qwen2(28, 1536, 12, 2, 8960),
    "qwen2.5-7b": _qwen2(28, 3584, 28, 4, 18944, vocab=152064, tied=False),
    "fuvavik-s": _fuvavik(896, 14, 64, 14, 64, 16, 4864),
    "fuvavik-m": _fuvavik(1536, 12, 128, 12, 128, 32, 8960),
}


# ------------------------------------------------------------------------------- the cases
def _step(model, requests=0, keys=0, tokens=0, cached=0):
    return {"kind": "step", "model": model, "dtype": "bfloat16", "requests": requests, "keys": keys, "tokens": tokens,
            "cached": cached}


def _replay(model, dtype, requests, tokens, steps):
    return {"kind": "replay", "model": model, "dtype": dtype, "requests": requests, "tokens": tokens, "steps": steps}


def listed():
    small, main, large = "qwen2.5-0.5b", "qwen2.5-1.5b", "qwen2.5-7b"
    return [
        # one user, a short conversation, the smallest model: launches and latency
        {"name": "decode_1x120_0.5b", **_step(small, requests=1, keys=120)},
        # the recorded benchmark's batch, requests of unequal length
        {"name": "decode_8x2048_1.5b", **_step(main, requests=8, keys=2048)},
        # a full server
        {"name": "decode_64x2048_1.5b", **_step(main, requests=64, keys=2048)},
        # a larger model: the step is its weights
        {"name": "decode_8x1000_7b", **_step(large, requests=8, keys=1000)},
        # a portion of a long prompt at the token budget (the recorded prefill)
        {"name": "prefill_2048_1.5b", **_step(main, tokens=2048)},
        # a chat turn of its own, of an odd length
        {"name": "prefill_137_1.5b", **_step(main, tokens=137)},
        # the last portion of a long document
        {"name": "portion_1000_behind_7000_1.5b", **_step(main, tokens=1000, cached=7000)},
        # a prompt that arrives while others decode
        {"name": "mixed_15x1500_and_300_1.5b", **_step(main, requests=15, keys=1500, tokens=300)},
        # the tokens of a full batch whose requests ask for different ways to choose
        {"name": "sample_64", "kind": "sample", "rows": 64, "vocab": 151936, "options": "mixed"},
        # float32, the dtype that results are checked in
        {"name": "replay_float32_0.5b", **_replay(small, "float32", 1, 300, 4)},
        # another architecture (windowed attention with mixed heads beside a recurrence): a prompt, and a few requests to their end
        {"name": "prefill_2048_fuvavik", **_replay("fuvavik-m", "bfloat16", 1, 2048, 0)},
        {"name": "replay_8x200_fuvavik", **_replay("fuvavik-m", "bfloat16", 8, 200, 16)},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choices(["decode", "prefill", "mixed", "sample", "float32", "fuvavik"], [5, 4, 2, 1, 1, 1])[0]
    model = rng.choices(["qwen2.5-0.5b", "qwen2.5-1.5b", "qwen2.5-7b"], [2, 4, 1])[0]
    if kind == "decode":
        requests = log_int(1, 8 if model == "qwen2.5-7b" else MAX_REQUESTS)
        longest = 2048 if requests > 4 else 12000  # the cached tokens of a step stay within a full server's
        return _step(model, requests=requests, keys=log_int(16, longest))
    if model == "qwen2.5-7b":
        model = "qwen2.5-1.5b"
    if kind == "prefill":
        cached = 0 if rng.random() < 0.6 else log_int(64, 8000)
        return _step(model, tokens=log_int(16, BUDGET if cached < 2000 else 1000), cached=cached)
    if kind == "mixed":
        return _step(model, requests=log_int(1, MAX_REQUESTS - 1), keys=log_int(64, 2048), tokens=log_int(16, 600),
                     cached=0 if rng.random() < 0.6 else log_int(64, 2048))
    if kind == "sample":
        return {"kind": "sample", "rows": log_int(1, 64), "vocab": rng.choice([151936, 152064, 32768]),
                "options": rng.choice(["greedy", "temperature", "top_k", "top_p", "mixed"])}
    if kind == "float32":
        return _replay("qwen2.5-0.5b", "float32", 1, log_int(16, 400), rng.randint(0, 4))
    requests = log_int(1, 8)
    return _replay(rng.choice(["fuvavik-s", "fuvavik-m"]), "bfloat16", requests, log_int(16, BUDGET // requests),
                   rng.randint(0, 16))


# ------------------------------------------------------------------------------- the models
def _shapes(config):
    """Checkpoint tensor name -> shape."""
    s = {}
    if "model_type" in config:
        h, n, kv, inner = (config[k] for k in ("hidden_size", "num_attention_heads", "num_key_value_heads", "intermediate_size"))
        d = h // n
        s["model.embed_tokens.weight"] = (config["vocab_size"], h)
        for i in range(config["num_hidden_layers"]):
            p = f"model.layers.{i}."
            s[p + "input_layernorm.weight"] = s[p + "post_attention_layernorm.weight"] = (h,)
            for name, rows in (("q", n * d), ("k", kv * d), ("v", kv * d)):
                s[p + f"self_attn.{name}_proj.weight"], s[p + f"self_attn.{name}_proj.bias"] = (rows, h), (rows,)
            s[p + "self_attn.o_proj.weight"] = (h, n * d)
            s[p + "mlp.gate_proj.weight"] = s[p + "mlp.up_proj.weight"] = (inner, h)
            s[p + "mlp.down_proj.weight"] = (h, inner)
        s["model.norm.weight"] = (h,)
        if not config["tie_word_embeddings"]:
            s["lm_head.weight"] = (config["vocab_size"], h)
        return s
    w = config["width"]
    s["embed"], s["pos"] = (config["vocab"], w), (config["max_positions"], w)
    for i, layer in enumerate(config["layers"]):
        m, r, ff = layer["mixer"]["left"], layer["mixer"]["right"], layer["mlp"]["ff"]
        p, left, right = f"l{i}.", f"l{i}.mix.left.", f"l{i}.mix.right."
        q, k, v = m["heads"] * m["dim"], m["kv_heads"] * m["dim"], m["kv_heads"] * m["vdim"]
        rq, rv = r["heads"] * r["dim"], r["heads"] * r["vdim"]
        s.update({p + "norm1": (w,), p + "norm1.b": (w,), left + "q": (q, w), left + "k": (k, w), left + "v": (v, w),
                  left + "q.norm": (q,), left + "k.norm": (k,), left + "r1": (m["heads"],), left + "r2": (m["heads"],),
                  left + "sink": (m["heads"],), left + "talk": (m["heads"], m["heads"]), left + "o": (w, m["heads"] * m["vdim"]),
                  right + "q": (rq, w), right + "k": (rq, w), right + "v": (rv, w), right + "g": (rv, w),
                  right + "a1": (r["rank"], w), right + "a2": (rq, r["rank"]), right + "a2.b": (rq,),
                  right + "norm": (r["vdim"],), right + "o": (w, rv), left + "out": (w,), right + "out": (w,),
                  p + "mlp.gate": (ff, w), p + "mlp.up": (ff, w), p + "mlp.down": (w, ff),
                  p + "rg1": (w, w), p + "rg2": (w, w), p + "rg1.b": (w,), p + "rg2.b": (w,)})
    s["final.norm"] = s["final.norm.b"] = (w,)
    return s


class Weights:
    """A checkpoint whose tensors are drawn when they are read: the names, shapes and dtypes under
    ``entries``, a tensor's values from its name alone."""

    def __init__(self, config):
        self.entries = {name: SimpleNamespace(shape=shape, dtype="BF16") for name, shape in _shapes(config).items()}
        self.branches = 2 * config["num_hidden_layers"] if "model_type" in config else 0

    def read(self, name):
        shape = self.entries[name].shape
        gen = torch.Generator(device="cuda").manual_seed(zlib.crc32(name.encode()))
        t = torch.empty(shape, device="cuda")
        last = name.rsplit(".", 1)[-1]
        if "norm" in name and not name.endswith((".b", "bias")) or last == "out":
            t.uniform_(0.9, 1.1, generator=gen)
        elif last in ("r1", "r2"):
            t.uniform_(0.0, 1.0, generator=gen)
        elif last == "talk":
            t.normal_(0.0, 0.2, generator=gen).add_(torch.eye(*shape, device="cuda"))
        else:
            std = 1.0 if last == "sink" or name.endswith("a2.b") else 0.5 if last == "a2" or name.endswith(("rg1.b", "rg2.b")) else 0.02
            if self.branches and name.endswith("_proj.weight"):
                # Scores that spread over a few keys, and branches that together add as much to the stream as it
                # began with, as in trained models. With one spread for every matrix the first branches drown the
                # embedding and bfloat16's roundings grow, through 28 layers, to five hundredths of the logits.
                fan_in = math.sqrt(shape[1])
                std = (0.17 / (fan_in * math.sqrt(self.branches)) if name.endswith(("o_proj.weight", "down_proj.weight"))
                       else 1.6 / fan_in if name.endswith(("q_proj.weight", "k_proj.weight")) else 0.8 / fan_in)
            elif "embed" in name:
                std = 0.05 if self.branches else 0.02
            t.normal_(0.0, std, generator=gen)
        return t.to(torch.bfloat16)


_held: dict = {}              # the model that is being served
_ids = itertools.count()


def _longest(case):
    return max(case.get("keys", 0), case.get("cached", 0) + case["tokens"], case["tokens"] + case.get("steps", 0)) + 1


def _runner(case):
    """The runner that serves the case's model; another one that was held is let go first."""
    context = 4096 if _longest(case) <= 4096 else 16384
    key = (case["model"], case["dtype"], context)
    if key not in _held:
        _held.clear()
        gc.collect()
        torch.cuda.empty_cache()
        cfg = EngineConfig.defaults(case["model"], dtype=case["dtype"], max_model_len=context, block_size=BLOCK, num_blocks=40960,
                                    watermark=0.0, max_num_seqs=MAX_REQUESTS, max_num_batched_tokens=BUDGET)
        config = MODELS[case["model"]]
        _held[key] = ModelRunner(cfg, weight_source=Weights(config), config_dict=dict(config))
    return _held[key]


# ------------------------------------------------------------------------------- preparing and running
class State:
    """One case's requests: what they hold, and the entries of the step that is timed."""

    def __init__(self, case, runner):
        self.case, self.runner, self.ids, self.entries = case, runner, [], []

    def __del__(self):
        for seq_id in self.ids:
            self.runner.release(seq_id)


def _lengths(case):
    """Tokens that each decoding request holds: from half of ``keys`` to all of them."""
    n, keys = case["requests"], case["keys"]
    return [keys - (i * (keys // 2)) // n for i in range(n)]


def _tokens(case, seed):
    """A list of token ids for each request of the case: uniform, as the benchmark's."""
    config = MODELS[case["model"]]
    vocab = config.get("vocab_size", config.get("vocab"))
    gen = torch.Generator().manual_seed(seed)
    if case["kind"] == "step":
        counts = [n + 1 for n in _lengths(case)] + ([case["cached"] + case["tokens"]] if case["tokens"] else [])
    else:
        counts = [case["tokens"] + case["steps"]] * case["requests"]
    return [torch.randint(0, vocab, (n,), generator=gen).tolist() for n in counts]


def _sampling(case, row):
    options = {"greedy": dict(temperature=0.0), "temperature": dict(temperature=0.8),
               "top_k": dict(temperature=0.9, top_k=50), "top_p": dict(temperature=0.7, top_p=0.9)}
    name = case["options"] if case["options"] != "mixed" else list(options)[row % 4]
    return SamplingParams(seed=row, **options[name])


def prepare(case, seed):
    if case["kind"] == "sample":
        gen = torch.Generator(device="cuda").manual_seed(seed)
        # a spread that leaves some hundred likely tokens, as a model's own logits have
        logits = 3.0 * torch.randn(case["rows"], case["vocab"], generator=gen, device="cuda")
        requests = [Sequence(str(i), [1], _sampling(case, i), arrival_time=float(i)) for i in range(case["rows"])]
        return SimpleNamespace(case=case, logits=logits, requests=requests, sampler=Sampler(logits.device))
    state = State(case, _runner(case))
    state.tokens = _tokens(case, seed)
    if case["kind"] == "replay":
        return state
    runner = state.runner
    decoding = case["requests"]
    for i, tokens in enumerate(state.tokens):
        seq_id = f"r{next(_ids)}"
        start = len(tokens) - 1 if i < decoding else case["cached"]
        runner.reserve(seq_id, 0, len(tokens))
        state.ids.append(seq_id)
        for at in range(0, start, BUDGET):
            runner.step([StepEntry(seq_id, at, tokens[at:min(at + BUDGET, start)])])
        state.entries.append(StepEntry(seq_id, start, tokens[start:], [len(tokens) - start - 1]))
    return state


def run(state):
    case = state.case
    if case["kind"] == "sample":
        return state.sampler.launch(state.logits, state.requests)
    runner = state.runner
    if case["kind"] == "step":
        return runner.step(state.entries)
    n = case["tokens"]
    ids = [f"p{next(_ids)}" for _ in state.tokens]
    logits = []
    for at, count in [(0, n)] + [(n + i, 1) for i in range(case["steps"])]:
        for seq_id in ids:
            runner.reserve(seq_id, at, count)
        entries = [StepEntry(seq_id, at, t[at:at + count], [count - 1]) for seq_id, t in zip(ids, state.tokens)]
        logits.append(runner.step(entries).clone())  # the next step may write over them
    for seq_id in ids:
        runner.release(seq_id)
    return logits


# ------------------------------------------------------------------------------- what a pass cannot do without
def _counts(case):
    """(new tokens, keys read by all of them, keys cached before, rows of logits) over the case's steps."""
    if case["kind"] == "step":
        lens, n, cached = _lengths(case), case["tokens"], case["cached"]
        return (len(lens) + n, sum(k + 1 for k in lens) + n * cached + n * (n + 1) // 2, sum(lens) + cached, len(lens) + (n > 0))
    n, steps, r = case["tokens"], case["steps"], case["requests"]
    return r * (n + steps), r * (n * (n + 1) // 2 + sum(n + i + 1 for i in range(steps))), r * sum(n + i for i in range(steps)), r * (1 + steps)


def work(case):
    if case["kind"] == "sample":
        values = case["rows"] * case["vocab"]
        return {"bytes": 4 * values + 4 * case["rows"], "flops": 2 * values}
    config = MODELS[case["model"]]
    shapes = _shapes(config)
    size = 4 if case["dtype"] == "float32" else 2
    qwen = "model_type" in config
    vocab, width = shapes["model.embed_tokens.weight" if qwen else "embed"]
    head = vocab * width
    matrices = sum(math.prod(s) for name, s in shapes.items() if len(s) == 2 and "embed" not in name and name not in ("pos", "lm_head.weight"))
    new, seen, before, rows = _counts(case)
    passes = 1 + case.get("steps", 0)
    if qwen:
        layers, heads = config["num_hidden_layers"], config["num_attention_heads"]
        dim, kv = width // heads, config["num_key_value_heads"]
        state_flops = 0
    else:
        left, right = config["layers"][0]["mixer"]["left"], config["layers"][0]["mixer"]["right"]
        layers, heads, dim, kv = len(config["layers"]), left["heads"], left["dim"], left["kv_heads"]
        window = left["mask"]["size"]
        if case["tokens"] > window:  # a token sees the window's keys at most
            seen = case["requests"] * (window * (window + 1) // 2 + (case["tokens"] - window) * window + case["steps"] * window)
        before = min(before, case["requests"] * case["steps"] * window)
        state_flops = new * layers * right["heads"] * right["dim"] * (5 * right["vdim"]) + 2 * seen * layers * heads * heads
    attention = 4 * seen * layers * heads * dim
    bytes_ = passes * (matrices + head) * size + 2 * (before + new) * layers * kv * dim * size + new * width * size + 4 * rows * vocab
    return {"bytes": bytes_, "flops": 2 * new * matrices + 2 * rows * head + attention + state_flops}


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"
    # measured against 64 bits: float32 1e-6; bfloat16 0.007 to 0.015, so that two such lie up to 0.02 apart
    return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 0.025}


# ------------------------------------------------------------------------------- the same in 64 bits
def _rms(x, weight, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight


def _attend(q, k, v, scale):
    """q, k, v [T, heads, dim], causal; a few queries at a time."""
    q, k, v = (t.transpose(0, 1).contiguous() for t in (q, k, v))
    out = torch.empty_like(q)
    key = torch.arange(k.shape[1], device=q.device)
    for at in range(0, q.shape[1], 1024):
        part = q[:, at:at + 1024]
        scores = part @ k.transpose(1, 2).contiguous() * scale
        scores.masked_fill_(key[None, :] > key[at:at + part.shape[1], None], float("-inf"))
        out[:, at:at + 1024] = torch.softmax(scores, -1) @ v
    return out.transpose(0, 1).reshape(q.shape[1], -1)


def _qwen2_exact(config, tokens, rows):
    """Logits at ``rows`` of the requests' tokens laid one after the other."""
    weights = Weights(config)

    def w(name):
        return weights.read(name).double()

    heads, kv, eps = config["num_attention_heads"], config["num_key_value_heads"], config["rms_norm_eps"]
    dim = config["hidden_size"] // heads
    embed = weights.read("model.embed_tokens.weight")
    x = embed[torch.tensor(list(itertools.chain(*tokens)), device="cuda")].double()
    # the model's angles are float32 products of a position and a frequency; all else is in 64 bits
    freq = 1.0 / (config["rope_theta"] ** (torch.arange(0, dim, 2, dtype=torch.float32) / dim))
    angle = torch.cat([torch.arange(len(t), dtype=torch.float32) for t in tokens])[:, None] * freq
    cos, sin = (f(angle.double()).cuda()[:, None, :] for f in (torch.cos, torch.sin))

    def rotate(t):
        a, b = t.chunk(2, -1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    for i in range(config["num_hidden_layers"]):
        p = f"model.layers.{i}."
        n = _rms(x, w(p + "input_layernorm.weight"), eps)
        q, k, v = ((n @ w(p + f"self_attn.{c}_proj.weight").t() + w(p + f"self_attn.{c}_proj.bias")).view(len(n), -1, dim) for c in "qkv")
        q, k = rotate(q), rotate(k)
        k, v = (t.repeat_interleave(heads // kv, 1) for t in (k, v))
        out, at = torch.empty_like(n), 0
        for t in tokens:
            to = at + len(t)
            out[at:to] = _attend(q[at:to], k[at:to], v[at:to], dim ** -0.5)
            at = to
        x = x + out @ w(p + "self_attn.o_proj.weight").t()
        if i == config["num_hidden_layers"] - 1:
            x = x[rows]
        n = _rms(x, w(p + "post_attention_layernorm.weight"), eps)
        gate, up, down = (w(p + f"mlp.{c}_proj.weight") for c in ("gate", "up", "down"))
        for at in range(0, len(n), 16384):
            part = n[at:at + 16384]
            x[at:at + 16384] += (torch.nn.functional.silu(part @ gate.t()) * (part @ up.t())) @ down.t()
    head = embed if config["tie_word_embeddings"] else weights.read("lm_head.weight")
    return _rms(x, w("model.norm.weight"), eps) @ head.double().t()


def _fuvavik_attention(n, w, p, m, eps):
    """n [T, width]; windowed, with a falling score by distance, a sink and weights mixed across heads."""
    count, heads, kv = n.shape[0], m["heads"], m["kv_heads"]
    q = _rms(n @ w(p + "q").t(), w(p + "q.norm"), eps).view(count, heads, -1).transpose(0, 1).contiguous()
    k = _rms(n @ w(p + "k").t(), w(p + "k.norm"), eps).view(count, kv, -1).repeat_interleave(heads // kv, 1).permute(1, 2, 0).contiguous()
    v = (n @ w(p + "v").t()).view(count, kv, -1).repeat_interleave(heads // kv, 1).transpose(0, 1).contiguous()
    at = torch.arange(count, device=n.device)
    distance = at[:, None] - at[None, :]
    hidden = (distance < 0) | (distance >= m["mask"]["size"])
    distance = distance.clamp(min=0).double()
    scores = torch.empty(heads, count, count + 1, dtype=torch.float64, device=n.device)
    r1, r2, sink = w(p + "r1"), w(p + "r2"), w(p + "sink")
    for a in range(heads):
        scores[a, :, :count] = (q[a] @ k[a] * m["scale"] - r1[a] * torch.log1p(r2[a] * distance)).masked_fill(hidden, float("-inf"))
        scores[a, :, count] = sink[a]
    weights = torch.softmax(scores, -1)[:, :, :count]
    mixed = (w(p + "talk") @ weights.reshape(heads, -1)).view(heads, count, count)
    return (mixed @ v).transpose(0, 1).reshape(count, -1) @ w(p + "o").t()


def _fuvavik_recurrence(n, w, p, m, eps):
    """n [requests, T, width]: a matrix state a head with a decay a key channel and token."""
    r, count, heads, dim = n.shape[0], n.shape[1], m["heads"], m["dim"]
    q = (n @ w(p + "q").t()).view(r, count, heads, dim) * dim ** -0.5
    k = (n @ w(p + "k").t()).view(r, count, heads, dim)
    v = (n @ w(p + "v").t()).view(r, count, heads, -1)
    decay = (torch.sigmoid(n @ w(p + "a1").t() @ w(p + "a2").t() + w(p + "a2.b")) ** (1.0 / m["tau"])).view(r, count, heads, dim)
    state = torch.zeros(r, heads, dim, v.shape[-1], dtype=torch.float64, device=n.device)
    out = torch.empty_like(v)
    for t in range(count):
        state = decay[:, t, :, :, None] * state + k[:, t, :, :, None] * v[:, t, :, None, :]
        out[:, t] = (q[:, t, :, :, None] * state).sum(-2)
    out = _rms(out, w(p + "norm"), eps).reshape(r, count, -1)
    return (out * torch.nn.functional.silu(n @ w(p + "g").t())) @ w(p + "o").t()


def _fuvavik_exact(config, tokens, first):
    """Logits of every token from the ``first`` on, [requests, tokens, vocab]."""
    weights, eps = Weights(config), config["norm"]["eps"]

    def w(name):
        return weights.read(name).double()

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], w(name), w(name + ".b"), eps)

    ids = torch.tensor(tokens, device="cuda")
    x = w("embed")[ids] * config["embedding"]["scale"] + w("pos")[:ids.shape[1]]
    for i, layer in enumerate(config["layers"]):
        p, left, right = f"l{i}.", f"l{i}.mix.left.", f"l{i}.mix.right."
        n = norm(x, p + "norm1")
        a = torch.stack([_fuvavik_attention(row, w, left, layer["mixer"]["left"], eps) for row in n])
        b = _fuvavik_recurrence(n, w, right, layer["mixer"]["right"], eps)
        mixed = 0.5 * (_rms(a, w(left + "out"), eps) + _rms(b, w(right + "out"), eps))
        inner = torch.nn.functional.gelu(n @ w(p + "mlp.gate").t(), approximate="tanh") * (n @ w(p + "mlp.up").t())
        x = x + torch.sigmoid(n @ w(p + "rg1").t() + w(p + "rg1.b")) * mixed
        x = x + torch.sigmoid(n @ w(p + "rg2").t() + w(p + "rg2.b")) * (inner @ w(p + "mlp.down").t())
    cap = config["logit_softcap"]
    return cap * torch.tanh(norm(x[:, first:], "final.norm") @ w("embed").t() / cap)


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "sample":
        return None  # whole numbers
    config, tokens = MODELS[case["model"]], _tokens(case, seed)
    if case["kind"] == "step":
        if sum(work(_step(case["model"], tokens=len(t)))["flops"] for t in tokens) > 5e14:
            return None  # too long in 64 bits
        ends = list(itertools.accumulate(map(len, tokens)))
        return _qwen2_exact(config, tokens, [e - 1 for e in ends])
    n, steps, r = case["tokens"], case["steps"], case["requests"]
    if "model_type" in config:
        total = n + steps
        logits = _qwen2_exact(config, tokens, [i * total + j for i in range(r) for j in range(n - 1, total)])
        logits = logits.view(r, steps + 1, -1)
    else:
        logits = _fuvavik_exact(config, tokens, n - 1)
    return [logits[:, i].contiguous() for i in range(steps + 1)]
