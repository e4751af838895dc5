"""The work that is timed: requests of a generation service, from the first prompt token to the last decoded one.

A case is one batch of requests on one model of random weights (the layer sizes are the presets'). Its pass takes
slots, runs the prompts in one step (captured where they are short, as the engine does), decodes ``steps`` tokens per
sequence through a captured step, and gives the slots back. The tokens that are fed are given (teacher forcing, as a
scoring program feeds them): logits can then be compared step by step, which tokens chosen near a tie cannot. Every
decoding step still chooses greedily, as the generation loop does; the chosen token's logit is returned.

``work`` counts what a pass cannot do without; ``exact`` is each model in plain torch and 64 bits, whole sequences
at once, with no cache and none of the package's arithmetic (it takes the weights from the package's seeded
initialiser, since they are inputs).
"""

from __future__ import annotations

import math

import torch

from dryft_amd import Engine
from dryft_amd.cache.spec import KVNeed, PAGE_TOKENS, pages_for
from dryft_amd.engine.engine import PROMPT_GRAPH_ROWS, pick_bucket
from dryft_amd.engine.graph import DecodeGraph, PromptGraph
from dryft_amd.engine.model import DecoderModel
from dryft_amd.engine.step import SeqStep
from dryft_amd.models import load_preset, resolve_architecture
from dryft_amd.sampling import Sampler
from dryft_amd.weights.random_init import random_tensors

SHORT_STEP = 256               # prompts of at most so many tokens in all start in a captured step (the engine's default)
# A model is a preset and how many of its layers run (0: all of them). Qwen3-4B runs a third of its layers: each layer
# does what it does in the whole model, and with all 36 two equally good bfloat16 implementations are 3 to 4 % apart on
# random weights, too far to tell a mistake from rounding (12 layers: 2 %; Qwen3-0.6B, all 28: 1.4 %). Piralix likewise
# (18 layer runs: 5 %). Designs whose router ranks sigmoid scores or ranks within groups flip experts on random weights
# by rounding alone (4 to 13 % of the logits' norm), so their kernels are met here in their relatives: experts by table
# and by softmax, several copies of a stream, windows, chunks, latents.
QWEN3 = (("qwen3-0.6b", 0), ("qwen3-4b", 12))
DESIGNS = (("piralix-w2048", 6), ("barilix-w2048", 0), ("fubinex-w2048", 0), ("kaditar-w2048", 0))


def _case(name, model, layers, batch, shortest, longest, steps, dtype="bfloat16"):
    """``steps`` tokens are decoded after prompts of ``shortest`` to ``longest`` tokens."""
    case = dict(model=model, layers=layers, dtype=dtype, batch=batch, shortest=shortest, longest=longest, steps=steps)
    return dict(name=name, **case) if name else case


# ------------------------------------------------------------------------------------------ the cases
def listed():
    return [
        # one user's first token: a question of a sentence or two, where launches and small products are the time
        _case("first token", "qwen3-4b", 12, 1, 77, 77, 0),
        # the headline prompt: 2,048 tokens, prefilled alone
        _case("prompt 2048", "qwen3-4b", 12, 1, 2048, 2048, 0),
        # a batch of documents of unequal, odd lengths prefilled in one step
        _case("prompts ragged", "qwen3-4b", 12, 6, 301, 3967, 0),
        # one user's answer: decoding alone, bound by the weights
        _case("decode 1", "qwen3-4b", 12, 1, 517, 517, 96),
        # a few answers on a small model, where a step is mostly launches
        _case("decode 3 small", "qwen3-0.6b", 0, 3, 129, 387, 64),
        # the headline decode: eight sequences of up to 2,048 tokens
        _case("decode 8", "qwen3-4b", 12, 8, 1555, 2048, 96),
        # a full server: sixty-four shorter sequences, where attention and the products weigh alike
        _case("decode 64", "qwen3-4b", 12, 64, 65, 450, 64),
        # the path that checks the others, every product in 32 bits: prompts scored at every place, and generation
        _case("float32", "qwen3-0.6b", 0, 4, 9, 253, 24, "float32"),
        # the other designs: a batch of conversations, prompts and the start of the answers. Two kinds of recurrence and
        # attention with a capped score, a sink and a gate, on a float32 stream
        _case("piralix", "piralix-w2048", 6, 4, 501, 2048, 24),
        # the delta rule, a state-space recurrence beside windowed attention, experts chosen by a table
        _case("barilix", "barilix-w2048", 0, 4, 501, 2048, 24),
        # linear attention of two kinds beside chunks, a cache of latents, a polynomial feed-forward
        _case("fubinex", "fubinex-w2048", 0, 4, 501, 2048, 24),
        # differential attention, routed experts, several copies of the stream, a looped layer; one sequence alone
        _case("kaditar", "kaditar-w2048", 0, 1, 1999, 1999, 48),
    ]


def _log_between(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("prompt", "prompt", "decode", "decode", "decode", "float32", "design", "design", "design"))
    if kind == "prompt":
        batch, longest, steps = _log_between(rng, 1, 8), _log_between(rng, 16, 4096), 0
        longest = min(longest, 12800 // batch)
    elif kind == "decode":
        batch, steps = _log_between(rng, 1, 64), rng.randint(24, 64)
        longest = _log_between(rng, 16, min(2048, 16000 // batch))
    elif kind == "float32":
        batch, longest, steps = rng.randint(1, 4), _log_between(rng, 5, 253), rng.randint(8, 24)
    else:
        batch, longest, steps = _log_between(rng, 1, 8), _log_between(rng, 64, 2048), rng.randint(8, 48)
        longest = min(longest, 8000 // batch)
    model, layers = ("qwen3-0.6b", 0) if kind == "float32" else rng.choice(DESIGNS if kind == "design" else QWEN3)
    shortest = rng.randint(max(1, longest // 8), longest) if batch > 1 else longest
    return _case(None, model, layers, batch, shortest, longest, steps, "float32" if kind == "float32" else "bfloat16")


def lengths_of(case):
    """The prompts' lengths: evenly between the shortest and the longest, the longest somewhere in the middle."""
    n, lo, hi = case["batch"], case["shortest"], case["longest"]
    spread = [hi - (hi - lo) * i // max(1, n - 1) for i in range(n)]
    return spread[1::2] + spread[0::2]


def _config(case):
    raw = load_preset(case["model"])
    if not case["layers"]:
        return raw
    if "num_hidden_layers" in raw:
        return dict(raw, num_hidden_layers=case["layers"])
    return dict(raw, layers=raw["layers"][:case["layers"]], loop=None)


# ------------------------------------------------------------------------------------------ one pass
def _ids(case, seed, vocab):
    """Uniform token ids of the whole sequences ``[batch, longest + steps]``; a prompt is the first of its row, the
    tokens that are fed afterwards follow it."""
    gen = torch.Generator().manual_seed(seed)
    return torch.randint(0, vocab, (case["batch"], case["longest"] + case["steps"]), generator=gen)


def prepare(case, seed):
    """The engine with its weights, the prompts, the captured steps and a place for the logits."""
    lengths, steps, batch = lengths_of(case), case["steps"], case["batch"]
    longest = case["longest"] + steps
    engine = Engine(config=_config(case), seed=seed, dtype=case["dtype"], max_batch=batch,
                    max_len=max(4096, pages_for(longest) * PAGE_TOKENS),
                    max_tokens=sum(pages_for(n + steps + 1) for n in lengths) * PAGE_TOKENS)
    vocab = engine.stepper.vocab
    ids = _ids(case, seed, vocab)
    state = dict(case=case, engine=engine, lengths=lengths, steps=steps,
                 prompts=[ids[i, :n].tolist() for i, n in enumerate(lengths)])
    if case["dtype"] == "float32":
        engine.warm([batch], [longest])
        return state
    rows = sum(lengths)
    if rows <= SHORT_STEP:
        # one captured step for so many rows; a sequence more than the batch has owns the rows left over
        seqs = 1 << batch.bit_length()
        state["prompt_step"] = PromptGraph(engine.stepper, seqs, next(r for r in PROMPT_GRAPH_ROWS if r >= rows))
        state["prompt_step"].capture()
    if steps:
        width = pick_bucket(engine.batch_buckets, batch)
        reach = next(r for r in engine.context_ranges() if r >= longest)
        state["step"] = DecodeGraph(engine.stepper, width, reach)
        state["step"].capture()
        feed = torch.zeros((steps, width), dtype=torch.int32)
        for i, n in enumerate(lengths):
            feed[:, i] = ids[i, n:n + steps]
        state["feed"] = feed.to(engine.device)
        state["logits"] = torch.empty((steps, batch, vocab), dtype=torch.float32, device=engine.device)
        state["chosen"] = torch.empty((steps, width), dtype=torch.int32, device=engine.device)
        state["sampler"] = Sampler()
    return state


def run(state):
    engine, lengths, steps = state["engine"], state["lengths"], state["steps"]
    batch = len(lengths)
    if state["case"]["dtype"] == "float32":
        slots = engine.acquire(batch)
        scores = engine.step([SeqStep(s, p, list(range(len(p)))) for s, p in zip(slots, state["prompts"])])
        engine.release(slots)
        return {"scores": scores, "tokens": torch.tensor(engine.generate_all(state["prompts"], steps))}
    slots = engine.acquire(batch)
    engine.reserve(slots, [n + steps for n in lengths])
    if "prompt_step" in state:
        engine.cache.begin_step(slots, lengths)
        first = state["prompt_step"].replay(slots, state["prompts"])[:batch].clone()
        engine.cache.end_step(slots, lengths)
    else:
        first = engine.step([SeqStep(s, p, [len(p) - 1]) for s, p in zip(slots, state["prompts"])])
    out = {"first": first}
    if steps:
        ones = [1] * batch
        graph = state["step"]
        padded = slots + [-1] * (graph.batch - batch)                # rows that fill the captured step up sit out
        for i in range(steps):
            engine.cache.begin_step(slots, ones)
            logits = graph.replay(padded, state["feed"][i])
            engine.cache.end_step(slots, ones)
            state["sampler"].choose(logits, out=state["chosen"][i])
            state["logits"][i].copy_(logits[:batch])
        out["next"] = state["logits"]
        out["best"] = state["logits"].gather(2, state["chosen"][:, :batch, None].long())[..., 0]
    engine.release(slots)
    return out


# ------------------------------------------------------------------------------------------ what it cannot do without
def _model(case, device):
    raw = _config(case)
    arch = resolve_architecture(raw)
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    return raw, DecoderModel(arch.plan(arch.config_class.from_dict(raw)), dtype, device)


def work(case):
    """Each step reads the weights that its rows use once and what its sequences have cached; the logits are written."""
    raw, model = _model(case, "cpu")
    size = 4 if case["dtype"] == "float32" else 2
    lengths, steps, batch = lengths_of(case), case["steps"], case["batch"]
    specs = model.tensor_specs()
    tied = not any(s.name in ("lm_head.weight", "head") for s in specs)
    vocab, width = next(s.shape for s in specs if "embed" in s.name)
    routed = {id(s): layer for s in specs for layer in [_routed_layer(raw, s.name)] if layer is not None}

    def weights(rows):
        total = 0.0
        for s in specs:
            n = math.prod(s.shape) if s.shape else 1
            if "embed" in s.name and not tied:
                n = rows * width
            if id(s) in routed:
                router = routed[id(s)]["router"]
                n *= min(1.0, rows * router["top"] / router["experts"])
            total += n * size
        return total

    def cached(context):
        total = 0.0
        for need in model.cache_needs().values():
            for one in (need.values() if isinstance(need, dict) else (need,)):
                if isinstance(one, KVNeed):
                    seen = min(context, one.window) if one.window else context
                    total += one.num_kv_heads * (one.head_dim + one.values) * size * seen
                elif one is not None:
                    total += 2.0 * 4 * math.prod(one.shape)
        return total

    spans = [(0, n) for n in lengths]
    if case["dtype"] == "float32":
        # the prompts twice: scored at every place, and as the beginning of what is generated
        moved = 2 * weights(sum(lengths)) + sum(lengths) * vocab * 4.0
        flops = model.step_flops(spans, sum(lengths)) + model.step_flops(spans, batch)
        decoded = range(steps - 1)
    else:
        moved = weights(sum(lengths)) + batch * vocab * 4.0
        flops = model.step_flops(spans, batch)
        decoded = range(steps)
    moved += sum(cached(n) for n in lengths)
    for i in decoded:
        moved += weights(batch) + sum(cached(n + i) for n in lengths) + batch * vocab * 4.0
        flops += model.step_flops([(n + i, 1) for n in lengths], batch)
    return {"bytes": moved, "flops": flops}


def _routed_layer(raw, name):
    """The feed-forward that the expert tensor ``name`` belongs to, or None."""
    parts = name.split(".")
    if len(parts) >= 4 and parts[1] == "mlp" and parts[2][0] == "e" and parts[2][1:].isdigit():
        return raw["layers"][int(parts[0][1:])]["mlp"]
    return None


def tolerance(case):
    if case["dtype"] == "float32":
        # 2e-6 from 64 bits; a chosen token changes only where two logits agree to that
        return {"rel": 1e-5, "max": 1e-4, "differ": 0.01}
    # the same sequences through other kernels (in one step, or one by one) differ by 0.6 to 2.1 %; the largest single
    # differences are some six times that
    return {"rel": 0.03, "max": 0.3}


# ------------------------------------------------------------------------------------------ the models in 64 bits
def exact(case, seed):
    raw, model = _model(case, "cuda")
    dtype = torch.float32 if case["dtype"] == "float32" else torch.bfloat16
    tensors = random_tensors(model.tensor_specs(), seed, dtype, device="cuda")
    vocab = model.plan.vocab_size
    ids = _ids(case, seed, vocab).cuda()
    lengths, steps = lengths_of(case), case["steps"]
    if case["dtype"] == "float32":
        x, head = FORWARDS[case["model"].split("-")[0]](raw, _Weights(tensors), ids[:, :case["longest"]])
        scores = torch.cat([x[i, :n] for i, n in enumerate(lengths)]) @ head.T
        return {"scores": scores, "tokens": None}
    # a row's padding lies behind everything that is read of it, and nothing looks ahead
    x, head = FORWARDS[case["model"].split("-")[0]](raw, _Weights(tensors), ids)
    at = torch.tensor(lengths, device="cuda")
    cap = raw.get("logit_softcap")
    rows = torch.arange(len(lengths), device="cuda")
    first = x[rows, at - 1] @ head.T
    first = cap * torch.tanh(first / cap) if cap else first
    out = {"first": first}
    if steps:
        out["next"] = torch.empty((steps, len(lengths), vocab), dtype=torch.float64, device="cuda")
        for i in range(steps):
            logits = x[rows, at + i] @ head.T
            out["next"][i] = cap * torch.tanh(logits / cap) if cap else logits
        out["best"] = out["next"].amax(-1)
    return out


class _Weights:
    """Tensors by name, in 64 bits when asked for; ``w("l0.mix.")`` is a view below a prefix."""

    def __init__(self, tensors, prefix=""):
        self.tensors, self.prefix = tensors, prefix

    def __call__(self, prefix):
        return _Weights(self.tensors, self.prefix + prefix)

    def __getitem__(self, name):
        t = self.tensors[self.prefix + name]
        return t.double() if t.is_floating_point() else t

    def __contains__(self, name):
        return self.prefix + name in self.tensors


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, eps):
    return _rms(x - x.mean(-1, keepdim=True), eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return torch.logaddexp(x, torch.zeros_like(x))


def _turned(x, freqs, halves, both=1.0):
    """``x [B, T, heads, D]``: the first ``2 len(freqs)`` features of a head turn by position times frequency, feature
    ``i`` with ``i + len(freqs)`` (``halves``) or neighbours with one another."""
    n = freqs.numel()
    angle = torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * freqs.to(x.device)[None, :]
    cos, sin = (angle.cos() * both)[None, :, None, :], (angle.sin() * both)[None, :, None, :]
    u, v = (x[..., :n], x[..., n:2 * n]) if halves else (x[..., 0:2 * n:2], x[..., 1:2 * n:2])
    a, b = u * cos - v * sin, v * cos + u * sin
    turned = torch.cat([a, b], -1) if halves else torch.stack([a, b], -1).flatten(-2)
    return torch.cat([turned, x[..., 2 * n:]], -1)


def _plain_frequencies(rot):
    return rot["base"] ** (-torch.arange(0, rot["dims"], 2, dtype=torch.float64) / rot["dims"])


def _yarn_frequencies(rot):
    """The stretched frequencies and the factor on cosine and sine."""
    f, scaling, dims = _plain_frequencies(rot), rot.get("scaling"), rot["dims"]
    if not scaling:
        return f, 1.0

    def dim_of(turns):
        return dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))

    lo, hi = max(math.floor(dim_of(scaling["fast"])), 0), min(math.ceil(dim_of(scaling["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=torch.float64) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / scaling["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(scaling["factor"]) + 1


def _banded_frequencies(rot):
    """Long wavelengths stretched, short ones kept, those between blended."""
    f, scaling = _plain_frequencies(rot), rot.get("scaling")
    if not scaling:
        return f
    blend = ((scaling["original"] * f / (2 * math.pi) - scaling["low"]) / (scaling["high"] - scaling["low"])).clamp(0, 1)
    return (1 - blend) * f / scaling["factor"] + blend * f


def _seen(T, device, window=None, chunk=None):
    i = torch.arange(T, device=device)
    back = i[:, None] - i[None, :]
    seen = back >= 0
    if window:
        seen &= back < window
    if chunk:
        seen &= (i[:, None] // chunk) == (i[None, :] // chunk)
    return seen


def _attend(q, k, v, scale, seen, softcap=None, sink=None):
    """``q [B, T, H, D]``, ``k, v [B, T, G, .]``: query head ``h`` reads kv head ``h // (H / G)``; a sink joins the
    denominator only."""
    B, T, H, _ = q.shape
    per = H // k.shape[2]
    out = torch.empty((B, T, H, v.shape[-1]), dtype=q.dtype, device=q.device)
    for b in range(B):
        for h in range(H):
            s = (q[b, :, h] @ k[b, :, h // per].T) * scale
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            s = s.masked_fill(~seen, -math.inf)
            if sink is not None:
                s = torch.cat([s, sink[h].expand(T, 1)], 1)
            p = torch.softmax(s, -1)
            out[b, :, h] = (p[:, :T] if sink is not None else p) @ v[b, :, h // per]
    return out


def _conv(u, taps_of, bias=None):
    """A causal convolution over time per channel; the last tap meets the current token."""
    taps = taps_of.shape[1]
    padded = torch.nn.functional.pad(u, (0, 0, taps - 1, 0))
    y = sum(padded[:, j:j + u.shape[1]] * taps_of[:, j] for j in range(taps))
    return y if bias is None else y + bias


def _clamped(h, w, limit):
    g, u = (h @ w["gate"].T).clamp(max=limit), (h @ w["up"].T).clamp(-limit, limit)
    return (g * torch.sigmoid(1.702 * g) * (u + 1)) @ w["down"].T


def _gated(h, w, act=_silu):
    return (act(h @ w["gate"].T) * (h @ w["up"].T)) @ w["down"].T


def _qwen3(raw, w, ids):
    B, T = ids.shape
    H, G, D, eps = raw["num_attention_heads"], raw["num_key_value_heads"], raw["head_dim"], raw["rms_norm_eps"]
    # the model's angles are products of 32-bit numbers
    freqs = 1.0 / (raw["rope_theta"] ** (torch.arange(0, D, 2, dtype=torch.int64).to(torch.float32) / D))
    angle = (torch.arange(T, dtype=torch.float32)[:, None] * freqs[None, :]).double().cuda()
    cos, sin = angle.cos()[None, :, None, :], angle.sin()[None, :, None, :]

    def turned(x):
        u, v = x[..., :D // 2], x[..., D // 2:]
        return torch.cat([u * cos - v * sin, v * cos + u * sin], -1)

    seen = _seen(T, ids.device)
    x = w.tensors["model.embed_tokens.weight"][ids].double()
    for i in range(raw["num_hidden_layers"]):
        p = w(f"model.layers.{i}.")
        a = p("self_attn.")
        h = _rms(x, eps) * p["input_layernorm.weight"]
        q = turned(_rms((h @ a["q_proj.weight"].T).view(B, T, H, D), eps) * a["q_norm.weight"])
        k = turned(_rms((h @ a["k_proj.weight"].T).view(B, T, G, D), eps) * a["k_norm.weight"])
        v = (h @ a["v_proj.weight"].T).view(B, T, G, D)
        x = x + _attend(q, k, v, D ** -0.5, seen).reshape(B, T, H * D) @ a["o_proj.weight"].T
        h = _rms(x, eps) * p["post_attention_layernorm.weight"]
        m = p("mlp.")
        x = x + (_silu(h @ m["gate_proj.weight"].T) * (h @ m["up_proj.weight"].T)) @ m["down_proj.weight"].T
    head = w["model.embed_tokens.weight" if raw.get("tie_word_embeddings") else "lm_head.weight"]
    return _rms(x, eps) * w["model.norm.weight"], head


def _runs(raw):
    """``(layer, which pass of the loop it opens or None)`` in order."""
    n, loop = len(raw["layers"]), raw.get("loop")
    if not loop:
        return [(i, None) for i in range(n)]
    a, b = loop["start"], loop["stop"]
    return [(i, None) for i in range(a)] + [(i, t if i == a else None) for t in range(loop["times"]) for i in range(a, b)] + \
        [(i, None) for i in range(b, n)]


def _piralix(raw, w, ids):
    eps = raw["norm"]["eps"]
    B, T = ids.shape
    embedded = x = w["embed"][ids]
    for i, opens in _runs(raw):
        layer, p = raw["layers"][i], w(f"l{i}.")
        if opens is not None:
            x = x + (embedded if opens > 0 else 0) + w["loop.step"][opens]
        h, m, c = _rms(x, eps) * p["norm1"], p("mix."), layer["mixer"]
        if layer["type"] == "attention":
            H, G, D, Dv = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
            freqs, both = _yarn_frequencies(c["rot"])
            q = _turned((h @ m["q"].T).view(B, T, H, D), freqs, False, both)
            k = _turned((h @ m["k"].T).view(B, T, G, D), freqs, False, both)
            o = _attend(q, k, (h @ m["v"].T).view(B, T, G, Dv), c["scale"], _seen(T, ids.device), c.get("softcap"), m["sink"])
            y = (o.reshape(B, T, H * Dv) * torch.sigmoid(h @ m["g"].T)) @ m["o"].T
        elif layer["type"] == "mlstm":
            H, D, Dv, cap = c["heads"], c["dim"], c["vdim"], c["gate_cap"]
            q = (h @ m["q"].T).view(B, T, H, D) * D ** -0.5
            k, v = (h @ m["k"].T).view(B, T, H, D), (h @ m["v"].T).view(B, T, H, Dv)
            take = cap * torch.tanh((h @ m["i"].T + m["i.b"]) / cap)
            keep = -_softplus(-cap * torch.tanh((h @ m["f"].T + m["f.b"]) / cap))
            S, n, top = h.new_zeros(B, H, D, Dv), h.new_zeros(B, H, D), h.new_zeros(B, H)
            o = h.new_empty(B, T, H, Dv)
            for t in range(T):
                new = torch.maximum(keep[:, t] + top, take[:, t])
                old, now = torch.exp(keep[:, t] + top - new)[..., None], torch.exp(take[:, t] - new)[..., None]
                S = old[..., None] * S + (now * k[:, t])[..., None] * v[:, t, :, None, :]
                n, top = old * n + now * k[:, t], new
                den = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
                o[:, t] = (S * q[:, t][..., None]).sum(-2) / den[..., None]
            y = (_rms(o, eps).reshape(B, T, H * Dv) * m["norm"] * torch.sigmoid(h @ m["g"].T)) @ m["o"].T
        else:
            W, blocks = c["width"], c["blocks"]
            side = torch.nn.functional.gelu(h @ m["y"].T + m["y.b"], approximate="tanh")
            u = _conv(h @ m["x"].T + m["x.b"], m["conv"], m["conv.b"])
            ub = u.view(B, T, blocks, 1, W // blocks)
            r = torch.sigmoid((ub * m["ra"]).sum(-1) + m["ra.b"].view(blocks, -1)).reshape(B, T, W)
            g = torch.sigmoid((ub * m["ri"]).sum(-1) + m["ri.b"].view(blocks, -1)).reshape(B, T, W)
            a = torch.exp(-8.0 * r * _softplus(m["lam"]))
            b = torch.sqrt(1 - a * a) * g * u
            S, o = h.new_zeros(B, W), torch.empty_like(u)
            for t in range(T):
                S = a[:, t] * S + b[:, t]
                o[:, t] = S
            y = (o * side) @ m["o"].T
        x = x + _rms(y, eps) * p["norm1b"]
        if layer.get("mlp"):
            y = _clamped(_rms(x, eps) * p["norm2"], p("mlp."), layer["mlp"]["limit"])
            x = x + _rms(y, eps) * p["norm2b"]
    return _rms(x, eps) * w["final.norm"], w["embed"]


def _streams(streams, hc, y):
    mix, out = hc["mix"], hc["out"]
    return [sum(mix[s, t] * streams[s] for s in range(len(streams))) + out[t] * y for t in range(len(streams))]


def _routed(h, w, chosen, weights, experts, one):
    """Every expert on every row, times the weight of the rows that chose it."""
    share = torch.zeros(h.shape[:-1] + (experts,), dtype=h.dtype, device=h.device).scatter(-1, chosen, weights)
    return sum(share[..., e:e + 1] * one(h, w(f"e{e}.")) for e in range(experts))


def _state_space(h, m, c, eps):
    B, T, _ = h.shape
    H, P, N, G = c["heads"], c["vdim"], c["state"], c["groups"]
    inner = H * P
    proj = h @ m["in"].T
    z, xbc, dt = proj[..., :inner], proj[..., inner:2 * inner + 2 * G * N], proj[..., 2 * inner + 2 * G * N:]
    xbc = _silu(_conv(xbc, m["conv"], m["conv.b"]))
    x = xbc[..., :inner].view(B, T, H, P)
    into, read = (xbc[..., inner + s * G * N:inner + (s + 1) * G * N].view(B, T, G, N).repeat_interleave(H // G, 2)
                  for s in (0, 1))
    dt = _softplus(dt + m["dt_bias"])
    keep = torch.exp(-torch.exp(m["A_log"]) * dt)
    S, y = h.new_zeros(B, H, N, P), torch.empty_like(x)
    for t in range(T):
        S = keep[:, t, :, None, None] * S + (dt[:, t, :, None] * into[:, t])[..., None] * x[:, t, :, None, :]
        y[:, t] = (S * read[:, t][..., None]).sum(-2)
    y = (y + m["D"][:, None] * x).reshape(B, T, inner) * _silu(z)
    return (_rms(y.view(B, T, c["norm_groups"], -1), eps).reshape(B, T, inner) * m["norm"]) @ m["o"].T


def _barilix(raw, w, ids):
    eps = raw["norm"]["eps"]
    B, T = ids.shape
    x = w["embed"][ids] * raw["embedding"]["scale"]
    for i, layer in enumerate(raw["layers"]):
        m, c = w(f"l{i}.mix."), layer["mixer"]
        if layer["type"] == "parallel":
            a, left = m("left."), c["left"]
            H, G, D, Dv = left["heads"], left["kv_heads"], left["dim"], left["vdim"]
            q, k, v = (_conv(x @ a[n].T + a[n + ".b"], a[n + ".conv"]) for n in "qkv")
            freqs = _banded_frequencies(left["rot"])
            q = _turned(_rms(q.view(B, T, H, D), eps) * a["q.norm"], freqs, True)
            k = _turned(_rms(k.view(B, T, G, D), eps) * a["k.norm"], freqs, True)
            o = _attend(q, k, v.view(B, T, G, Dv), left["scale"], _seen(T, ids.device, left["mask"]["size"]))
            one = o.reshape(B, T, H * Dv) @ a["o"].T + a["o.b"]
            two = _state_space(x, m("right."), c["right"], eps)
            y = 0.5 * (_rms(one, eps) * m["left.out"] + _rms(two, eps) * m["right.out"])
        else:
            H, G, D, P = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
            q, k, v = (_silu(_conv(x @ m[n].T, m[n + ".conv"])) for n in "qkv")
            q, k, v = q.view(B, T, G, D), k.view(B, T, G, D), v.view(B, T, H, P)
            q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
            q, k = (q * D ** -0.5).repeat_interleave(H // G, 2), k.repeat_interleave(H // G, 2)
            beta = torch.sigmoid(x @ m["b"].T)
            decay = torch.exp(-torch.exp(m["A_log"]) * _softplus(x @ m["a"].T + m["dt_bias"]))
            S, o = x.new_zeros(B, H, D, P), torch.empty_like(v)
            for t in range(T):
                S = decay[:, t, :, None, None] * S
                u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t][..., None]).sum(-2))
                S = S + k[:, t][..., None] * u[:, :, None, :]
                o[:, t] = (S * q[:, t][..., None]).sum(-2)
            o = _rms(o, eps) * m["norm"] * _silu(x @ m["g"].T).view(B, T, H, P)
            y = o.reshape(B, T, H * P) @ m["o"].T
        x = x + _layer_norm(y, eps) * w[f"l{i}.norm1"]
        if layer.get("mlp"):
            m, c = w(f"l{i}.mlp."), layer["mlp"]
            if c["kind"] == "dense":
                y = _gated(x, m)
            else:
                chosen, r = m["table"][ids].long(), c["router"]
                y = _routed(x, m, chosen, torch.full(chosen.shape, 1.0 / r["top"], dtype=x.dtype, device=x.device),
                            r["experts"], _gated)
                y = y + _gated(x, m("shared."))
            x = x + _layer_norm(y, eps) * w[f"l{i}.norm2"]
    return _layer_norm(x, eps) * w["final.norm"], w["head"]


def _linear_walk(q, k, v, decay):
    S, out = q.new_zeros(q.shape[0], q.shape[2], q.shape[3], v.shape[3]), torch.empty_like(v)
    for t in range(q.shape[1]):
        S = decay[:, t][..., None] * S + k[:, t][..., None] * v[:, t, :, None, :]
        out[:, t] = (S * q[:, t][..., None]).sum(-2)
    return out


def _fubinex(raw, w, ids):
    eps, groups = raw["norm"]["eps"], raw["norm"]["groups"]
    B, T = ids.shape

    def normed(x, weight):
        return _rms(x.view(B, T, groups, -1), eps).reshape(B, T, -1) * weight

    x, latents = w["embed"][ids] * raw["embedding"]["scale"], {}
    for i, layer in enumerate(raw["layers"]):
        p, c = w(f"l{i}."), layer["mixer"]
        h, m = normed(x, p["norm1"]), p("mix.")
        if layer["type"] == "parallel":
            a, left = m("left."), c["left"]
            H, G, D, Dv = left["heads"], left["kv_heads"], left["dim"], left["vdim"]
            freqs = _plain_frequencies(left["rot"])
            q = _rms(_turned((h @ a["q"].T).view(B, T, H, D), freqs, True), eps)
            k = _rms(_turned((h @ a["k"].T).view(B, T, G, D), freqs, True), eps)
            o = _attend(q, k, (h @ a["v"].T).view(B, T, G, Dv), left["scale"], _seen(T, ids.device, chunk=left["mask"]["size"]))
            one = o.reshape(B, T, H * Dv) @ a["o"].T
            a, right = m("right."), c["right"]
            H, D, Dv = right["heads"], right["dim"], right["vdim"]
            decay = torch.sigmoid((h @ a["a1"].T) @ a["a2"].T + a["a2.b"]) ** (1.0 / right["tau"])
            o = _linear_walk((h @ a["q"].T).view(B, T, H, D) * D ** -0.5, (h @ a["k"].T).view(B, T, H, D),
                             (h @ a["v"].T).view(B, T, H, Dv), decay.view(B, T, H, D))
            o = (_rms(o, eps) * a["norm"]).reshape(B, T, H * Dv)
            y = c["left_scale"] * one + c["right_scale"] * ((o * _silu(h @ a["g"].T)) @ a["o"].T)
        elif layer["type"] == "retention":
            H, D, Dv = c["heads"], c["dim"], c["vdim"]
            freqs = _plain_frequencies(c["rot"])
            q = _turned((h @ m["q"].T).view(B, T, H, D), freqs, True)
            k = _turned((h @ m["k"].T).view(B, T, H, D), freqs, True) * D ** -0.5
            decay = torch.tensor(c["decay"], dtype=h.dtype, device=h.device)[None, None, :, None].expand(B, T, H, D)
            o = _rms(_linear_walk(q, k, (h @ m["v"].T).view(B, T, H, Dv), decay), eps)
            y = (o.reshape(B, T, H * Dv) * _silu(h @ m["g"].T)) @ m["o"].T
        else:
            H, D, R, Dv, L = c["heads"], c["dim"], c["rot_dim"], c["vdim"], c["kv_rank"]
            freqs, both = _yarn_frequencies(c["rot"])
            q = ((_rms(h @ m["dq"].T, eps) * m["dq.norm"]) @ m["uq"].T).view(B, T, H, D + R)
            q = torch.cat([q[..., :D], _turned(q[..., D:], freqs, False, both)], -1)
            if c.get("kv_from") is None:
                down = h @ m["dkv"].T
                latents[i] = (_rms(down[..., :L], eps) * m["dkv.norm"], _turned(down[:, :, None, L:], freqs, False, both))
            latent, k_rot = latents[i if c.get("kv_from") is None else c["kv_from"]]
            k = torch.cat([(latent @ m["uk"].T).view(B, T, H, D), k_rot.expand(B, T, H, R)], -1)
            o = _attend(q, k, (latent @ m["uv"].T).view(B, T, H, Dv), c["scale"], _seen(T, ids.device))
            y = o.reshape(B, T, H * Dv) @ m["o"].T
        x = x + y
        if layer.get("mlp"):
            m = p("mlp.")
            z = normed(x, p["norm2"]) @ m["up"].T
            a, b, cube, e = m["act"]
            x = x + (a * _rms(z, eps) + b * _rms(z ** 2, eps) + cube * _rms(z ** 3, eps) + e) @ m["down"].T
    return normed(x, w["final.norm"]), w["head"]


def _kaditar(raw, w, ids):
    eps = raw["norm"]["eps"]
    B, T = ids.shape
    streams = [w["embed"][ids]] * raw["streams"]
    for i, _ in _runs(raw):
        layer = raw["layers"][i]
        for part, kind in ((1, "mix"), (2, "mlp")):
            if kind == "mlp" and layer["mlp"] is None:
                continue
            hc, m = w(f"l{i}.hc{part}."), w(f"l{i}.{kind}.")
            into = hc["in"]
            h = _layer_norm(sum(into[s] * x for s, x in enumerate(streams)), eps) * w[f"l{i}.norm{part}"] + \
                w[f"l{i}.norm{part}.b"]
            if kind == "mix":
                c = layer["mixer"]
                H, G, D, Dv = c["heads"], c["kv_heads"], c["dim"], c["vdim"]
                freqs = _plain_frequencies(c["rot"])
                q = _turned((h @ m["q"].T + m["q.b"]).view(B, T, 2 * H, D), freqs, False).view(B, T, H, 2, D)
                k = _turned((h @ m["k"].T + m["k.b"]).view(B, T, 2 * G, D), freqs, False).view(B, T, G, 2, D)
                v = (h @ m["v"].T + m["v.b"]).view(B, T, G, Dv)
                seen = _seen(T, ids.device, (c.get("mask") or {}).get("size"))
                one, two = (_attend(q[:, :, :, s], k[:, :, :, s], v, c["scale"], seen) for s in (0, 1))
                share = torch.exp((m["lq1"] * m["lk1"]).sum()) - torch.exp((m["lq2"] * m["lk2"]).sum()) + c["diff"]
                y = (_rms(one - share * two, eps) * (1 - c["diff"])).reshape(B, T, H * Dv) @ m["o"].T
            elif layer["mlp"]["kind"] == "dense":
                y = _gated(h, m, torch.relu)
            else:
                r = layer["mlp"]["router"]
                best = (h @ m["router"].T + m["router.b"]).topk(r["top"], -1)
                y = _routed(h, m, best.indices, torch.softmax(best.values, -1), r["experts"], _gated)
                y = y + torch.sigmoid(h @ m["shared.sg"].T) * _gated(h, m("shared."))
            streams = _streams(streams, hc, y)
    x = sum(streams)
    return _layer_norm(x, eps) * w["final.norm"] + w["final.norm.b"], w["embed"]


FORWARDS = {"qwen3": _qwen3, "piralix": _piralix, "barilix": _barilix, "fubinex": _fubinex,
            "kaditar": _kaditar}
