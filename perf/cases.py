"""What the library is measured on: listed calls of its public entry points, from the smallest to the
largest, and how to draw more of the same ranges.

A case says which model, in which type, and one of four tasks:

* `prompt`: the prompts of new requests go through one step (`Engine.alloc`, `Engine.step`, `Engine.free`);
* `decode`: requests whose prompts lie in the cache already bring one token each (`Engine.step`), the next
  pass the next token, as in a serving loop that goes on;
* `replay`: a trace of given tokens, prompts and then one token a step, as `bin/trace_run` goes through it;
* `sample`: tokens are drawn from logits (`Sampler.sample`).

Prompt lengths follow from the case alone: the last request's is `high`, the others lie between `low`
and `high`.  Weights and tokens are made from the seed.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch

from torchless_rs_amd import SamplingConfig, config_from_dict
from torchless_rs_amd.engine import Engine, SeqInput, model_from_tensors
from torchless_rs_amd.kernels.page import PAGE, round_up
from torchless_rs_amd.models import model_spec_for
from torchless_rs_amd.sampling.sampler import Sampler

DEVICE = "cuda:0"
F64 = torch.float64
EXACT_TOKENS = {"7b-v0.1": 10000, "7b-v0.3": 16400, "nemo-12b": 5000, "2b": 4096, "nepisun": 6000, "giforax": 8000}
ROOM = 4096                 # positions that a decoding request can still grow by

# The shapes of the benchmark: two 7B ones with and without a window, the 12B one, and four layers of the
# 2B sizes for the 32-bit path
_7B = dict(num_hidden_layers=32, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8, head_dim=128,
           intermediate_size=14336, vocab_size=32000, rope_theta=1e4, sliding_window=4096, rms_norm_eps=1e-5)
SHAPES = {
    "7b-v0.1": _7B,
    "7b-v0.3": dict(_7B, vocab_size=32768, rope_theta=1e6, sliding_window=None),
    "nemo-12b": dict(_7B, num_hidden_layers=40, hidden_size=5120, vocab_size=131072, rope_theta=1e6, sliding_window=None),
    "2b": dict(_7B, num_hidden_layers=4, hidden_size=2048, head_dim=64, intermediate_size=8192, sliding_window=1024),
}
VOCAB = {"7b-v0.1": 32000, "7b-v0.3": 32768, "nemo-12b": 131072, "2b": 32000, "nepisun": 32000, "giforax": 32000}


def _design(model: str) -> dict:
    """config.json of the two designs with routed experts, four layers at the sizes of a 7B model as the
    benchmark builds them: between them a state-space mixer, a recurrence, windows, chunks, values
    mixed and keys shared between layers, plain and gated experts with and without groups."""
    rot = {"base": 10000.0}
    att = {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5}
    if model == "nepisun":
        ssm = {"heads": 128, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
        moe = {"kind": "moe", "router": {"experts": 16, "top": 4, "groups": {"count": 4, "keep": 2}},
               "expert": {"ff": 3584}, "shared": {"ff": 7168}}
        a = dict(att, rot=dict(rot, dims=128), v_mix=True)
        layers = [("mamba2", ssm, {"kind": "dense", "ff": 14336}), ("mamba2", ssm, moe),
                  ("attention_2", dict(a, mask={"size": 4096, "keep_first": 64}), moe), ("attention", a, moe)]
        extra = {}
    else:
        moe = {"kind": "moe", "router": {"experts": 16, "top": 4}, "expert": {"ff": 1792, "limit": 7.0},
               "shared": {"ff": 7168, "limit": 7.0}}
        a = dict(att, rot=dict(rot, dims=64), mask={"size": 4096})
        layers = [("attention", a, moe), ("attention", dict(a, kv_from=0), moe), ("mingru", {"width": 4096}, moe),
                  ("attention", a, moe)]
        extra = {"embedding": {"scale": 1.0}}
    return dict({"architecture": model.capitalize(), "vocab": 32000, "width": 4096, "norm": {"eps": 1e-6},
                 "layers": [{"type": t, "mixer": m, "mlp": f} for t, m, f in layers]}, **extra)


def _config(model: str) -> dict:
    return dict(SHAPES[model], architectures=["MistralForCausalLM"]) if model in SHAPES else _design(model)


def listed():
    bf = {"dtype": "bfloat16"}
    return [
        # one draw for a batch of requests at a temperature, the largest vocabulary: what follows every step
        {"name": "sample_b16_v131072", "task": "sample", "model": "nemo-12b", "batch": 16, "temperature": 0.7,
         "top_k": 50, "top_p": 0.95},
        # a chat with one user, a token at a time: every launch counts
        {"name": "decode_b1", "task": "decode", "model": "7b-v0.1", **bf, "batch": 1, "low": 1024, "high": 1024},
        # the benchmark's headline: eight requests past a full window of 4,096
        {"name": "decode_b8_window", "task": "decode", "model": "7b-v0.1", **bf, "batch": 8, "low": 4096, "high": 4300},
        # a server under load: many requests of unequal lengths
        {"name": "decode_b64", "task": "decode", "model": "7b-v0.1", **bf, "batch": 64, "low": 128, "high": 2048},
        # long documents without a window
        {"name": "decode_b8_long", "task": "decode", "model": "7b-v0.3", **bf, "batch": 8, "low": 1024, "high": 8192},
        # the benchmark's prompt
        {"name": "prompt_2048", "task": "prompt", "model": "7b-v0.1", **bf, "batch": 1, "low": 2048, "high": 2048},
        # a few questions that arrive together: more rows than the decode kernels take, too few to fill the chip
        {"name": "prompt_3x64", "task": "prompt", "model": "7b-v0.1", **bf, "batch": 3, "low": 37, "high": 91},
        # a long document in one step
        {"name": "prompt_16384", "task": "prompt", "model": "7b-v0.3", **bf, "batch": 1, "low": 16384, "high": 16384},
        # ragged prompts through state-space layers and routed experts
        {"name": "nepisun_prompt", "task": "prompt", "model": "nepisun", **bf, "batch": 4, "low": 128, "high": 1024},
        # tokens through recurrent states and every expert
        {"name": "nepisun_decode_b8", "task": "decode", "model": "nepisun", **bf, "batch": 8, "low": 256, "high": 2048},
        # ragged prompts through logistic attention, a recurrence and gated experts
        {"name": "giforax_prompt", "task": "prompt", "model": "giforax", **bf, "batch": 3, "low": 300, "high": 1100},
        # a trace in 32 bits, as results are checked
        {"name": "replay_f32", "task": "replay", "model": "2b", "dtype": "float32", "batch": 2, "low": 20, "high": 48,
         "new": 8},
    ]


def draw(rng):
    def spread(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))

    task = rng.choice(["decode", "decode", "prompt", "prompt", "prompt", "sample", "replay"])
    if task == "sample":
        greedy = rng.random() < 0.3
        return {"task": task, "model": rng.choice(["7b-v0.1", "nemo-12b"]), "batch": spread(1, 64),
                "temperature": 0.0 if greedy else round(rng.uniform(0.3, 1.2), 2),
                "top_k": 0 if greedy else rng.choice([0, spread(2, 200)]),
                "top_p": 0.0 if greedy else rng.choice([0.0, round(rng.uniform(0.5, 0.99), 2)])}
    if task == "replay":
        high = spread(4, 64)
        return {"task": task, "model": "2b", "dtype": "float32", "batch": spread(1, 4), "low": max(1, high // 2),
                "high": high, "new": spread(2, 8)}
    model = rng.choice(["7b-v0.1", "7b-v0.1", "7b-v0.3", "nemo-12b", "nepisun", "giforax"])
    batch = spread(1, 64)
    most = {"prompt": 8192, "decode": 60000 if model in ("7b-v0.1", "7b-v0.3") else 24000}[task]
    most = max(8, min(most // batch, 2048 if model in ("nepisun", "giforax") else 8192))
    high = spread(8 if task == "prompt" else min(most, 128), most)
    return {"task": task, "model": model, "dtype": "bfloat16", "batch": batch, "low": max(1, int(high * rng.uniform(0.2, 1.0))),
            "high": high}


def lengths(case):
    rng = random.Random(f"{case['batch']} {case['low']} {case['high']}")
    return [rng.randint(case["low"], case["high"]) for _ in range(case["batch"] - 1)] + [case["high"]]


def _checked(case) -> int:
    """How many of the leading requests `exact` goes through."""
    left, n = EXACT_TOKENS[case["model"]], 0
    for l in lengths(case):
        left -= l
        if left < 0:
            break
        n += 1
    return n


def _tokens(case, seed, gen):
    """Prompts, and rows of tokens that follow them, as lists of ids."""
    v = VOCAB[case["model"]]
    ids = [torch.randint(0, v, (n,), generator=gen).tolist() for n in lengths(case)]
    after = torch.randint(0, v, (256, case["batch"]), generator=gen).tolist()
    return ids, after


def weights(case, seed):
    """Random weights by their names in the checkpoint: products N(0, 1 / fan in), an embedding N(0, 1), norms
    of one or near it.  The designs: decays and steps of the state-space layers as such layers are
    initialised, and a router that tells tokens apart: a token's embedding leans to the rows of the
    experts that it uses, as a trained router's choice is not a toss-up."""
    model = case["model"]
    specs = model_spec_for(config_from_dict(_config(model))).weight_specs()
    dtype = getattr(torch, case["dtype"])
    gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def randn(*shape):
        return torch.randn(shape, generator=gen, device=DEVICE, dtype=torch.float32)

    out = {}
    for name, spec in specs.items():
        shape = tuple(spec.shape)
        if model in SHAPES:
            out[name] = (torch.ones(shape, dtype=dtype, device=DEVICE) if len(shape) == 1 else
                         torch.randn(shape, generator=gen, device=DEVICE, dtype=dtype).mul_(
                             1.0 if "embed_tokens" in name else shape[-1] ** -0.5))
            continue
        leaf = name.split(".", 1)[1] if name.startswith("l") else name
        if leaf.endswith(".b"):
            t = 0.1 * randn(*shape)
        elif "norm" in leaf:
            t = 1.0 + 0.1 * randn(*shape)
        elif leaf == "dwa":
            t = 1.0 / shape[0] + 0.05 * randn(*shape)
        elif leaf == "mix.vmix":
            t = torch.full(shape, 0.5, device=DEVICE)
        elif leaf == "mix.pb":
            t = -4.0 + randn(*shape)
        elif leaf == "mix.A_log":
            t = torch.log(torch.empty(shape, device=DEVICE).uniform_(1.0, 16.0, generator=gen))
        elif leaf == "mix.dt_bias":
            dt = torch.exp(torch.empty(shape, device=DEVICE).uniform_(math.log(1e-3), math.log(1e-1), generator=gen))
            t = torch.log(torch.expm1(dt))
        elif leaf == "mix.D":
            t = 1.0 + 0.1 * randn(*shape)
        elif leaf == "mix.conv":
            t = randn(*shape) * 0.5
        elif leaf == "embed" or name == "embed":
            t = randn(*shape)
        else:
            t = torch.randn(shape, generator=gen, device=DEVICE, dtype=dtype).mul_(shape[-1] ** -0.5)
        out[name] = t.to(dtype)
    if model not in SHAPES:
        rows = randn(16, 4096)
        V = VOCAB[model]
        pick = torch.rand((V, 16), generator=gen, device=DEVICE)
        if model == "nepisun":                       # two experts of each of two groups of four
            groups = torch.zeros((V, 4), device=DEVICE).scatter_(
                1, torch.rand((V, 4), generator=gen, device=DEVICE).topk(2).indices, 1.0)
            best = pick.view(V, 4, 4)
            used = (best >= best.topk(2, dim=-1).values[..., -1:]).float() * groups[:, :, None]
            used = used.view(V, 16)
        else:
            used = (pick >= pick.topk(4, dim=-1).values[:, -1:]).float()
        out["embed"] = (out["embed"].float() + 0.6 * used @ rows).to(dtype)
        for i in range(4):
            if f"l{i}.mlp.router" in out:            # each layer has the experts in another order
                out[f"l{i}.mlp.router"] = (rows.roll(4 * i, 0) / 400.0).to(dtype)
    return out


def prepare(case, seed):
    gen = torch.Generator().manual_seed(seed)
    if case["task"] == "sample":
        g = torch.Generator(device=DEVICE).manual_seed(seed)
        logits = 2.5 * torch.randn((case["batch"], VOCAB[case["model"]]), generator=g, device=DEVICE)
        cfg = (SamplingConfig(case["temperature"], case["top_k"] or None, case["top_p"] or None, seed)
               if case["temperature"] else SamplingConfig.greedy())
        return {"case": case, "sampler": Sampler(cfg, torch.device(DEVICE)), "logits": logits,
                "requests": list(range(case["batch"])), "steps": [seed % 97 + i for i in range(case["batch"])]}
    cfg = config_from_dict(_config(case["model"]))
    model = model_from_tensors(cfg, weights(case, seed), case["dtype"], DEVICE)
    prompts, after = _tokens(case, seed, gen)
    window = SHAPES.get(case["model"], {}).get("sliding_window")
    room = {"decode": ROOM, "replay": case.get("new", 0)}.get(case["task"], 0)
    need = sum(round_up(min(len(p) + room, window) if window else len(p) + room) + PAGE for p in prompts)
    engine = Engine(model, max_tokens=need, max_slots=case["batch"])
    state = {"case": case, "engine": engine, "prompts": prompts, "after": after, "pass": 0}
    if case["task"] == "decode":
        state["slots"] = [engine.alloc() for _ in prompts]
        todo = [(s, p[i:i + 4096]) for s, p in zip(state["slots"], prompts) for i in range(0, len(p), 4096)]
        while todo:                                  # steps of up to 8,192 rows, a request at most once in each
            step, rows, later, seen = [], 0, [], set()
            for s, part in todo:
                if s not in seen and rows + len(part) <= 8192:
                    step.append(SeqInput(s, part, []))
                    rows += len(part)
                else:
                    later.append((s, part))
                seen.add(s)
            engine.step(step)
            todo = later
    return state


def _rows(case, logits):
    """The logits of the requests that `exact` covers, and the others'."""
    k = _checked(case)
    out = {"first": logits[:k], "rest": logits[k:]}
    return {name: t for name, t in out.items() if t.shape[0]}


def run(state):
    case, engine = state["case"], state.get("engine")
    if case["task"] == "sample":
        return np.asarray(state["sampler"].sample(state["logits"], state["requests"], state["steps"]))
    if case["task"] == "decode":
        tokens = state["after"][state["pass"] % len(state["after"])]
        state["pass"] += 1
        return _rows(case, engine.step([SeqInput(s, [t], [0]) for s, t in zip(state["slots"], tokens)]))
    slots = [engine.alloc() for _ in state["prompts"]]
    logits = engine.step([SeqInput(s, p, [len(p) - 1]) for s, p in zip(slots, state["prompts"])])
    if case["task"] == "replay":
        steps = [logits.clone()]                     # (a step's logits are overwritten by the next)
        for tokens in state["after"][:case["new"]]:
            steps.append(engine.step([SeqInput(s, [t], [0]) for s, t in zip(slots, tokens)]).clone())
        logits = torch.stack(steps, dim=1)           # [request, step, V]
    for s in slots:
        engine.free(s)
    return _rows(case, logits)


# ---- what a pass cannot do without ------------------------------------------------------------------------
def _visible(n, before, window):
    """Pairs of a query and a key that it sees: n new positions behind `before` old ones."""
    return sum(min(before + i + 1, window or before + i + 1) for i in range(n))


def _distinct(rows, top, experts):
    """Experts that `rows` rows can be expected to use."""
    return experts * (1.0 - (1.0 - top / experts) ** rows)


def work(case):
    V = VOCAB[case["model"]]
    if case["task"] == "sample":
        return {"bytes": 4.0 * case["batch"] * V, "flops": 0.0}
    lens = lengths(case)
    el = 4 if case["dtype"] == "float32" else 2
    total = {"bytes": 0.0, "flops": 0.0}

    def step(new, before):
        n, B = sum(new), len(new)
        att = lambda heads, d, window=None: 4.0 * heads * d * sum(_visible(a, b, window) for a, b in zip(new, before))  # noqa: E731
        # keys and values written, and those in the cache read
        kv = lambda nkv, d, window=None: el * 2.0 * nkv * d * sum(a + min(b, window or b) for a, b in zip(new, before))  # noqa: E731
        flops, nbytes = 2.0 * B * V * _width(case), el * V * _width(case) + el * n * _width(case) + 4.0 * B * V
        for kind, w, w_top, w_each, heads, d, nkv, window, state in _layers(case["model"]):
            flops += 2.0 * n * (w + w_top) + (att(heads, d, window) if kind == "attention" else 4.0 * n * state)
            nbytes += el * (w + w_each * _distinct(n, 4, 16))
            nbytes += kv(nkv, d, window) if kind == "attention" else 2 * 4.0 * B * state
        total["flops"] += flops
        total["bytes"] += nbytes

    if case["task"] == "decode":
        step([1] * len(lens), lens)
    else:
        step(lens, [0] * len(lens))
    for i in range(case.get("new", 0)):
        step([1] * len(lens), [l + i for l in lens])
    return total


def _width(case):
    return SHAPES[case["model"]]["hidden_size"] if case["model"] in SHAPES else 4096


def _layers(model):
    """A layer's (kind, weight elements that every row is multiplied by, those of its chosen experts, those of one
    expert, heads, head size, KV heads, window, elements of a sequence's state)."""
    if model in SHAPES:
        s = SHAPES[model]
        H, d, nq, nkv = s["hidden_size"], s["head_dim"], s["num_attention_heads"], s["num_key_value_heads"]
        w = (2 * nq + 2 * nkv) * d * H + 3 * s["intermediate_size"] * H
        return [("attention", w, 0, 0, nq, d, nkv, s["sliding_window"], 0)] * s["num_hidden_layers"]
    out, H = [], 4096
    for layer in _design(model)["layers"]:
        m, f, kind = layer["mixer"], layer["mlp"], layer["type"]
        if kind == "mamba2":
            inner, GN = m["heads"] * m["vdim"], m["groups"] * m["state"]
            w, state = (2 * inner + 2 * GN + m["heads"]) * H + H * inner, inner * m["state"]
        elif kind == "mingru":
            w, state = 4 * m["width"] * H, m["width"]
        else:
            own = 0 if "kv_from" in m else 2 * 8 * 128 * H
            w, state = 2 * 4096 * H + own + (4096 * H if model == "nepisun" and kind == "attention" else 0), 0
        wide = 3 if model == "giforax" else 2
        if f["kind"] == "dense":
            w, top, each = w + 3 * f["ff"] * H, 0, 0
        else:
            each = wide * f["expert"]["ff"] * H
            w, top = w + wide * f["shared"]["ff"] * H + 16 * H, 4 * each
        out.append(("state" if state else "attention", w, top, each, 32, 128, 0 if "kv_from" in m else 8,
                    m.get("mask", {}).get("size"), state))
    return out


def tolerance(case):
    """bfloat16: activations are rounded to 8 bits at every product's input, which leaves 0.7 to 1 % against 64 bits
    through 32 layers and 0.07 to 0.25 % through the designs' four; 32 bits: the order of the sums (5e-6
    against 64 bits).  Tokens drawn are the same."""
    if case["task"] == "sample":
        return "exact"
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 0.03, "max": 0.3} if case["model"] in SHAPES else {"rel": 0.01, "max": 0.1}


# ---- the same in 64 bits, from the designs' equations -------------------------------------------------------
def _rms(t, eps, w=None):
    y = t / torch.sqrt((t * t).mean(dim=-1, keepdim=True) + eps)
    return y if w is None else y * w


def _layer_norm(t, eps, w, b):
    return torch.nn.functional.layer_norm(t, t.shape[-1:], w, b, eps)


def _rotate(t, base, dims):
    """t [T, heads, d]: channel i < dims / 2 pairs with i + dims / 2, angle position * base^(-2 i / dims)."""
    half = dims // 2
    f = torch.pow(torch.tensor(base, dtype=F64, device=t.device), -2.0 * torch.arange(half, dtype=F64, device=t.device) / dims)
    a = torch.arange(t.shape[0], dtype=F64, device=t.device)[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = t[..., :half], t[..., half:dims]
    return torch.cat([u * c - v * s, v * c + u * s, t[..., dims:]], dim=-1)


def _attend(q, k, v, scale, sees, weigh):
    """q [T, H, d], k and v [T, G, d]; `sees(p, j)`: is key j visible to position p; `weigh(scores, visible, heads)`."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty_like(q)
    j = torch.arange(T, device=q.device)
    rep = H // G
    for p0 in range(0, T, 1024):
        p = torch.arange(p0, min(T, p0 + 1024), device=q.device)
        ok = sees(p[:, None], j[None, :])
        for g in range(G):
            hs = slice(g * rep, (g + 1) * rep)
            s = torch.matmul(q[p0:p0 + 1024, hs].transpose(0, 1), k[:, g].t().contiguous()) * scale     # [rep, rows, T]
            out[p0:p0 + 1024, hs] = torch.matmul(weigh(s, ok, hs), v[:, g].contiguous()).transpose(0, 1)
    return out


def _softmax(s, ok, hs):
    return torch.softmax(s.masked_fill(~ok, -math.inf), dim=-1)


def _softmax_plus_one(s, ok, hs):
    s = s.masked_fill(~ok, -math.inf)
    m = s.amax(dim=-1, keepdim=True).clamp(min=0.0)
    e = torch.exp(s - m)
    return e / (e.sum(dim=-1, keepdim=True) + torch.exp(-m))


def _causal(p, j, window=None, keep=0):
    ok = j <= p
    return ok & ((p - j < window) | (j < keep)) if window else ok


def _mistral_exact(s, w, ids):
    """Logits [len(ids), V] at every id list's last position or positions: a list of (ids, rows wanted)."""
    H, d, nq, nkv, eps, win = (s["hidden_size"], s["head_dim"], s["num_attention_heads"], s["num_key_value_heads"],
                               s["rms_norm_eps"], s["sliding_window"])
    xs = [w("model.embed_tokens.weight")[torch.tensor(i, device=DEVICE)] for i, _ in ids]
    for l in range(s["num_hidden_layers"]):
        p = f"model.layers.{l}."
        q_, k_, v_, o_ = (w(p + f"self_attn.{n}_proj.weight") for n in "qkvo")
        n1, n2 = w(p + "input_layernorm.weight"), w(p + "post_attention_layernorm.weight")
        for i, x in enumerate(xs):
            y = _rms(x, eps, n1)
            T = y.shape[0]
            q, k = _rotate((y @ q_.T).view(T, nq, d), s["rope_theta"], d), _rotate((y @ k_.T).view(T, nkv, d), s["rope_theta"], d)
            a = _attend(q, k, (y @ v_.T).view(T, nkv, d), d ** -0.5, lambda p, j: _causal(p, j, win), _softmax)
            xs[i] = x + a.reshape(T, nq * d) @ o_.T
        del q_, k_, v_, o_
        g_, u_, d_ = (w(p + f"mlp.{n}_proj.weight") for n in ("gate", "up", "down"))
        for i, x in enumerate(xs):
            for r in range(0, x.shape[0], 4096):
                y = _rms(x[r:r + 4096], eps, n2)
                x[r:r + 4096] += (torch.nn.functional.silu(y @ g_.T) * (y @ u_.T)) @ d_.T
        del g_, u_, d_
    head = w("lm_head.weight")
    return [_rms(x[-rows:], eps, w("model.norm.weight")) @ head.T for x, (_, rows) in zip(xs, ids)]


def _experts(h, w, p, chosen_weight, expert, shared):
    y = shared(h, p + "shared.")
    for e in range(16):
        rows = chosen_weight[:, e].nonzero().flatten()
        if len(rows):
            y[rows] += expert(h[rows], chosen_weight[rows, e:e + 1], f"{p}e{e}.")
    return y


def _nepisun_exact(w, ids):
    cfg, eps, out = _design("nepisun"), 1e-6, []
    for toks, rows in ids:
        x = w("embed")[torch.tensor(toks, device=DEVICE)]
        T, first = x.shape[0], None
        for i, layer in enumerate(cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = _rms(x, eps, w(f"l{i}.norm1"))
            if layer["type"] == "mamba2":
                x = x + _state_space_exact(h, w, p, m, eps)
            else:
                windowed = layer["type"] == "attention_2"
                q, k, v = ((h @ w(p + n).T + (w(p + n + ".b") if windowed else 0.0)).view(T, -1, 128) for n in "qkv")
                if not windowed:
                    q, k = _rms(q, eps, w(p + "q.norm")), _rms(k, eps, w(p + "k.norm"))
                q, k = _rotate(q, 1e4, 128), _rotate(k, 1e4, 128)
                if first is None:
                    first = v
                else:
                    v = (1.0 - w(p + "vmix")) * v + w(p + "vmix") * first
                win, keep = (4096, 64) if windowed else (None, 0)
                a = _attend(q, k, v, m["scale"], lambda a, b: _causal(a, b, win, keep),
                            _softmax if windowed else _softmax_plus_one).reshape(T, 4096)
                x = x + (a @ w(p + "o").T + w(p + "o.b") if windowed else (a * torch.sigmoid(h @ w(p + "g").T)) @ w(p + "o").T)
            h, p = _rms(x, eps, w(f"l{i}.norm2")), f"l{i}.mlp."
            if layer["mlp"]["kind"] == "dense":
                x = x + (torch.relu(h @ w(p + "gate").T) * (h @ w(p + "up").T)) @ w(p + "down").T
                continue
            s = torch.softmax(h @ w(p + "router").T, dim=-1)
            best = s.view(T, 4, 4).amax(dim=-1)
            allowed = torch.zeros_like(best).scatter_(1, best.topk(2).indices, 1.0).repeat_interleave(4, dim=1)
            top = (s * allowed).topk(4)
            wt = torch.zeros_like(s).scatter_(1, top.indices, top.values)

            def small(h, p):
                return torch.relu(h @ w(p + "up").T) ** 2 @ w(p + "down").T
            x = x + _experts(h, w, p, wt, lambda h, g, p: g * small(h, p), small)
        out.append(_rms(x[-rows:], eps, w("final.norm")) @ w("embed").T)
    return out


def _state_space_exact(h, w, p, m, eps):
    T, Hd, dv, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
    inner, per = Hd * dv, Hd // G
    proj = h @ w(p + "in").T
    z, u, dt = proj[:, :inner], proj[:, inner:-Hd], proj[:, -Hd:]
    conv = w(p + "conv")
    padded = torch.cat([torch.zeros_like(u[:m["conv"] - 1]) if T >= m["conv"] - 1 else
                        torch.zeros((m["conv"] - 1, u.shape[1]), dtype=F64, device=DEVICE), u])
    u = torch.nn.functional.silu(sum(padded[j:j + T] * conv[:, j] for j in range(m["conv"])) + w(p + "conv.b"))
    xs, Bm, Cm = u[:, :inner].view(T, Hd, dv), u[:, inner:inner + G * N].view(T, G, N), u[:, inner + G * N:].view(T, G, N)
    dt = torch.nn.functional.softplus(dt + w(p + "dt_bias"), threshold=1e9)
    decay = torch.exp(-torch.exp(w(p + "A_log")) * dt).view(T, G, per, 1, 1)
    xdt = (xs * dt[:, :, None]).view(T, G, per, 1, dv)
    S = torch.zeros((G, per, N, dv), dtype=F64, device=DEVICE)
    y = torch.empty((T, Hd, dv), dtype=F64, device=DEVICE)
    for t in range(T):
        S = torch.addcmul(S * decay[t], Bm[t].view(G, 1, N, 1), xdt[t])
        y[t] = torch.matmul(Cm[t].view(G, 1, 1, N), S).view(Hd, dv)
    y = (y + w(p + "D")[:, None] * xs).reshape(T, inner) * torch.nn.functional.silu(z)
    return (_rms(y.view(T, m["norm_groups"], -1), eps).reshape(T, inner) * w(p + "norm")) @ w(p + "o").T


def _giforax_exact(w, ids):
    cfg, eps, out = _design("giforax"), 1e-6, []

    def norm(t, name):
        return _layer_norm(t, eps, w(name), w(name + ".b"))

    def expert(h, p):
        g, u = torch.clamp(h @ w(p + "gate").T, max=7.0), torch.clamp(h @ w(p + "up").T, min=-7.0, max=7.0)
        return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w(p + "down").T

    for toks, rows in ids:
        x = w("embed")[torch.tensor(toks, device=DEVICE)]
        T, results, kept = x.shape[0], [x], {}
        for i, layer in enumerate(cfg["layers"]):
            p, m = f"l{i}.mix.", layer["mixer"]
            h = norm(x, f"l{i}.norm1")
            if layer["type"] == "attention":
                src = m.get("kv_from", i)
                if src == i:
                    kept[i] = (_rms(_rotate((h @ w(p + "k").T).view(T, 8, 128), 1e4, 64), eps), (h @ w(p + "v").T).view(T, 8, 128))
                q = _rms(_rotate((h @ w(p + "q").T).view(T, 32, 128), 1e4, 64), eps)
                pb = w(p + "pb")
                a = _attend(q, *kept[src], m["scale"], lambda a, b: (b <= a) & (a // 4096 == b // 4096),
                            lambda s, ok, hs: torch.sigmoid(s + pb[hs, None, None]) * ok)
                y = (a * torch.sigmoid(h @ w(p + "g").T)[:, :, None]).reshape(T, 4096) @ w(p + "o").T
            else:
                z, c = torch.sigmoid(h @ w(p + "z").T + w(p + "z.b")), h @ w(p + "x").T + w(p + "x.b")
                c = torch.where(c >= 0, c + 0.5, torch.sigmoid(c))
                S, states = torch.zeros_like(z[0]), []
                for t in range(T):
                    S = torch.lerp(S, c[t], z[t])
                    states.append(S)
                y = (torch.stack(states) * torch.nn.functional.silu(h @ w(p + "g").T)) @ w(p + "o").T
            x = x + norm(y, f"l{i}.norm1b")
            h, p = norm(x, f"l{i}.norm2"), f"l{i}.mlp."
            top = torch.sigmoid(h @ w(p + "router").T).topk(4)
            wt = torch.zeros((T, 16), dtype=F64, device=DEVICE).scatter_(1, top.indices, top.values)
            y = _experts(h, w, p, wt, lambda h, g, p: expert(h * g, p), expert)
            x = x + norm(y, f"l{i}.norm2b")
            results.append(x)
            mix = w(f"l{i}.dwa")
            x = sum(mix[j] * results[j] for j in range(i + 2))
        out.append(norm(x[-rows:], "final.norm") @ w("head").T)
    return out


def exact(case, seed):
    k = 0 if case["task"] == "sample" else _checked(case)
    if not k:
        return None
    stored = weights(case, seed)
    prompts, after = _tokens(case, seed, torch.Generator().manual_seed(seed))
    new = {"decode": 1, "replay": case.get("new", 0)}.get(case["task"], 0)
    ids = [(prompts[b] + [after[t][b] for t in range(new)], new + 1 if case["task"] == "replay" else 1) for b in range(k)]

    def w(name):
        return stored[name].to(F64)

    if case["model"] in SHAPES:
        logits = _mistral_exact(SHAPES[case["model"]], w, ids)
    else:
        logits = (_nepisun_exact if case["model"] == "nepisun" else _giforax_exact)(w, ids)
    first = torch.stack(logits) if case["task"] == "replay" else torch.cat(logits)
    return {"first": first, "rest": None} if k < case["batch"] else {"first": first}
