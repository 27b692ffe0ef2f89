"""The engine's work as its users give it, as a list of cases that can be timed and checked.

A pass of a case answers a batch of requests through `Engine.step`: prompts come in portions under
a token budget beside the decode tokens of the requests that are further on (the order in which
the scheduler forms its steps), every request then takes the tokens that follow its prompt one a
step, and leaves with its last.  The tokens are given and not drawn, as in a replay of a trace, so
that two implementations see the same inputs in every step; the logits of every place a token
would be drawn from come back.  A case that draws has the device draw from those logits as well.

The models have the sizes of the served shapes that the benchmarks name: the Qwen3 shapes at full
depth where three states fit the card side by side (at fewer layers the 14B and 32B widths), the
six other architectures at their benchmark's sizes.  Weights are random with the scales that
trained models show: a residual stream that outweighs what a layer adds, output projections that shrink with the
depth, decays that remember.
"""
from __future__ import annotations

import math
import zlib
from typing import Dict, List, Optional, Tuple

import numpy as np
import torch

DEVICE = "cuda:0"
PAGE = 16
VOCAB = 32768                       # of the six smaller architectures' shapes
MAX_POSITIONS = 40960


# --------------------------------------------------------------------------- the models' sizes
def _qwen3(layers, hidden, heads, inter, tied=False):
    return dict(architectures=["Qwen3ForCausalLM"], model_type="qwen3", num_hidden_layers=layers,
                hidden_size=hidden, num_attention_heads=heads, num_key_value_heads=8,
                head_dim=128, intermediate_size=inter, vocab_size=151936, rope_theta=1000000.0,
                rms_norm_eps=1e-6, tie_word_embeddings=tied, max_position_embeddings=MAX_POSITIONS,
                torch_dtype="bfloat16")


QWEN3 = {"qwen3-0.6b": (28, 1024, 16, 3072, True), "qwen3-1.7b": (28, 2048, 16, 6144, True),
         "qwen3-4b": (36, 2560, 32, 9728, True), "qwen3-8b": (36, 4096, 32, 12288),
         "qwen3-14b": (40, 5120, 40, 17408), "qwen3-32b": (64, 5120, 64, 25600)}


def _fezupel(layers, width, heads, kv, dim, window, experts, top, ff, shared):
    layer = {"type": "attention",
             "mixer": {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim,
                       "scale": dim ** -0.5, "mask": {"size": window}},
             "mlp": {"kind": "moe", "router": {"experts": experts, "top": top},
                     "expert": {"ff": ff, "limit": 7.0}, "shared": {"ff": shared, "limit": 7.0}}}
    return {"architecture": "Fezupel", "vocab": VOCAB, "width": width, "max_positions": 4096,
            "norm": {"eps": 1e-6}, "layers": [layer] * layers}


def _lodenex(layers, kinds):
    layer = {
        "attention": {
            "mixer": {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                      "softcap": 30.0, "mask": {"size": 8192},
                      "rot": {"base": 500000.0, "dims": 64, "scaling": {
                          "factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}}},
        "latent_attention": {
            "mixer": {"heads": 32, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 1536,
                      "kv_rank": 128, "scale": 192 ** -0.5, "mask": {"size": 4096},
                      "rot": {"base": 1000000.0, "dims": 64, "scaling": {
                          "factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}}
    return {"architecture": "Lodenex", "vocab": VOCAB, "width": 4096, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0}, "logit_softcap": 30.0,
            "layers": [{"type": kinds[i % len(kinds)], "mlp": {"kind": "dense", "ff": 16384},
                        **layer[kinds[i % len(kinds)]]} for i in range(layers)]}


def _nupovik(layers):
    wkv = {"type": "wkv", "mixer": {"heads": 32, "dim": 64}, "mlp": {"kind": "dense", "ff": 7168}}
    gla = {"type": "gla", "mixer": {"heads": 8, "dim": 128, "vdim": 256, "tau": 16.0},
           "mlp": {"kind": "dense", "ff": 7168}}
    return {"architecture": "Nupovik", "vocab": VOCAB, "width": 2048, "norm": {"eps": 1e-6},
            "logit_scale": 1.0, "loop": None, "layers": [(wkv, gla)[i % 2] for i in range(layers)]}


def _kugisun(layers, width, heads, kv, r_kv, dense, outputs, top, ff, shared):
    mixer = {"left": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128,
                      "scale": 128 ** -0.5, "rot": {"dims": 64, "base": 1000000.0}},
             "right": {"heads": heads, "kv_heads": r_kv, "dim": 128, "vdim": 128, "conv": 4},
             "left_scale": 0.75, "right_scale": 1.25}
    moe = {"kind": "moe", "expert": {"ff": ff}, "shared": {"ff": shared},
           "router": {"experts": outputs - 2, "identity": 2, "top": top, "scale": 2.5,
                      "groups": {"count": 8, "keep": 4}}}
    plain = {"kind": "dense", "ff": dense}
    return {"architecture": "Kugisun", "vocab": VOCAB, "width": width, "max_positions": 4096,
            "streams": 4, "norm": {"eps": 1e-6},
            "layers": [{"type": "parallel", "mixer": mixer, "mlp": moe if i else plain}
                       for i in range(layers)]}


def _fumanex(layers, width, heads, kv, ff):
    attention = dict(heads=heads, kv_heads=kv, dim=128, vdim=128, scale=128 ** -0.5, softcap=30.0,
                     bias_max=256, v_mix=True, mask=dict(size=1024, keep_first=4))

    def recurrent(n, dim, **more):
        return dict(heads=n, dim=dim, vdim=dim, **more,
                    decay=[1.0 - 2.0 ** (-4.0 - 5.0 * i / (n - 1)) for i in range(n)])
    kinds = [("attention", attention),
             ("retention", recurrent(heads, 128, rot=dict(dims=128, base=10000.0))),
             ("lightning", recurrent(2 * heads, 64))]
    return {"architecture": "Fumanex", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-6},
            "embedding": {"scale": 1.0}, "logit_scale": 1.0,
            "layers": [{"type": k, "mixer": m, "mlp": {"kind": "dense", "ff": ff}}
                       for k, m in (kinds[i % 3] for i in range(layers))]}


def _tigesun(layers, width, heads, kv, ff, groups):
    attention = dict(heads=heads, kv_heads=kv, dim=128, vdim=128, scale=128 ** -0.5,
                     rot=dict(base=10000.0, dims=128,
                              scaling=dict(factor=8.0, original=4096, fast=32.0, slow=1.0)))
    latent = dict(heads=heads, dim=128, vdim=128, kv_rank=128, scale=128 ** -0.5,
                  mask=dict(size=1024))
    space = dict(heads=4 * heads, vdim=64, state=128, groups=groups, conv=4, norm_groups=groups)
    kinds = [("attention", attention), ("mamba2", space), ("latent_attention", latent),
             ("mamba2", space)]
    return {"architecture": "Tigesun", "vocab": VOCAB, "width": width, "norm": {"eps": 1e-6},
            "logit_softcap": 30.0,
            "layers": [{"type": k, "mixer": m,
                        "mlp": None if k == "mamba2" else {"kind": "dense", "ff": ff}}
                       for k, m in (kinds[i % 4] for i in range(layers))]}


SMALLER = {
    "fezupel": lambda n: _fezupel(n, 2048, 16, 4, 128, 2048, 32, 4, 768, 1024),
    "fezupel-medium": lambda n: _fezupel(n, 4096, 32, 8, 128, 2048, 64, 8, 1024, 2048),
    "fezupel-narrow-heads": lambda n: _fezupel(n, 3072, 32, 8, 96, 1024, 16, 2, 2048, 2048),
    "lodenex": lambda n: _lodenex(n, ("attention", "attention", "latent_attention", "attention")),
    "lodenex-latent": lambda n: _lodenex(n, ("latent_attention",)),
    "nupovik": _nupovik,
    "kugisun": lambda n: _kugisun(n, 2048, 16, 4, 8, 5632, 32, 4, 1024, 1536),
    "kugisun-wide": lambda n: _kugisun(n, 4096, 32, 8, 16, 11264, 64, 6, 1536, 2048),
    "fumanex": lambda n: _fumanex(n, 2048, 16, 4, 8192),
    "fumanex-wide": lambda n: _fumanex(n, 4096, 32, 8, 16384),
    "tigesun": lambda n: _tigesun(n, 2048, 16, 4, 8192, 1),
    "tigesun-wide": lambda n: _tigesun(n, 4096, 32, 8, 14336, 8),
}


def _raw(case) -> dict:
    if case["model"] in QWEN3:
        sizes = QWEN3[case["model"]]
        return _qwen3(case["layers"], *sizes[1:])
    return SMALLER[case["model"]](case["layers"])


# --------------------------------------------------------------------------- the cases
def _case(name, model, layers, requests, prompt, new, budget=2048, dtype="bfloat16", draw=False):
    case = dict(model=model, layers=layers, requests=requests, prompt=prompt, new=new,
                budget=budget, dtype=dtype, draw=draw)
    return dict(case, name=name) if name else case


def listed() -> List[dict]:
    return [
        # one user of the smallest shape: a short prompt and a short answer, launches and latency
        _case("0.6b-one-user", "qwen3-0.6b", 28, 1, 61, 32),
        # one user of the served shape: a middling prompt, then one token after the other
        _case("8b-one-user", "qwen3-8b", 36, 1, 512, 48),
        # a handful of users: ragged prompts of 512 tokens on average, 64 tokens each
        _case("8b-eight-users", "qwen3-8b", 36, 8, 512, 64),
        # a busy server: 64 short ragged prompts, 48 tokens each
        _case("8b-64-users", "qwen3-8b", 36, 64, 96, 48),
        # the headline prompt, read and answered with its first token
        _case("8b-prompt-2048", "qwen3-8b", 36, 1, 2048, 1),
        # a long document on the largest shape's widths, in one portion
        _case("32b-prompt-8191", "qwen3-32b", 8, 1, 8191, 1, budget=8192),
        # continuous batching: portions of 512 tokens beside the others' decode tokens
        _case("14b-continuous", "qwen3-14b", 10, 24, 800, 24, budget=512),
        # the 32-bit path, with a token drawn on the device behind every step
        _case("0.6b-float32-drawn", "qwen3-0.6b", 28, 4, 96, 12, budget=256, dtype="float32",
              draw=True),
        # a mixture of experts behind attention whose values are its keys
        _case("fezupel-eight-users", "fezupel", 4, 8, 512, 32),
        # attention beside a delta rule, four streams, a mixture of experts
        _case("kugisun-eight-users", "kugisun", 4, 8, 512, 32),
        # the state space between grouped-query and latent attention
        _case("tigesun-wide-eight-users", "tigesun-wide", 4, 8, 512, 32),
        # recurrences with a fixed-size memory alone
        _case("nupovik-16-users", "nupovik", 4, 16, 256, 32),
    ]


def _spread(rng, lo, hi) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng) -> dict:
    """A case of the listed ones' ranges: any of the models, from one request to 64, prompts from
    a few tokens to thousands, answers of one token to 64, every step's budget in use."""
    while True:
        if rng.random() < 0.5:
            model = rng.choice(list(QWEN3))
            layers = QWEN3[model][0]
            if model in ("qwen3-14b", "qwen3-32b"):
                layers = rng.randint(2, 10 if model == "qwen3-14b" else 8)
            longest = 8191
        else:
            model = rng.choice(list(SMALLER))
            layers = rng.randint(3, 6)
            longest = 2000
        requests = _spread(rng, 1, 64)
        prompt = _spread(rng, 5, longest)
        new = 1 if rng.random() < 0.2 else _spread(rng, 2, 64)
        if model not in QWEN3 and prompt + prompt // 2 + new > 3000:
            continue
        dtype = "float32" if model in ("qwen3-0.6b", "nupovik", "fezupel") \
            and rng.random() < 0.25 else "bfloat16"
        case = _case(None, model, layers, requests, prompt, new,
                     budget=rng.choice((512, 1024, 2048, 4096)), dtype=dtype,
                     draw=dtype == "float32" and rng.random() < 0.5)
        if _cost(case) <= max(_cost(c) for c in listed()) \
                and _work_size(case) <= max(_work_size(c) for c in listed()):
            return case


# --------------------------------------------------------------------------- what a pass runs
def _lengths(case) -> List[int]:
    """The prompts' lengths: one request has the case's, several lie between half of it and one
    and a half times, in no order."""
    n, p = case["requests"], case["prompt"]
    if n == 1:
        return [p]
    return [max(1, p // 2 + p * ((i * 7 + 3) % n) // max(1, n - 1)) for i in range(n)]


def _plan(case) -> List[List[Tuple[int, int, int]]]:
    """The steps: per step (request, first token, behind its last), decode tokens before portions
    of prompts, at most ``budget`` tokens a step."""
    lens = _lengths(case)
    total = [n + case["new"] - 1 for n in lens]
    done = [0] * len(lens)
    steps = []
    while any(d < t for d, t in zip(done, total)):
        room, step = case["budget"], []
        for i, d in enumerate(done):
            if lens[i] <= d < total[i] and room > 0:
                step.append((i, d, d + 1))
                room -= 1
        for i, d in enumerate(done):
            if d < lens[i] and room > 0:
                n = min(room, lens[i] - d)
                step.append((i, d, d + n))
                room -= n
        for i, _, b in step:
            done[i] = b
        steps.append(step)
    return steps


def _tokens(case, seed) -> List[List[int]]:
    rng = np.random.default_rng([int(seed) & 0xFFFFFFFF, 17])
    vocab = 151936 if case["model"] in QWEN3 else VOCAB
    return [rng.integers(0, vocab, n + case["new"] - 1).tolist() for n in _lengths(case)]


# --------------------------------------------------------------------------- weights
def _draw_weight(name, decl, seed, case, tied) -> torch.Tensor:
    """The tensor ``name`` of ``seed`` in 32-bit on the device: every tensor from a stream of its
    own."""
    shape = decl.drawn_shape()
    g = torch.Generator(device=DEVICE)
    g.manual_seed((zlib.crc32(name.encode()) << 31) ^ (int(seed) & 0x7FFFFFFF))
    last = name.rsplit(".", 1)[-1]

    def uniform(lo, hi):
        return torch.rand(shape, generator=g, device=DEVICE) * (hi - lo) + lo

    def normal(std):
        return torch.randn(shape, generator=g, device=DEVICE) * std

    if name in ("embed", "model.embed_tokens.weight"):
        # beside what the layers add: an identity expert's whole row, small ones of narrow shapes
        return normal(4.0 if case["model"].startswith("kugisun") else
                      0.1 if case["model"] in QWEN3 and tied else 1.0)
    if ".hc" in name:                     # several streams: read as a mean, kept as they are
        if last == "in":
            return uniform(0.2, 0.3)
        if last == "mix":
            return normal(0.03) + 0.9 * torch.eye(shape[0], device=DEVICE)
        return uniform(0.8, 1.2)
    if last == "A_log":                   # decays of 1 to 16 a unit of step size
        return torch.log(uniform(1.0, 16.0))
    if last == "dt_bias":                 # step sizes of 0.001 to 0.1 behind the softplus
        return torch.log(torch.expm1(torch.exp(uniform(math.log(1e-3), math.log(0.1)))))
    if last == "D":
        return uniform(0.9, 1.1)
    if last == "conv" and len(shape) == 2:
        return uniform(-0.5, 0.5)
    if last == "w0":                      # decays exp(-exp(.)) from 0.7 to 0.998
        return uniform(-6.0, -1.0)
    if ".mu." in name:
        return uniform(0.0, 1.0)
    if last in ("u", "rel", "sink"):
        return normal(0.5)
    if last == "vmix":
        return uniform(0.4, 0.6)
    if last == "router":                  # logits of the scale their soft-max is trained to: among
        sharp = case["model"].startswith("fezupel")          # the chosen alone, or over all outputs
        return normal((6.0 if sharp else 1.0) / math.sqrt(shape[1]))
    if decl.init == "gain":
        return uniform(0.9, 1.1)
    if last in ("o", "down") or name.endswith(("o_proj.weight", "down_proj.weight")):
        return normal(0.02 / math.sqrt(2 * case["layers"]))
    return normal(0.02)


class _Weights(dict):
    """A model's tensors by name, drawn when they are asked for and not kept."""

    def __init__(self, case, seed, decls, tied, head_name):
        super().__init__({n: d for n, d in decls.items()
                          if not (tied and n == head_name and d.optional)})
        self.case, self.seed, self.tied = case, seed, tied
        self.store = torch.float32 if case["dtype"] == "float32" else torch.bfloat16

    def __getitem__(self, name):
        t = _draw_weight(name, super().__getitem__(name), self.seed, self.case, self.tied)
        return t.to(self.store)

    def items(self):
        return ((n, self[n]) for n in self)

    def values(self):
        return (self[n] for n in self)

    def get(self, name, default=None):
        return self[name] if name in self else default


def _spec(case):
    from zinfer_amd.config import entry_for
    raw = _raw(case)
    return entry_for(raw).config_type.from_dict(raw).model_spec()


def _weights(case, seed, spec) -> _Weights:
    from zinfer_amd.models.build import declare_tensors
    return _Weights(case, seed, declare_tensors(spec), spec.tie_word_embeddings, spec.head_name)


# --------------------------------------------------------------------------- a pass
class State:
    pass


def prepare(case, seed):
    """A bound model, an engine with room for every request at once, the steps' entries and a
    buffer for the logits."""
    from zinfer_amd.engine import Engine, StepEntry
    from zinfer_amd.models.build import build_model
    spec = _spec(case)
    model = build_model(spec, _weights(case, seed, spec), case["dtype"], DEVICE)
    lens, tokens = _lengths(case), _tokens(case, seed)
    pages = sum((len(t) + PAGE - 1) // PAGE + 1 for t in tokens) + 8
    s = State()
    s.engine = Engine(model, page_size=PAGE, num_pages=pages, max_requests=max(64, len(lens)))
    s.steps, n = [], 0
    rng = np.random.default_rng([int(seed) & 0xFFFFFFFF, 23])
    for step in _plan(case):
        entries, end, wanted = [], [], 0
        for i, a, b in step:
            want = [b - a - 1] if b >= lens[i] else []
            wanted += len(want)
            entries.append(StepEntry(i, tokens[i][a:b], want))
            if b == len(tokens[i]):
                end.append(i)
        records = None
        if case["draw"] and wanted:
            from zinfer_amd.ops import SAMPLE_ROW_DTYPE
            records = np.zeros((wanted,), dtype=SAMPLE_ROW_DTYPE)
            records["temperature"], records["top_p"], records["top_k"] = 0.8, 1.0, 50
            records["u"] = rng.random(wanted)
        s.steps.append((entries, end, n, wanted, records))
        n += wanted
    s.logits = torch.empty((n, spec.vocab_size), dtype=torch.float32, device=DEVICE)
    s.drawn = case["draw"]
    return s


def run(s):
    drawn = []
    for entries, end, at, wanted, records in s.steps:
        logits = s.engine.step(entries, end)
        if wanted:
            s.logits[at:at + wanted].copy_(logits)
            if records is not None:
                drawn += s.engine.sample(logits, records)
    if s.drawn:
        return {"logits": s.logits, "tokens": torch.tensor(drawn, dtype=torch.int64)}
    return {"logits": s.logits}


# --------------------------------------------------------------------------- work and tolerance
def _numbers(case):
    """(numbers in the matrices every token meets, of one expert and how many experts a token and
    a layer have, in all of them; numbers of the head)."""
    from zinfer_amd.models.build import declare_tensors
    spec = _spec(case)
    every, expert, head = 0, 0, spec.vocab_size * spec.hidden_size
    for name, decl in declare_tensors(spec).items():
        shape = decl.drawn_shape()
        if len(shape) < 2 or name in ("embed", "pos", "head", "lm_head.weight",
                                      "model.embed_tokens.weight"):
            continue
        if ".mlp.e" in name:
            expert += shape[0] * shape[1]
        else:
            every += shape[0] * shape[1]
    return every, expert, head


def _attention_costs(case):
    """Per layer: (numbers of a cached token, operations a pair of query and key, window)."""
    raw = _raw(case)
    if case["model"] in QWEN3:
        kv, hd = raw["num_key_value_heads"], raw["head_dim"]
        return [(2 * kv * hd, 4 * raw["num_attention_heads"] * hd, None)] * case["layers"]
    out = []
    for layer in raw["layers"]:
        m = layer["mixer"].get("left", layer["mixer"])
        if layer["type"] not in ("attention", "latent_attention", "parallel"):
            continue
        if "kv_rank" in m:
            row = m["kv_rank"] + m.get("rot_dim", 0)
        else:
            row = m["kv_heads"] * (m["dim"] + (0 if raw["architecture"] == "Fezupel" else m["vdim"]))
        out.append((row, 2 * m["heads"] * (m["dim"] + m.get("rot_dim", 0) + m["vdim"]),
                    (m.get("mask") or {}).get("size")))
    return out


def _state_costs(case) -> List[Tuple[int, int]]:
    """Per layer with a state: (numbers of a request's state, operations a token)."""
    if case["model"] in QWEN3:
        return []
    out = []
    for layer in _raw(case)["layers"]:
        m = layer["mixer"].get("right", layer["mixer"])
        if layer["type"] in ("attention", "latent_attention"):
            continue
        n = m["heads"] * m.get("vdim", m.get("dim")) * m.get("state", m.get("dim", 0))
        out.append((n, 4 * n))
    return out


def work(case) -> Dict[str, float]:
    """What the steps of a pass cannot do without: every step reads the matrices its tokens meet
    once (an expert's only if a token can have chosen it), the cached rows its queries see once
    and its requests' states, and writes its own rows, states and logits."""
    elem = 4 if case["dtype"] == "float32" else 2
    every, expert, head = _numbers(case)
    raw = _raw(case)
    moes = [L["mlp"] for L in raw.get("layers", []) if (L.get("mlp") or {}).get("kind") == "moe"] \
        if case["model"] not in QWEN3 else []
    experts = moes[0]["router"]["experts"] if moes else 1
    top = moes[0]["router"]["top"] if moes else 1
    attention, states = _attention_costs(case), _state_costs(case)
    lens, width = _lengths(case), raw.get("hidden_size", raw.get("width"))
    vocab = raw.get("vocab_size", raw.get("vocab"))
    n_bytes = n_flops = 0.0
    for step in _plan(case):
        tokens = sum(b - a for _, a, b in step)
        wanted = sum(1 for i, _, b in step if b >= lens[i])
        n_bytes += elem * (every + expert * min(1.0, tokens * top / experts))
        n_bytes += elem * width * tokens + (elem * head if wanted else 0) + 4 * wanted * vocab
        n_flops += 2.0 * tokens * (every + expert * top / experts) + 2.0 * wanted * head
        for row, pair, window in attention:
            for _, a, b in step:
                seen = b if window is None else min(b, window + b - a - 1)
                n_bytes += elem * row * (seen + b - a)
                if window is None:
                    n_flops += pair * ((a + 1 + b) * (b - a) / 2.0)
                else:
                    n_flops += pair * float(np.minimum(np.arange(a + 1, b + 1), window).sum())
        for numbers, operations in states:
            n_bytes += 8 * numbers * len(step)
            n_flops += float(operations) * tokens
    return {"bytes": n_bytes, "flops": n_flops}


def _work_size(case) -> float:
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _cost(case) -> float:
    """Seconds a pass takes, roughly: for keeping drawn cases within the listed ones' range."""
    w = work(case)
    rate = 8e13 if case["dtype"] == "float32" else 7e14
    return w["bytes"] / 4e12 + w["flops"] / rate + 1e-3 * len(_plan(case)) \
        + 2e-7 * sum(b - a for step in _plan(case) for _, a, b in step) * case["layers"]


def tolerance(case):
    """Measured against 64 bits: the bfloat16 path is 0.2 to 0.6 % off (two summation orders of it
    are about as far from each other), 0.8 to 1.0 % with norms around every sublayer or behind a
    router, where a near tie may choose another expert for a token; the 32-bit path 2e-6."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3, "differ": 0.01}
    if case["model"].startswith(("fezupel", "tigesun")):
        return {"rel": 0.03, "max": 0.99}
    return {"rel": 0.02, "max": 0.5}


# --------------------------------------------------------------------------- in 64 bits
F64 = torch.float64


def _lin(h, w, b=None):
    """w stored [out, in]; in pieces, so that a large matrix never exists whole in 64 bits."""
    out = torch.empty((h.shape[0], w.shape[0]), dtype=F64, device=h.device)
    for a in range(0, w.shape[0], 16384):
        out[:, a:a + 16384] = h @ w[a:a + 16384].to(F64).T
    return out if b is None else out + b.to(F64)


def _rms(v, eps, w=None):
    y = v / torch.sqrt((v * v).mean(dim=-1, keepdim=True) + eps)
    return y if w is None else y * w.to(F64)


def _layer_norm(v, w, b, eps):
    d = v - v.mean(dim=-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(dim=-1, keepdim=True) + eps) * w.to(F64) + b.to(F64)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _softplus(z):
    return z.clamp(min=0.0) + torch.log1p(torch.exp(-z.abs()))


def _frequencies(rot):
    """(the pairs' frequencies, the factor on cosine and sine)."""
    base, dims, sc = float(rot["base"]), int(rot["dims"]), rot.get("scaling")
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=F64)
    if not sc:
        return f, 1.0
    factor, original = float(sc["factor"]), float(sc["original"])
    if "low" in sc:                       # by wavelength
        turns = original * f / (2.0 * math.pi)
        blend = ((turns - sc["low"]) / (sc["high"] - sc["low"])).clamp(0.0, 1.0)
        return f * blend + f / factor * (1.0 - blend), 1.0

    def number(turns):                    # by the pair's number
        return dims * math.log(original / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
    lo = max(math.floor(number(sc["fast"])), 0)
    hi = min(math.ceil(number(sc["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=F64) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / factor * ramp + f * (1.0 - ramp), 0.1 * math.log(factor) + 1.0


def _rotate(z, pos, rot, neighbours=False):
    """z [N, heads, d]: pairs (i, i + dims/2), or (2i, 2i + 1), of a head's first elements turned."""
    dims = int(rot["dims"])
    f, length = _frequencies(rot)
    a = pos[:, None] * f.to(z.device)
    c, s = (length * torch.cos(a))[:, None], (length * torch.sin(a))[:, None]
    out = z.clone()
    if neighbours:
        u, v = z[..., 0:dims:2], z[..., 1:dims:2]
        out[..., 0:dims:2], out[..., 1:dims:2] = u * c - v * s, v * c + u * s
    else:
        u, v = z[..., :dims // 2], z[..., dims // 2:dims]
        out[..., :dims // 2], out[..., dims // 2:dims] = u * c - v * s, v * c + u * s
    return out


def _attend(q, k, v, scale, bounds, window=None, chunk=None, keep=0, cap=None, sink=None, bias=None):
    """q [N, H, d], k [N, G, d], v [N, G, dv], sequence by sequence -> [N, H dv].  ``sink`` [H]:
    one more term of the denominator; ``bias`` (T) -> [H, T, T]."""
    H, G = q.shape[1], k.shape[1]
    per = H // G
    out = torch.empty((q.shape[0], H, v.shape[2]), dtype=F64, device=q.device)
    for a, b in bounds:
        T = b - a
        i, j = torch.arange(T, device=q.device)[:, None], torch.arange(T, device=q.device)[None, :]
        seen = j <= i
        if window is not None:
            seen = seen & ((i - j < window) | (j < keep))
        if chunk is not None:
            seen = seen & (i // chunk == j // chunk)
        at = bias(T) if bias is not None else None
        piece = max(1, (1 << 28) // (T * T))          # heads at a time: 2 GiB of scores
        for g in range(G):
            for lo in range(g * per, (g + 1) * per, piece):
                hi = min(lo + piece, (g + 1) * per)
                s = torch.matmul(q[a:b, lo:hi].transpose(0, 1), k[a:b, g].T) * scale
                if cap is not None:
                    s = cap * torch.tanh(s / cap)
                if at is not None:
                    s = s + at[lo:hi]
                s = s.masked_fill(~seen, -math.inf)
                m = s.max(dim=-1, keepdim=True).values
                if sink is not None:
                    last = sink[lo:hi].to(F64)[:, None, None]
                    m = torch.maximum(m, last)
                e = torch.exp(s - m)
                total = e.sum(dim=-1, keepdim=True)
                if sink is not None:
                    total = total + torch.exp(last - m)
                out[a:b, lo:hi] = torch.matmul(e / total, v[a:b, g]).transpose(0, 1)
    return out.reshape(q.shape[0], -1)


class _Rows:
    """Rows of several sequences behind one another, and the same rows padded [B, L, ...]."""

    def __init__(self, bounds, device):
        self.bounds = bounds
        L = max(b - a for a, b in bounds)
        self.shape = (len(bounds), L)
        self.at = torch.cat([torch.arange(b - a, device=device) + i * L
                             for i, (a, b) in enumerate(bounds)])

    def pad(self, x):
        out = torch.zeros((self.shape[0] * self.shape[1],) + x.shape[1:], dtype=F64, device=x.device)
        out[self.at] = x
        return out.view(self.shape + x.shape[1:])

    def flat(self, x):
        return x.reshape((-1,) + x.shape[2:])[self.at]

    def before(self, x, n):
        """The rows n places earlier in their sequence, zeros before its start."""
        p = self.pad(x)
        out = torch.zeros_like(p)
        if n < p.shape[1]:
            out[:, n:] = p[:, :p.shape[1] - n]
        return self.flat(out)

    def conv(self, x, taps):
        n = taps.shape[1]
        return sum(self.before(x, n - 1 - j) * taps[:, j].to(F64) for j in range(n))

    def recur(self, q, k, v, decay, bonus=None, beta=None):
        """q, k [N, H, d], v [N, H, dv]; decay [N, H] or [N, H, d], or [H]; S <- decay S (in between,
        with ``beta``, v - S^T k takes v's place) + k v^T; o = S^T q; with ``bonus`` o is read
        before the decay, with the token's own product times the bonus."""
        q, k, v = self.pad(q), self.pad(k), self.pad(v)
        B, L, H, d = q.shape
        if decay.dim() == 1:
            decay = decay[None, None, :, None].expand(B, L, H, 1)
        else:
            decay = self.pad(decay)
            decay = decay[..., None] if decay.dim() == 3 else decay
        beta = None if beta is None else self.pad(beta)
        S = torch.zeros((B, H, d, v.shape[3]), dtype=F64, device=q.device)
        o = torch.empty((B, L, H, v.shape[3]), dtype=F64, device=q.device)
        for t in range(L):
            if bonus is not None:
                own = (q[:, t] * bonus * k[:, t]).sum(dim=-1, keepdim=True) * v[:, t]
                o[:, t] = torch.matmul(q[:, t, :, None], S)[:, :, 0] + own
            S = S * decay[:, t, :, :, None]
            w = v[:, t]
            if beta is not None:
                w = beta[:, t, :, None] * (w - torch.matmul(k[:, t, :, None], S)[:, :, 0])
            S = S + k[:, t, :, :, None] * w[:, :, None]
            if bonus is None:
                o[:, t] = torch.matmul(q[:, t, :, None], S)[:, :, 0]
        return self.flat(o)


class _Exact:
    """The seven decoders over whole sequences, without a cache, in 64 bits."""

    def __init__(self, case, seed):
        spec = _spec(case)
        self.raw, self.w = _raw(case), _weights(case, seed, spec)
        self.spec, self.case = spec, case
        tokens = _tokens(case, seed)
        self.bounds, n = [], 0
        for t in tokens:
            self.bounds.append((n, n + len(t)))
            n += len(t)
        self.ids = torch.tensor(sum(tokens, []), device=DEVICE)
        self.pos = torch.cat([torch.arange(len(t), device=DEVICE) for t in tokens])
        self.rows = _Rows(self.bounds, DEVICE)
        lens, want = _lengths(case), []
        for step in _plan(case):
            want += [self.bounds[i][0] + b - 1 for i, _, b in step if b >= lens[i]]
        self.want = torch.tensor(want, device=DEVICE)
        self.fposition = self.pos.to(F64)
        self.eps = float(self.raw.get("rms_norm_eps", (self.raw.get("norm") or {}).get("eps", 0)))

    def logits(self):
        if self.case["model"] in QWEN3:
            return self.qwen3()
        return getattr(self, self.raw["architecture"].lower())()

    def embed(self):
        name = "model.embed_tokens.weight" if self.case["model"] in QWEN3 else "embed"
        return self.w[name][self.ids].to(F64)

    def heads(self, y, n):
        return y.view(y.shape[0], n, -1)

    # ---- Qwen3
    def qwen3(self):
        r, w, eps = self.raw, self.w, self.eps
        H, G = r["num_attention_heads"], r["num_key_value_heads"]
        rot = {"base": r["rope_theta"], "dims": r["head_dim"]}
        x = self.embed()
        for i in range(r["num_hidden_layers"]):
            p = f"model.layers.{i}."
            h = _rms(x, eps, w[p + "input_layernorm.weight"])
            a = p + "self_attn."
            q = _rms(self.heads(_lin(h, w[a + "q_proj.weight"]), H), eps, w[a + "q_norm.weight"])
            k = _rms(self.heads(_lin(h, w[a + "k_proj.weight"]), G), eps, w[a + "k_norm.weight"])
            v = self.heads(_lin(h, w[a + "v_proj.weight"]), G)
            o = _attend(_rotate(q, self.fposition, rot), _rotate(k, self.fposition, rot), v,
                        r["head_dim"] ** -0.5, self.bounds)
            x = x + _lin(o, w[a + "o_proj.weight"])
            h = _rms(x, eps, w[p + "post_attention_layernorm.weight"])
            m = p + "mlp."
            x = x + _lin(_silu(_lin(h, w[m + "gate_proj.weight"])) * _lin(h, w[m + "up_proj.weight"]),
                         w[m + "down_proj.weight"])
        x = _rms(x[self.want], eps, w["model.norm.weight"])
        return _lin(x, w["model.embed_tokens.weight" if r["tie_word_embeddings"]
                         else "lm_head.weight"])

    # ---- Fezupel
    def fezupel(self):
        w, eps = self.w, self.eps

        def expert(h, p, limit):
            g = _lin(h, w[p + "gate"]).clamp(max=limit)
            u = _lin(h, w[p + "up"]).clamp(-limit, limit)
            return _lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), w[p + "down"])

        x = self.embed() + w["pos"].to(F64)[self.pos]
        for i, L in enumerate(self.raw["layers"]):
            p, m, f = f"l{i}.", L["mixer"], L["mlp"]
            h = _layer_norm(x, w[p + "norm1"], w[p + "norm1.b"], eps)
            k = self.heads(_lin(h, w[p + "mix.k"]), m["kv_heads"])
            o = _attend(self.heads(_lin(h, w[p + "mix.q"]), m["heads"]), k, k, m["scale"],
                        self.bounds, window=m["mask"]["size"],
                        sink=torch.zeros(m["heads"], device=DEVICE))
            y = _lin(o * torch.sigmoid(_lin(h, w[p + "mix.g"])), w[p + "mix.o"])
            x = x + _layer_norm(y, w[p + "norm1b"], w[p + "norm1b.b"], eps)
            h = _layer_norm(x, w[p + "norm2"], w[p + "norm2.b"], eps)
            value, ids = torch.topk(_lin(h, w[p + "mlp.router"], w[p + "mlp.router.b"]),
                                    f["router"]["top"], dim=-1)
            share = torch.softmax(value, dim=-1)
            y = expert(h, p + "mlp.shared.", f["shared"]["limit"])
            for e in range(f["router"]["experts"]):
                part = (share * (ids == e)).sum(dim=-1, keepdim=True)
                rows = (ids == e).any(dim=-1).nonzero()[:, 0]
                if len(rows):
                    y[rows] += part[rows] * expert(h[rows], f"{p}mlp.e{e}.", f["expert"]["limit"])
            x = x + _layer_norm(y, w[p + "norm2b"], w[p + "norm2b.b"], eps)
        return _lin(_layer_norm(x[self.want], w["final.norm"], w["final.norm.b"], eps), w["head"])

    # ---- Lodenex
    def lodenex(self):
        w, eps, cap = self.w, self.eps, self.raw["logit_softcap"]
        x = self.embed() * self.raw["embedding"]["scale"]
        for i, L in enumerate(self.raw["layers"]):
            p, m, H = f"l{i}.mix.", L["mixer"], L["mixer"]["heads"]
            if L["type"] == "attention":
                G = m["kv_heads"]
                q = self.heads(_rms(_lin(x, w[p + "q"]), eps, w[p + "q.norm"]), H)
                k = self.heads(_rms(_lin(x, w[p + "k"]), eps, w[p + "k.norm"]), G)
                o = _attend(_rotate(q, self.fposition, m["rot"]),
                            _rotate(k, self.fposition, m["rot"]), self.heads(_lin(x, w[p + "v"]), G),
                            m["scale"], self.bounds, chunk=m["mask"]["size"], cap=m["softcap"],
                            sink=w[p + "sink"])
                gate = torch.sigmoid(_lin(x, w[p + "g"])).repeat_interleave(m["vdim"], dim=1)
            else:
                d, rank = m["dim"], m["kv_rank"]
                q = self.heads(_lin(_rms(_lin(x, w[p + "dq"]), eps, w[p + "dq.norm"]),
                                    w[p + "uq"]), H)
                row = _lin(x, w[p + "dkv"])
                c = _rms(row[:, :rank], eps, w[p + "dkv.norm"])
                turned = _rotate(row[:, None, rank:], self.fposition, m["rot"])
                k = torch.cat([self.heads(_lin(c, w[p + "uk"]), H), turned.expand(-1, H, -1)], dim=-1)
                q = torch.cat([q[..., :d], _rotate(q[..., d:], self.fposition, m["rot"])], dim=-1)
                o = _attend(q, k, self.heads(_lin(c, w[p + "uv"]), H), m["scale"], self.bounds,
                            window=m["mask"]["size"])
                gate = torch.sigmoid(_lin(x, w[p + "g"]))
            x = x + _rms(_lin(o * gate, w[p + "o"]), eps, w[f"l{i}.norm1"])
            z = _lin(x, w[f"l{i}.mlp.up"])
            z = 0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0)))
            x = x + _rms(_lin(z, w[f"l{i}.mlp.down"]), eps, w[f"l{i}.norm2"])
        return cap * torch.tanh(_lin(_rms(x[self.want], eps, w["final.norm"]), w["head"]) / cap)

    # ---- Nupovik
    def nupovik(self):
        w, eps, W = self.w, self.eps, self.raw["width"]
        f = torch.tensor([10000.0 ** (-2.0 * i / W) for i in range(W // 2)], dtype=F64, device=DEVICE)
        a = self.fposition[:, None] * f
        x = self.embed() + torch.stack([torch.sin(a), torch.cos(a)], dim=-1).view(-1, W)
        for i, L in enumerate(self.raw["layers"]):
            p, m, H = f"l{i}.mix.", L["mixer"], L["mixer"]["heads"]
            h = _rms(x, eps, w[f"l{i}.norm1"])
            if L["type"] == "gla":
                z = _lin(_lin(h, w[p + "a1"]), w[p + "a2"], w[p + "a2.b"])
                o = self.rows.recur(self.heads(_lin(h, w[p + "q"]), H) * m["dim"] ** -0.5,
                                    self.heads(_lin(h, w[p + "k"]), H),
                                    self.heads(_lin(h, w[p + "v"]), H),
                                    self.heads(torch.sigmoid(z).pow(1.0 / m["tau"]), H))
                o = _rms(o, eps, w[p + "norm"]).reshape(len(x), -1)
                gate = _silu(_lin(h, w[p + "g"]))
            else:
                before = self.rows.before(h, 1)
                mixed = {n: h + (before - h) * w[p + "mu." + n].to(F64) for n in "rkvgw"}
                z = _lin(torch.tanh(_lin(mixed["w"], w[p + "w1"])), w[p + "w2"], w[p + "w0"])
                r, k, v = (self.heads(_lin(mixed[n], w[p + n]), H) for n in "rkv")
                o = self.rows.recur(r, k, v, self.heads(torch.exp(-torch.exp(z)), H),
                                    bonus=w[p + "u"].to(F64))
                o = _rms(o, eps).reshape(len(x), -1) * w[p + "norm"].to(F64)
                gate = _silu(_lin(mixed["g"], w[p + "g"]))
            y = _lin(o * gate, w[p + "o"])
            h = _rms(x, eps, w[f"l{i}.norm2"])
            x = x + y + _lin(_lin(h, w[f"l{i}.mlp.up"]).clamp(min=0.0) ** 2, w[f"l{i}.mlp.down"])
        return _lin(_rms(x[self.want], eps, w["final.norm"]), w["head"]) * self.raw["logit_scale"]

    # ---- Kugisun
    def kugisun(self):
        w, eps = self.w, self.eps

        def norm(v, name):
            return _rms(v, eps) * (1.0 + w[name].to(F64))

        def gated(h, p):
            return _lin(_silu(_lin(h, w[p + "gate"])) * _lin(h, w[p + "up"]), w[p + "down"])

        def left(h, p, m):
            q, k, v = (self.heads(_lin(h, w[p + n], w[p + n + ".b"]), m[c])
                       for n, c in (("q", "heads"), ("k", "kv_heads"), ("v", "kv_heads")))
            q, k = (_rotate(_rms(z, eps, w[p + n]), self.fposition, m["rot"], neighbours=True)
                    for z, n in ((q, "q.norm"), (k, "k.norm")))
            return _lin(_attend(q, k, v, m["scale"], self.bounds), w[p + "o"])

        def right(h, p, m):
            def unit(v):
                return v / torch.sqrt((v * v).sum(dim=-1, keepdim=True) + 1e-6)
            per = m["heads"] // m["kv_heads"]
            q, k, v = (_silu(self.rows.conv(_lin(h, w[p + n]), w[p + n + ".conv"])) for n in "qkv")
            q = (unit(self.heads(q, m["kv_heads"])) * m["dim"] ** -0.5).repeat_interleave(per, dim=1)
            k = unit(self.heads(k, m["kv_heads"])).repeat_interleave(per, dim=1)
            g = torch.exp(-torch.exp(w[p + "A_log"].to(F64))
                          * _softplus(_lin(h, w[p + "a"], w[p + "dt_bias"])))
            o = self.rows.recur(q, k, self.heads(v, m["heads"]), g,
                                beta=torch.sigmoid(_lin(h, w[p + "b"])))
            o = _rms(o, eps, w[p + "norm"]) * self.heads(_silu(_lin(h, w[p + "g"])), m["heads"])
            return _lin(o.reshape(len(h), -1), w[p + "o"])

        def mixture(h, p, f):
            r = f["router"]
            s = torch.softmax(_lin(h, w[p + "router"]), dim=-1)
            c = s + w[p + "correction"].to(F64)
            size = c.shape[1] // r["groups"]["count"]
            marks = c.view(len(h), -1, size).max(dim=-1).values
            kept = torch.zeros_like(marks, dtype=torch.bool).scatter_(
                1, torch.topk(marks, r["groups"]["keep"], dim=-1).indices, True)
            c = c.masked_fill(~kept.repeat_interleave(size, dim=1), -math.inf)
            ids = torch.topk(c, r["top"], dim=-1).indices
            part = torch.zeros_like(s).scatter_(1, ids, torch.gather(s, 1, ids) * r["scale"])
            y = torch.sigmoid(_lin(h, w[p + "shared.sg"])) * gated(h, p + "shared.")
            y = y + part[:, r["experts"]:].sum(dim=-1, keepdim=True) * h
            for e in range(r["experts"]):
                rows = (ids == e).any(dim=-1).nonzero()[:, 0]
                if len(rows):
                    y[rows] += part[rows, e:e + 1] * gated(h[rows], f"{p}e{e}.")
            return y

        x = self.embed() + w["pos"].to(F64)[self.pos]
        X = torch.stack([x] * self.raw["streams"])
        for i, L in enumerate(self.raw["layers"]):
            p, m, f = f"l{i}.", L["mixer"], L["mlp"]

            def mix(h):
                return m["left_scale"] * left(h, p + "mix.left.", m["left"]) \
                    + m["right_scale"] * right(h, p + "mix.right.", m["right"])

            def feed(h):
                return gated(h, p + "mlp.") if f["kind"] == "dense" else mixture(h, p + "mlp.", f)
            for c, sublayer in ((1, mix), (2, feed)):
                a, M, b = (w[f"{p}hc{c}.{n}"].to(F64) for n in ("in", "mix", "out"))
                y = sublayer(norm(torch.tensordot(a, X, dims=1), f"{p}norm{c}"))
                X = torch.tensordot(M.T, X, dims=1) + b[:, None, None] * y
        return _lin(norm(X.sum(dim=0)[self.want], "final.norm"), w["embed"])

    # ---- Fumanex
    def fumanex(self):
        w, eps = self.w, self.eps
        x, first = self.embed() * self.raw["embedding"]["scale"], None
        for i, L in enumerate(self.raw["layers"]):
            p, m, H = f"l{i}.mix.", L["mixer"], L["mixer"]["heads"]
            h = _rms(x, eps, w[f"l{i}.norm1"])
            if L["type"] == "attention":
                G = m["kv_heads"]
                q = _rms(self.heads(_lin(h, w[p + "q"], w[p + "q.b"]), H), eps)
                k = _rms(self.heads(_lin(h, w[p + "k"], w[p + "k.b"]), G), eps)
                v = self.heads(_lin(h, w[p + "v"], w[p + "v.b"]), G)
                if first is None:
                    first = v
                else:
                    lam = w[p + "vmix"].to(F64)
                    v = (1.0 - lam) * v + lam * first
                table = w[p + "rel"].to(F64)

                def bias(T):
                    B, near = table.shape[0], table.shape[0] // 2
                    far = [min(B - 1, near + math.floor(math.log(n / near) / math.log(
                        m["bias_max"] / near) * (B - near) + 1e-9)) for n in range(near, T)]
                    rows = torch.tensor((list(range(near)) + far)[:T], device=DEVICE)
                    at = torch.arange(T, device=DEVICE)
                    return table[rows][(at[:, None] - at).clamp(min=0)].permute(2, 0, 1)
                o = _attend(q, k, v, m["scale"], self.bounds, window=m["mask"]["size"],
                            keep=m["mask"]["keep_first"], cap=m["softcap"], sink=w[p + "sink"],
                            bias=bias)
                y = _lin(o, w[p + "o"], w[p + "o.b"])
            else:
                q, k, v = (self.heads(_lin(h, w[p + n]), H) for n in "qkv")
                if L["type"] == "retention":
                    q = _rotate(q, self.fposition, m["rot"])
                    k = _rotate(k, self.fposition, m["rot"]) * m["dim"] ** -0.5
                else:
                    q, k, v = _silu(q), _silu(k), _silu(v)
                o = self.rows.recur(q, k, v, torch.tensor(m["decay"], dtype=F64, device=DEVICE))
                z = _lin(h, w[p + "g"])
                if L["type"] == "retention":
                    o = _rms(o, eps).reshape(len(x), -1) * _silu(z)
                else:
                    o = _rms(o.reshape(len(x), -1), eps, w[p + "norm"]) * torch.sigmoid(z)
                y = _lin(o, w[p + "o"])
            f = f"l{i}.mlp."
            x = x + y + _lin(_gelu_tanh(_lin(h, w[f + "up"], w[f + "up.b"])), w[f + "down"],
                             w[f + "down.b"])
        return _lin(_rms(x[self.want], eps, w["final.norm"]), w["head"]) * self.raw["logit_scale"]

    # ---- Tigesun
    def tigesun(self):
        w, eps, cap = self.w, self.eps, self.raw["logit_softcap"]
        x = _rms(self.embed(), eps, w["embed.norm"])
        for i, L in enumerate(self.raw["layers"]):
            p, m, H = f"l{i}.mix.", L["mixer"], L["mixer"]["heads"]
            h = _rms(x, eps, w[f"l{i}.norm1"])
            if L["type"] == "attention":
                G = m["kv_heads"]
                q = _rms(self.heads(_lin(h, w[p + "q"]), H), eps, w[p + "q.norm"])
                k = _rms(self.heads(_lin(h, w[p + "k"]), G), eps, w[p + "k.norm"])
                y = _attend(_rotate(q, self.fposition, m["rot"]),
                            _rotate(k, self.fposition, m["rot"]), self.heads(_lin(h, w[p + "v"]), G),
                            m["scale"], self.bounds)
            elif L["type"] == "latent_attention":
                c = _rms(_lin(h, w[p + "dkv"]), eps, w[p + "dkv.norm"])
                y = _attend(self.heads(_lin(h, w[p + "q"]), H), self.heads(_lin(c, w[p + "uk"]), H),
                            self.heads(_lin(c, w[p + "uv"]), H), m["scale"], self.bounds,
                            window=m["mask"]["size"])
            else:
                inner, N, G = H * m["vdim"], m["state"], m["groups"]
                z, u, s = torch.split(_lin(h, w[p + "in"]), [inner, inner + 2 * G * N, H], dim=1)
                u = _silu(self.rows.conv(u, w[p + "conv"]) + w[p + "conv.b"].to(F64))
                u, B, C = torch.split(u, [inner, G * N, G * N], dim=1)
                u = self.heads(u, H)
                dt = _softplus(s + w[p + "dt_bias"].to(F64))
                B, C = (self.heads(t, G).repeat_interleave(H // G, dim=1) for t in (B, C))
                y = self.rows.recur(C, B, u * dt[:, :, None],
                                    torch.exp(-torch.exp(w[p + "A_log"].to(F64)) * dt))
                y = (y + w[p + "D"].to(F64)[:, None] * u).reshape(len(x), inner) * _silu(z)
                y = _rms(self.heads(y, m["norm_groups"]), eps).reshape(len(x), inner) \
                    * w[p + "norm"].to(F64)
            x = x + _rms(_lin(y, w[p + "o"]), eps, w[f"l{i}.norm1b"])
            if L["mlp"] is not None:
                f = f"l{i}.mlp."
                h = _rms(x, eps, w[f"l{i}.norm2"])
                y = _lin(_gelu_tanh(_lin(h, w[f + "gate"], w[f + "gate.b"]))
                         * _lin(h, w[f + "up"], w[f + "up.b"]), w[f + "down"], w[f + "down.b"])
                x = x + _rms(y, eps, w[f"l{i}.norm2b"])
        x = _rms(x[self.want], eps, w["final.norm"])
        return cap * torch.tanh(_lin(x, w["embed"]) / cap)


def exact(case, seed) -> Optional[dict]:
    """The logits in 64 bits; tokens drawn have no such value.  Cases whose products would take
    too long in 64 bits have none."""
    if work(case)["flops"] > 4e14:
        return None
    with torch.no_grad():
        logits = _Exact(case, seed).logits()
    return {"logits": logits, "tokens": None} if case["draw"] else {"logits": logits}
