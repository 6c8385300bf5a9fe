"""The work this engine is timed on: steps of whole models through the cache manager and the step function.

One pass serves some requests as a program does that drives the engine itself (like the trace replay): contexts that are
already held get given next tokens, new prompts are opened, go through in portions beside them, decode a few tokens and are
closed. Every pass returns the logits of every token that a program would sample from. Tokens are given, not sampled: the
weights are random, and a sampled token would turn on the last bit of a logit.

Models have the widths, heads and vocabularies of the benchmark's sizes and few layers, so that a pass is short and
bfloat16's rounding, which grows with the depth, stays below what is compared; every layer kind of a design is there. Routed
experts run in float32 only: in bfloat16 one token in a hundred stands so near the edge between two experts that another
order of summation sends it to the other one, and its logits say nothing about either kernel then.
"""
from __future__ import annotations

import hashlib
import math

import numpy as np
import torch

DTYPES = {"bfloat16": torch.bfloat16, "float32": torch.float32}
VOCAB = 32000                     # of every design but Qwen2
PAGE = 16

# Qwen2.5 layer sizes: (hidden, heads, kv_heads, head_dim, intermediate, vocab, tied, eps)
QWEN = {"0.5b": (896, 14, 2, 64, 4864, 151936, True, 1e-6), "3b": (2048, 16, 2, 128, 11008, 151936, True, 1e-6),
        "7b": (3584, 28, 4, 128, 18944, 152064, False, 1e-6), "14b": (5120, 40, 8, 128, 13824, 152064, False, 1e-5)}
# The other designs' sizes: (width, heads, kv_heads, head_dim, feed-forward, window)
SIZES = {"1b": (2048, 16, 4, 128, 5632, 1024), "3b": (3072, 24, 4, 128, 8192, 2048)}
DESIGNS = ("kanavik", "dinutar", "rufusun", "tadalorn", "darolix", "vulosun")


def listed():
    """`held` contexts of about `context` tokens decode `steps` tokens; `prompts` new ones of about `prompt` tokens go through in
    portions of `chunk` beside them and then decode `steps` tokens too. (About: lengths are spread by `spread` percent.)"""
    def case(name, design, size, layers, held, context, prompts, prompt, steps, spread=0, chunk=2048, dtype="bfloat16"):
        return dict(name=name, design=design, size=size, layers=layers, dtype=dtype, held=held, context=context, prompts=prompts,
                    prompt=prompt, steps=steps, spread=spread, chunk=chunk)
    return [
        # one chat user on a small model: nothing but the latency of one step after another
        case("qwen2 0.5b decode 1", "qwen2", "0.5b", 4, 1, 200, 0, 0, 4),
        # the headline: a small batch at a context of 4,096
        case("qwen2 7b decode 8", "qwen2", "7b", 4, 8, 4088, 0, 0, 4),
        # a full server in steady state: 64 requests of unequal lengths
        case("qwen2 7b decode 64", "qwen2", "7b", 4, 64, 1200, 0, 0, 4, spread=40),
        # a prompt of 2,048 tokens up to its first tokens
        case("qwen2 7b prompt 2048", "qwen2", "7b", 4, 0, 0, 1, 2048, 1),
        # continuous batching: prompt portions of 512 beside decoding requests
        case("qwen2 14b mixed", "qwen2", "14b", 4, 24, 1500, 3, 700, 4, spread=30, chunk=512),
        # a long document in portions
        case("qwen2 7b prompt 8192", "qwen2", "7b", 4, 0, 0, 1, 8192, 1),
        # the other designs: a prompt and the begin of its answer, or some short dialogues
        case("kanavik prompt", "kanavik", "1b", 4, 0, 0, 1, 2047, 4),
        case("dinutar dialogues", "dinutar", "1b", 4, 0, 0, 8, 150, 24, spread=30),
        case("rufusun prompts", "rufusun", "1b", 4, 0, 0, 2, 1000, 8, spread=20),
        case("tadalorn prompt", "tadalorn", "1b", 4, 0, 0, 1, 2048, 8),
        # the true 32-bit path, with routed experts
        case("darolix float32 dialogues", "darolix", "1b", 4, 0, 0, 4, 120, 16, spread=50, dtype="float32"),
        case("vulosun dialogues", "vulosun", "1b", 4, 0, 0, 8, 400, 16, spread=30),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """A case of the same ranges: half of them Qwen2 (decoding, prompts, both), half of the other designs."""
    c = dict(layers=4, dtype="bfloat16", held=0, context=0, prompts=0, prompt=0, steps=rng.randint(1, 6), spread=rng.randint(0, 45),
             chunk=rng.choice((512, 1024, 2048)))
    if rng.random() < 0.5:
        c.update(design="qwen2", size=rng.choice(sorted(QWEN)))
        kind = rng.choice(("decode", "prompt", "mixed"))
        if kind != "prompt":
            c.update(held=_log(rng, 1, 64), context=_log(rng, 100, 4000))
            c["context"] = min(c["context"], 90000 // c["held"])
        if kind != "decode":
            c.update(prompts=_log(rng, 1, 4), prompt=_log(rng, 65, 2000))
        if kind == "prompt" and rng.random() < 0.5:
            c.update(prompts=1, prompt=_log(rng, 65, 6000))
        if c["size"] == "0.5b" and rng.random() < 0.5:
            c["dtype"] = "float32"
        c["prompt"] = min(c["prompt"], {"7b": 6000, "14b": 3500}.get(c["size"], 8000) // max(1, c["prompts"]))
    else:
        c.update(design=rng.choice(DESIGNS), size=rng.choice(sorted(SIZES)), prompts=_log(rng, 1, 8), steps=_log(rng, 4, 24))
        c["prompt"] = min(_log(rng, 40, 2200), 3500 // c["prompts"])
        if c["design"] in ("rufusun", "darolix", "vulosun", "tadalorn") and rng.random() < 0.3:
            c.update(dtype="float32", size="1b", prompt=min(c["prompt"], 800 // c["prompts"]))
    return c


# ---- what a case's requests do ---------------------------------------------------------------------------------------
def _requests(case):
    """[(tokens held at the start, tokens of the prompt behind them)]: lengths spread evenly over +- spread percent."""
    def spread(count, middle):
        s = case["spread"] / 100.0
        return [max(2, int(middle * (1 + s * (2 * (i * 7 % count) / max(1, count - 1) - 1 if count > 1 else 0)))) for i in range(count)]
    return [(n, 0) for n in spread(case["held"], case["context"])] + [(0, n) for n in spread(case["prompts"], case["prompt"])]


def _plan(case):
    """The steps of a pass: lists of (request, first token, one behind the last, are the last token's logits wanted).
    Requests that are past their prompt decode one token a step; prompts share the step's portion in order."""
    at = [held for held, _ in _requests(case)]
    until = [held + prompt for held, prompt in _requests(case)]
    end = [u + case["steps"] for u in until]
    steps = []
    while any(a < e for a, e in zip(at, end)):
        entries, room = [], case["chunk"]
        for r in range(len(at)):
            if at[r] < until[r]:
                n = min(room, until[r] - at[r])
                room -= n
                if n:
                    entries.append((r, at[r], at[r] + n, at[r] + n == until[r]))
            elif at[r] < end[r]:
                entries.append((r, at[r], at[r] + 1, True))
        for r, _, stop, _ in entries:
            at[r] = stop
        steps.append(entries)
    return steps


def _vocab(case):
    return QWEN[case["size"]][5] if case["design"] == "qwen2" else VOCAB


def _tokens(case, seed):
    rng = np.random.RandomState(seed % (1 << 31))
    return [rng.randint(0, _vocab(case), h + p + case["steps"]).tolist() for h, p in _requests(case)]


# ---- the models -------------------------------------------------------------------------------------------------------
def _config(case):
    if case["design"] == "qwen2":
        hidden, heads, kv, dim, ff, vocab, tied, eps = QWEN[case["size"]]
        return dict(architectures=["Qwen2ForCausalLM"], model_type="qwen2", num_hidden_layers=case["layers"], hidden_size=hidden,
                    num_attention_heads=heads, num_key_value_heads=kv, head_dim=dim, intermediate_size=ff, vocab_size=vocab,
                    rope_theta=1e6, rms_norm_eps=eps, tie_word_embeddings=tied, use_sliding_window=False,
                    max_position_embeddings=32768, hidden_act="silu")
    layers = _LAYERS[case["design"]](*SIZES[case["size"]], case["dtype"] == "float32")
    top = {"vocab": VOCAB, "width": SIZES[case["size"]][0], "norm": {"eps": 1e-6},
           "layers": [layers[i % len(layers)] for i in range(case["layers"])]}
    return {"architecture": case["design"].capitalize(), **top, **_TOP[case["design"]](SIZES[case["size"]][0])}


def _kanavik_layers(width, heads, kv, dim, ff, window, experts):
    return [{"type": "parallel", "mlp": {"kind": "dense", "ff": ff},
             "mixer": {"left": {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "mask": {"size": window}},
                       "right": {"width": width, "blocks": 16, "conv": 4}, "left_scale": 1.0, "right_scale": 1.0}}]


def _dinutar_layers(width, heads, kv, dim, ff, window, experts):
    rot = {"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}
    half = heads // 2
    latent = {"heads": heads, "dim": dim - 64, "rot_dim": 64, "vdim": dim, "kv_rank": 192, "scale": dim ** -0.5, "rot": rot}
    keep = {"heads": half, "dim": dim, "vdim": width // half, "decay": [1.0 - 2.0 ** (-5 - 3 * h / (half - 1)) for h in range(half)],
            "rot": {"base": 10000.0, "dims": dim}}
    mlp = {"kind": "dense", "ff": ff}
    return [{"type": "retention", "mixer": keep, "mlp": mlp}, {"type": "latent_attention", "mixer": latent, "mlp": mlp},
            {"type": "retention", "mixer": keep, "mlp": mlp}, {"type": "latent_attention", "mixer": dict(latent, kv_from=1), "mlp": mlp}]


def _rufusun_layers(width, heads, kv, dim, ff, window, experts):
    dense = {"kind": "dense", "ff": ff}
    routed = {"kind": "moe", "router": {"experts": 16, "top": 2}, "expert": {"ff": ff // 4, "limit": 7.0},
              "shared": {"ff": ff // 4, "limit": 7.0}}
    delta = {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "conv": 4}
    soft = {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "softcap": 30.0,
            "rot": {"base": 1e6, "dims": dim // 2}}
    return [{"type": "delta" if i < 2 else "attention", "mixer": delta if i < 2 else soft, "mlp": routed if experts and i % 2 else dense}
            for i in range(4)]


def _tadalorn_layers(width, heads, kv, dim, ff, window, experts):
    dense = {"kind": "dense", "ff": ff}
    routed = {"kind": "moe", "router": {"experts": 16, "top": 2}, "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}}
    latent = {"heads": heads, "dim": dim - 64, "rot_dim": 64, "vdim": dim, "kv_rank": 192, "scale": dim ** -0.5,
              "rot": {"base": 10000.0, "dims": 64}}
    memory = {"heads": heads, "dim": dim, "vdim": dim, "gate_cap": 15.0}
    near = {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "conv": 4,
            "mask": {"size": window, "keep_first": 8}, "rot": {"base": 1e6, "dims": dim // 2}}
    # the memory first: behind full attention, which random weights leave an average over all tokens, its values are all but
    # equal and a head's normed result turns its sign where its query happens to be orthogonal to the summed keys
    kinds = [("mlstm", memory), ("latent_attention", latent), ("attention", near), ("latent_attention", latent)]
    return [{"type": kind, "mixer": mixer, "mlp": routed if experts and i else dense} for i, (kind, mixer) in enumerate(kinds)]


def _darolix_layers(width, heads, kv, dim, ff, window, experts):
    mlp = {"kind": "moe", "router": {"experts": 16, "identity": 4, "top": 2}, "expert": {"ff": ff // 4}} if experts else None
    space = {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 8, "conv": 4, "norm_groups": 8}
    beside = {"left": {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5, "softcap": 30.0,
                       "q_temp": {"coef": 0.1, "every": 1024}},
              "right": {"heads": heads, "dim": dim // 2, "vdim": dim, "tau": 16.0}}
    return [{"type": "mamba2", "mixer": space, "mlp": mlp}, {"type": "parallel", "mixer": beside, "mlp": mlp}]


def _vulosun_layers(width, heads, kv, dim, ff, window, experts):
    dense = {"kind": "dense", "ff": ff}
    routed = {"kind": "moe", "router": {"experts": 16, "top": 2, "scale": 1.5, "groups": {"count": 4, "keep": 2}},
              "expert": {"ff": ff // 4}, "shared": {"ff": ff // 4}}
    plain = {"heads": heads, "kv_heads": kv, "dim": dim, "vdim": dim, "scale": dim ** -0.5}
    beside = {"left": dict(plain, rot={"base": 1e6, "dims": dim // 2}), "left_scale": 0.8, "right_scale": 0.5,
              "right": {"heads": heads, "dim": dim // 2, "vdim": dim, "decay": [1.0 - 2.0 ** (-3 - 6 * h / (heads - 1)) for h in range(heads)]}}
    maps = {"heads": heads // 2, "kv_heads": kv // 2, "dim": dim // 2, "vdim": dim, "scale": (dim // 2) ** -0.5, "diff": 0.3,
            "mask": {"size": window}, "rot": {"base": 50000.0, "dims": dim // 2, "scaling": {"factor": 4.0}}}
    kinds = [("attention_2", maps), ("parallel", beside), ("attention", dict(plain, rot={"base": 1e6, "dims": dim})),
             ("attention_2", dict(maps, kv_from=0))]
    return [{"type": kind, "mixer": mixer, "mlp": routed if experts and i else dense} for i, (kind, mixer) in enumerate(kinds)]


_LAYERS = {"kanavik": _kanavik_layers, "dinutar": _dinutar_layers, "rufusun": _rufusun_layers, "tadalorn": _tadalorn_layers,
           "darolix": _darolix_layers, "vulosun": _vulosun_layers}
_TOP = {"kanavik": lambda width: {"max_positions": 8192, "residual_mult": 1.0, "canon": {"taps": 4}, "token_side": {"dim": 128}},
        "dinutar": lambda width: {"postln_alpha": 1.0, "embedding": {"scale": 1.0, "bigram": {"buckets": 65521, "mul_prev": 31, "mul_cur": 7}}},
        "rufusun": lambda width: {"logit_scale": 1.0},
        "tadalorn": lambda width: {"residual_mult": 0.7, "logit_softcap": 30.0},
        "darolix": lambda width: {"embedding": {"scale": width ** 0.5}},
        "vulosun": lambda width: {}}


def _weight(seed, name, shape, kind="normal"):
    """One tensor of a model: N(0, 0.02), less for wide rows, so that a product keeps its input's size (norm weights around one,
    the depth average around 1 / entries, head mixing around the identity, forget gates around open, as they are trained to be:
    a memory of two tokens is often orthogonal to the query, and its norm then shows nothing but rounding), rounded to bfloat16:
    both precisions run the same values."""
    digest = hashlib.sha256(f"{seed}:{name}".encode()).digest()
    g = torch.Generator(device="cuda").manual_seed(int.from_bytes(digest[:7], "little"))
    std = min(0.02, 0.9 * shape[-1] ** -0.5) if len(shape) > 1 else 0.02
    t = torch.empty(shape, dtype=torch.float32, device="cuda").normal_(0.0, std, generator=g)
    if name.endswith(".mix.f.b"):
        t += 4.0
    elif kind == "one_plus_normal":
        t += 1.0
    elif kind == "average":
        t = (t + 1.0) / t.numel()
    elif kind == "identity_plus_normal":
        t += torch.eye(*shape, device="cuda")
    return t.to(torch.bfloat16)


# ---- one pass ---------------------------------------------------------------------------------------------------------
class State:
    """What a serving program has in hand: the model, the cache, the step function, and the contexts that are held."""

    def __init__(self, case, seed):
        from tessweave_engine_amd.cache import CacheManager
        from tessweave_engine_amd.config import build_model, config_from_dict
        from tessweave_engine_amd.engine.step import StepEntry, Stepper
        self.entry = StepEntry
        dtype = DTYPES[case["dtype"]]
        model = build_model(config_from_dict(_config(case)))
        tensors = {s.name: _weight(seed, s.name, s.shape, s.init).to(dtype if s.role == "matrix" else torch.float32)
                   for s in model.tensor_specs() if s.optional_alias_of is None}
        model.bind(tensors, dtype, torch.device("cuda:0"))
        self.requests, self.plan, self.tokens = _requests(case), _plan(case), _tokens(case, seed)
        lengths = [len(t) for t in self.tokens]
        pages = sum(-(-n // PAGE) for n in lengths) + 4 * len(lengths)
        self.cache = CacheManager(model.cache_layout(), PAGE, pages, len(lengths), dtype=case["dtype"], device=model.device,
                                  prefix_cache=False, max_request_tokens=-(-max(lengths) // 64) * 64)
        self.stepper = Stepper(model, self.cache, max_step_tokens=case["chunk"] + len(lengths))
        self.held = {}
        for r, (held, _) in enumerate(self.requests):
            if held:
                seq = self.held[r] = self.cache.open(r)
                for a in range(0, held, 2048):
                    self.stepper.step([StepEntry(seq, self.tokens[r][a:min(held, a + 2048)])])


def prepare(case, seed):
    return State(case, seed)


def run(state):
    seqs = dict(state.held)
    for r, seq in seqs.items():
        seq.computed = state.requests[r][0]       # other continuations of the same context: back to its end
    logits = []
    for step in state.plan:
        entries = []
        for r, start, stop, want in step:
            if r not in seqs:
                seqs[r] = state.cache.open(r)
            entries.append(state.entry(seqs[r], state.tokens[r][start:stop], [stop - start - 1] if want else []))
        out = state.stepper.step(entries)
        if out.shape[0]:
            logits.append(out.clone())            # the step's logits are scratch memory until the next step
    for r, seq in seqs.items():
        if r not in state.held:
            state.cache.close(seq)
    return logits


# ---- what a pass cannot do without ------------------------------------------------------------------------------------
def _attention_flops_bytes(case, config, layer, at, new, size):
    """Operations and cache bytes of NEW tokens behind AT others in one layer."""
    def pairs(window=None, chunk=None):
        """(query, key) pairs, keys read"""
        total, first = 0, at
        for p in (range(at, at + new) if window or chunk else ()):
            low = max(0, p + 1 - window) if window else p // chunk * chunk
            first = min(first, low)
            total += p + 1 - low
        return (total, at - first) if window or chunk else (new * at + new * (new + 1) // 2, at)
    if case["design"] == "qwen2":
        heads, kv, dim = QWEN[case["size"]][1:4]
        n, keys = pairs()
        return 4 * n * heads * dim, 2 * (keys + new) * kv * dim * size
    m, flops, moved = layer["mixer"], 0, 0
    for part in [m] if "left" not in m else [m["left"], m["right"]]:
        if "kv_rank" in part:
            n, keys = pairs()
            flops += 2 * n * part["heads"] * (part["dim"] + part["rot_dim"] + part["vdim"])
            moved += (keys + new) * (part["kv_rank"] + part["rot_dim"]) * size
        elif "state" in part or "blocks" in part or layer["type"] in ("retention", "delta", "mlstm") or (part is m.get("right")):
            cells = part["width"] if "blocks" in part else part["heads"] * part.get("state", part.get("dim")) * part["vdim"]
            flops += 4 * new * cells
            moved += 2 * cells * 4
        else:
            mask = part.get("mask") or {}
            n, keys = pairs(chunk=mask["size"]) if layer["type"] == "attention_2" else pairs(window=mask.get("size"))
            maps = 2 if layer["type"] == "attention_2" else 1
            flops += 2 * n * part["heads"] * (maps * part["dim"] + maps * part["vdim"])
            moved += (keys + new) * part["kv_heads"] * (maps * part["dim"] + part["vdim"]) * size
    return flops, moved


def work(case):
    """Weights once a step (experts: those that the step's tokens can choose), the cache's keys and states of the requests,
    the logits; two operations a weight and token, and the attention."""
    from tessweave_engine_amd.config import build_model, config_from_dict
    config = _config(case)
    size = 2 if case["dtype"] == "bfloat16" else 4
    model = build_model(config_from_dict(config))
    tables = {"model.embed_tokens.weight", "embed", "bigram", "pos", "side.embed"}
    shapes = [s for s in model.tensor_specs() if s.optional_alias_of is None and len(s.shape) >= 2 and s.name not in tables]
    head = _vocab(case) * (QWEN[case["size"]][0] if case["design"] == "qwen2" else SIZES[case["size"]][0])
    dense = sum(math.prod(s.shape) for s in shapes if ".mlp.e" not in s.name and s.name not in ("head", "lm_head.weight"))
    experts = sum(math.prod(s.shape) for s in shapes if ".mlp.e" in s.name)
    layers = config.get("layers") or [None] * case["layers"]
    total_bytes = total_flops = 0.0
    for step in _plan(case):
        n, wanted = sum(stop - start for _, start, stop, _ in step), sum(want for *_, want in step)
        total_bytes += (dense + experts * min(1.0, 2 * n / 16) + (head if wanted else 0)) * size + wanted * _vocab(case) * 4
        total_flops += 2.0 * (dense + experts * 2 / 16) * n + 2.0 * head * wanted
        for layer in layers:
            for _, start, stop, _ in step:
                f, b = _attention_flops_bytes(case, config, layer, start, stop - start, size)
                total_flops += f
                total_bytes += b
    return {"bytes": total_bytes, "flops": total_flops}


def tolerance(case):
    """Two to four times what the engine is off from `exact` over these ranges: in bfloat16, which rounds every activation to 8
    bits, 0.4 to 1.1 % (one logit by up to 5 % of their root mean square), in float32 1e-6 to 2.6e-6 (2e-5)."""
    return {"rel": 2.5e-2, "max": 0.2} if case["dtype"] == "bfloat16" else {"rel": 1.2e-5, "max": 8e-5}


# ---- the same in 64 bits, with plain torch: whole sequences, no cache -------------------------------------------------
def exact(case, seed):
    config, tokens = _config(case), _tokens(case, seed)
    wanted = {}
    for step in _plan(case):
        for r, _, stop, want in step:
            if want:
                wanted.setdefault(r, []).append(stop - 1)
    with torch.no_grad():
        rows = _Plain(config, seed).logits([tokens[r] for r in wanted], list(wanted.values()))
    found = {(r, p): row for r, out in zip(wanted, rows) for p, row in zip(wanted[r], out)}
    return [torch.stack([found[r, stop - 1] for r, _, stop, want in step if want]) for step in _plan(case) if any(e[3] for e in step)]


def _rms(x, eps, weight=1.0):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * weight


def _gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _silu(z):
    return z * torch.sigmoid(z)


def _softplus(z):
    return torch.clamp(z, min=0) + torch.log1p(torch.exp(-z.abs()))


def _conv(x, taps):
    """Causal convolution per channel; the last column of TAPS meets the current token."""
    k = taps.shape[1]
    padded = torch.cat([x.new_zeros(k - 1, x.shape[1]), x])
    return sum(padded[j:j + x.shape[0]] * taps[:, j] for j in range(k))


def _turn(x, rot, neighbours=False):
    """x [T, heads, D]: the first rot["dims"] elements of a head turn with the position, halves or neighbours together."""
    dims = rot["dims"]
    i = torch.arange(dims // 2, dtype=torch.float64, device=x.device)
    f, size, s = rot["base"] ** (-2.0 * i / dims), 1.0, rot.get("scaling")
    if s and "original" in s:
        def pair_of(turns):
            return dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(rot["base"]))
        lo, hi = max(math.floor(pair_of(s["fast"])), 0), min(math.ceil(pair_of(s["slow"])), dims - 1)
        ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, size = f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0
    elif s:
        f = f / s["factor"]
    angle = torch.arange(x.shape[0], dtype=torch.float64, device=x.device).view(-1, 1, 1) * f
    cos, sin = torch.cos(angle) * size, torch.sin(angle) * size
    u, v = (x[..., 0:dims:2], x[..., 1:dims:2]) if neighbours else (x[..., :dims // 2], x[..., dims // 2:dims])
    u, v = u * cos - v * sin, v * cos + u * sin
    return torch.cat([torch.stack([u, v], -1).flatten(-2) if neighbours else torch.cat([u, v], -1), x[..., dims:]], -1)


def _attend(q, k, v, scale, seen=None, sink=None, cap=None):
    """q [T, H, D], k [T, G, D], v [T, G, E]; SEEN [T, T] (default: causal); SINK [H]: more terms exp(sink) in the denominator."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    if seen is None:
        seen = torch.ones(T, T, dtype=torch.bool, device=q.device).tril()
    out = []
    for a in range(H):
        s = (q[:, a] @ k[:, a // (H // G)].T) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        s = s.masked_fill(~seen, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink[a].expand(T, 1)], 1)
        out.append(torch.softmax(s, -1)[:, :T] @ v[:, a // (H // G)])
    return torch.stack(out, 1)


def _linear_state(q, k, v, keep):
    """S <- keep S + k v^T, o = S^T q, token by token and for all heads: q, k [T, H, D], v [T, H, E], keep [T, H, D or 1]."""
    S, out = q.new_zeros(q.shape[1], q.shape[2], v.shape[2]), []
    for t in range(q.shape[0]):
        S = keep[t].unsqueeze(-1) * S + k[t].unsqueeze(-1) * v[t].unsqueeze(-2)
        out.append((q[t].unsqueeze(-2) @ S).squeeze(-2))
    return torch.stack(out)


class _Plain:
    def __init__(self, config, seed):
        self.c, self.seed = config, seed
        self.design = config["architecture"].lower() if "architecture" in config else "qwen2"
        self.eps = config["norm"]["eps"] if "norm" in config else config["rms_norm_eps"]

    def w(self, name, *shape, kind="normal"):
        return _weight(self.seed, name, shape, kind).double()

    def ones(self, name, *shape):
        return self.w(name, *shape, kind="one_plus_normal")

    def times(self, x, name, rows, bias=None):
        y = x @ self.w(name, rows, x.shape[-1]).T
        return y if bias is None else y + self.w(bias, rows)

    def logits(self, sequences, wanted):
        """One list of rows a sequence: the logits at its wanted positions."""
        ids = [torch.tensor(t, device="cuda") for t in sequences]
        streams = getattr(self, "run_" + self.design)(ids)
        at = torch.cat([x[torch.tensor(p, device="cuda")] for x, p in zip(streams, wanted)])
        c = self.c
        if self.design == "qwen2":
            name = "model.embed_tokens.weight" if c["tie_word_embeddings"] else "lm_head.weight"
            out = self.times(_rms(at, self.eps, self.ones("model.norm.weight", at.shape[1])), name, c["vocab_size"])
        else:
            width, vocab = c["width"], c["vocab"]
            if self.design == "vulosun":
                h = self.layer_norm(at, "final.norm")
            elif self.design == "rufusun":
                h = _rms(at, self.eps, 1.0 + self.w("final.norm", width))
            else:
                h = _rms(at, self.eps, self.ones("final.norm", width))
            out = self.times(h, "embed" if self.design == "dinutar" else "head", vocab)
        if self.design == "tadalorn":
            out = c["logit_softcap"] * torch.tanh(out / c["logit_softcap"])
        return out.split([len(p) for p in wanted])

    def embedded(self, ids):
        table = self.w("embed", self.c["vocab"], self.c["width"])
        return [table[t] for t in ids]

    # -- Qwen2
    def run_qwen2(self, ids):
        c = self.c
        hidden, H, G, D = c["hidden_size"], c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
        table = self.w("model.embed_tokens.weight", c["vocab_size"], hidden)
        xs = [table[t] for t in ids]
        del table
        rot = {"base": c["rope_theta"], "dims": D}
        for i in range(c["num_hidden_layers"]):
            p = f"model.layers.{i}."
            a = p + "self_attn."
            w = {n: (self.w(f"{a}{n}_proj.weight", r, hidden), self.w(f"{a}{n}_proj.bias", r)) for n, r in (("q", H * D), ("k", G * D), ("v", G * D))}
            o, n1, n2 = self.w(a + "o_proj.weight", hidden, H * D), self.ones(p + "input_layernorm.weight", hidden), self.ones(p + "post_attention_layernorm.weight", hidden)
            gate, up = (self.w(f"{p}mlp.{n}_proj.weight", c["intermediate_size"], hidden) for n in ("gate", "up"))
            down = self.w(p + "mlp.down_proj.weight", hidden, c["intermediate_size"])
            for s, x in enumerate(xs):
                h = _rms(x, self.eps, n1)
                q, k, v = ((h @ w[n][0].T + w[n][1]).view(len(x), -1, D) for n in ("q", "k", "v"))
                x = x + _attend(_turn(q, rot), _turn(k, rot), v, D ** -0.5).flatten(1) @ o.T
                h = _rms(x, self.eps, n2)
                xs[s] = x + (_silu(h @ gate.T) * (h @ up.T)) @ down.T
        return xs

    # -- shared by the other designs
    def layer_norm(self, x, name):
        x = x - x.mean(-1, keepdim=True)
        return _rms(x, self.eps, self.ones(name, x.shape[-1])) + self.w(name + ".b", x.shape[-1])

    def gated_ff(self, h, p, ff, act=_silu):
        return self.times(act(self.times(h, p + "gate", ff)) * self.times(h, p + "up", ff), p + "down", h.shape[1])

    def experts(self, h, p, n, ids, weights, expert):
        """Sum over the chosen experts: EXPERT(e, rows, their weights)."""
        out = torch.zeros_like(h)
        for e in range(n):
            rows, place = torch.nonzero(ids == e, as_tuple=True)
            if len(rows):
                out[rows] += expert(p + f"e{e}.", h[rows], weights[rows, place].unsqueeze(1))
        return out

    def shared_names(self, h, m, *names):
        return [self.times(h, n, r).view(len(h), k, -1) for n, r, k in names]

    # -- Kanavik
    def run_kanavik(self, ids):
        c, eps = self.c, self.eps
        width, taps, side = c["width"], c["canon"]["taps"], c["token_side"]["dim"]
        pos, table = self.w("pos", c["max_positions"], width), self.w("side.embed", c["vocab"], side * len(c["layers"]))
        out = []
        for t, x in zip(ids, self.embedded(ids)):
            x = x + pos[:len(x)]
            results = [x]
            for i, layer in enumerate(c["layers"]):
                p, m = f"l{i}.", layer["mixer"]
                h = _rms(x, eps, self.ones(p + "norm1", width))
                h = h + _conv(h, self.w(p + "canon1", width, taps))
                x = x + m["left_scale"] * self.mixed_attention(h, p + "mix.left.", m["left"]) + m["right_scale"] * self.recurrence(h, p + "mix.right.", m["right"])
                h = _rms(x, eps, self.ones(p + "norm2", width))
                x = x + self.gated_ff(h + _conv(h, self.w(p + "canon2", width, taps)), p + "mlp.", layer["mlp"]["ff"], _gelu_tanh)
                g = _gelu_tanh(self.times(x, p + "side.gate", side)) * table[t, i * side:(i + 1) * side]
                x = x + _rms(self.times(g, p + "side.proj", width), eps, self.ones(p + "side.norm", width))
                results.append(x)
                x = sum(a * r for a, r in zip(self.w(p + "dwa", i + 2, kind="average"), results))
            out.append(x)
        return out

    def mixed_attention(self, h, p, m):
        T, H, G = len(h), m["heads"], m["kv_heads"]
        q, k, v = (self.times(h, p + n, a * m["dim"]).view(T, a, -1) for n, a in (("q", H), ("k", G), ("v", G)))
        talk, sink = self.w(p + "talk", H, H, kind="identity_plus_normal"), self.w(p + "sink", H).view(H, 1, 1)
        i, out = torch.arange(T, device=h.device), []
        for a in range(0, T, 512):                                       # some rows at a time: all heads' scores meet
            rows = slice(a, min(T, a + 512))
            dist = i[rows].view(-1, 1) - i.view(1, -1)
            s = torch.stack([q[rows, b] @ k[:, b // (H // G)].T * m["scale"] - 2.0 ** (-8.0 * (b + 1) / H) * dist for b in range(H)])
            s = (talk @ s.flatten(1)).view_as(s).masked_fill((dist < 0) | (dist >= m["mask"]["size"]), -math.inf)
            pr = torch.softmax(torch.cat([s, sink.expand(H, s.shape[1], 1)], -1), -1)[..., :T]
            out.append(torch.stack([pr[b] @ v[:, b // (H // G)] for b in range(H)], 1))
        return self.times(torch.cat(out).flatten(1), p + "o", self.c["width"])

    def recurrence(self, h, p, m):
        T, R, B = len(h), m["width"], m["blocks"]
        y = _gelu_tanh(self.times(h, p + "y", R, p + "y.b"))
        u = _conv(self.times(h, p + "x", R, p + "x.b"), self.w(p + "conv", R, m["conv"])) + self.w(p + "conv.b", R)
        n = R // B

        def gate(name):
            z = torch.stack([b @ w.T for b, w in zip(u.view(T, B, n).unbind(1), self.w(p + name, B, n, n))], 1)
            return torch.sigmoid(z + self.w(p + name + ".b", B, n)).reshape(T, R)
        a = torch.exp(-8.0 * gate("ra") * _softplus(self.w(p + "lam", R)))
        new, S, out = torch.sqrt(1.0 - a * a) * gate("ri") * u, h.new_zeros(R), []
        for t in range(T):
            S = a[t] * S + new[t]
            out.append(S)
        return self.times(torch.stack(out) * y, p + "o", self.c["width"])

    # -- Dinutar
    def run_dinutar(self, ids):
        c, eps = self.c, self.eps
        width, b = c["width"], c["embedding"]["bigram"]
        pair, out = self.w("bigram", b["buckets"] + 1, width), []
        for t, x in zip(ids, self.embedded(ids)):
            rows = torch.cat([t.new_tensor([b["buckets"]]), (t[:-1] * b["mul_prev"] + t[1:] * b["mul_cur"]) % b["buckets"]])
            x, held = _rms(x * c["embedding"]["scale"] + pair[rows], eps, self.ones("embed.norm", width)), {}
            for i, layer in enumerate(c["layers"]):
                p, m = f"l{i}.", layer["mixer"]
                if layer["type"] == "retention":
                    y = self.retention(x, p + "mix.", m)
                else:
                    if m.get("kv_from") is None:
                        held[i] = self.latent(x, p + "mix.", m, False)
                    y = self.latent_attention(x, p + "mix.", m, held[m.get("kv_from", i)], False).flatten(1)
                    y = self.times(y, p + "mix.o", width)
                x = _rms(c["postln_alpha"] * x + self.ones(p + "ls1", width) * y, eps, self.ones(p + "norm1", width))
                y = self.times(torch.relu(self.times(x, p + "mlp.up", layer["mlp"]["ff"])) ** 2, p + "mlp.down", width)
                x = _rms(c["postln_alpha"] * x + self.ones(p + "ls2", width) * y, eps, self.ones(p + "norm2", width))
            out.append(x)
        return out

    def latent(self, h, p, m, neighbours):
        L, R = m["kv_rank"], m["rot_dim"]
        down = self.times(h, p + "dkv", L + R)
        return _rms(down[:, :L], self.eps, self.ones(p + "dkv.norm", L)), _turn(down[:, L:].unsqueeze(1), m["rot"], neighbours)

    def latent_attention(self, h, p, m, held, neighbours, sink=None):
        T, H, D, R, E = len(h), m["heads"], m["dim"], m["rot_dim"], m["vdim"]
        c, shared = held
        q = self.times(h, p + "q", H * (D + R)).view(T, H, D + R)
        q = torch.cat([q[..., :D], _turn(q[..., D:], m["rot"], neighbours)], -1)
        k = torch.cat([self.times(c, p + "uk", H * D).view(T, H, D), shared.expand(T, H, R)], -1)
        return _attend(q, k, self.times(c, p + "uv", H * E).view(T, H, E), m["scale"], sink=sink)

    def retention(self, h, p, m):
        T, H, D, E = len(h), m["heads"], m["dim"], m["vdim"]
        q, k, v = (self.times(h, p + n, H * d).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
        keep = torch.tensor(m["decay"], dtype=torch.float64, device=h.device).view(1, H, 1).expand(T, H, 1)
        o = _linear_state(_turn(q, m["rot"]), _turn(k, m["rot"]) * D ** -0.5, v, keep)
        return self.times(_rms(o, self.eps).flatten(1) * _silu(self.times(h, p + "g", H * E)), p + "o", self.c["width"])

    # -- Rufusun
    def run_rufusun(self, ids):
        c, out = self.c, []
        width = c["width"]
        for x in self.embedded(ids):
            for i, layer in enumerate(c["layers"]):
                p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
                h = _rms(x, self.eps, 1.0 + self.w(p + "norm1", width))
                y = self.delta(h, p + "mix.", m) if layer["type"] == "delta" else self.capped(h, p + "mix.", m)
                h = _rms(x, self.eps, 1.0 + self.w(p + "norm2", width))
                if mlp["kind"] == "dense":
                    y = y + self.gated_ff(h, p + "mlp.", mlp["ff"])
                else:
                    def expert(q, rows, weights=1.0):
                        rows, ff, limit = rows * weights, mlp["expert"]["ff"], mlp["expert"]["limit"]
                        g, u = self.times(rows, q + "gate", ff).clamp(max=limit), self.times(rows, q + "up", ff).clamp(-limit, limit)
                        return self.times(g * torch.sigmoid(1.702 * g) * (u + 1.0), q + "down", width)
                    scores, chosen = torch.sigmoid(self.times(h, p + "mlp.router", mlp["router"]["experts"])).topk(mlp["router"]["top"])
                    y = y + self.experts(h, p + "mlp.", mlp["router"]["experts"], chosen, scores, expert) + expert(p + "mlp.shared.", h)
                x = x + y
            out.append(x)
        return out

    def capped(self, h, p, m):
        T, H, G, D = len(h), m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.times(h, p + n, a * D, p + n + ".b").view(T, a, D) for n, a in (("q", H), ("k", G), ("v", G)))
        o = _attend(_turn(q, m["rot"]), _turn(k, m["rot"]), v, m["scale"], cap=m["softcap"])
        return self.times(o.flatten(1), p + "o", self.c["width"], p + "o.b")

    def delta(self, h, p, m):
        T, H, G, D, E = len(h), m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (_silu(_conv(self.times(h, p + n, r), self.w(f"{p}{n}.conv", r, m["conv"]))).view(T, -1, d)
                   for n, r, d in (("q", G * D, D), ("k", G * D, D), ("v", H * E, E)))
        q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
        q, k = (q * D ** -0.5).repeat_interleave(H // G, 1), k.repeat_interleave(H // G, 1)
        beta = torch.sigmoid(self.times(h, p + "b", H)).unsqueeze(-1)
        keep = torch.exp(-torch.exp(self.w(p + "A_log", H)) * _softplus(self.times(h, p + "a", H) + self.w(p + "dt_bias", H)))
        S, out = h.new_zeros(H, D, E), []
        for t in range(T):
            S = keep[t].view(H, 1, 1) * S
            u = beta[t] * (v[t] - (k[t].unsqueeze(1) @ S).squeeze(1))
            S = S + k[t].unsqueeze(-1) * u.unsqueeze(1)
            out.append((q[t].unsqueeze(1) @ S).squeeze(1))
        o = _rms(torch.stack(out), self.eps, self.ones(p + "norm", E)).flatten(1)
        return self.times(o * _silu(self.times(h, p + "g", H * E)), p + "o", self.c["width"])

    # -- Tadalorn
    def run_tadalorn(self, ids):
        c, out = self.c, []
        width = c["width"]
        for x in self.embedded(ids):
            for i, layer in enumerate(c["layers"]):
                p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
                q = p + "mix."
                if layer["type"] == "latent_attention":
                    y = self.latent_attention(x, q, m, self.latent(x, q, m, True), True, self.w(q + "sink", m["heads"])).flatten(1)
                elif layer["type"] == "mlstm":
                    y = self.mlstm(x, q, m)
                else:
                    y = self.windowed(x, q, m)
                y = self.times(y * torch.sigmoid(self.times(x, q + "g", y.shape[1])), q + "o", width)
                x = x + c["residual_mult"] * _rms(y, self.eps, self.ones(p + "norm1", width))
                if mlp["kind"] == "dense":
                    y = self.gated_ff(x, p + "mlp.", mlp["ff"])
                else:
                    def expert(q, rows, weights=1.0):
                        z = self.times(rows, q + "up", mlp["expert"]["ff"])
                        return weights * self.times(0.5 * z * (1.0 + torch.erf(z / math.sqrt(2.0))), q + "down", width)
                    n = mlp["router"]["experts"]
                    best, chosen = self.times(x, p + "mlp.router", n, p + "mlp.router.b").topk(mlp["router"]["top"])
                    y = self.experts(x, p + "mlp.", n, chosen, torch.softmax(best, -1), expert) + expert(p + "mlp.shared.", x)
                x = x + c["residual_mult"] * _rms(y, self.eps, self.ones(p + "norm2", width))
            out.append(x)
        return out

    def windowed(self, h, p, m):
        T, H, G, D = len(h), m["heads"], m["kv_heads"], m["dim"]
        q, k = (_conv(self.times(h, p + n, a * D), self.w(f"{p}{n}.conv", a * D, m["conv"])) for n, a in (("q", H), ("k", G)))
        v = k.view(T, G, D)
        q, k = (_turn(_rms(z, self.eps, self.ones(f"{p}{n}.norm", a * D)).view(T, a, D), m["rot"], True) for z, n, a in ((q, "q", H), (k, "k", G)))
        i = torch.arange(T, device=h.device)
        dist = i.view(-1, 1) - i
        seen = (dist >= 0) & ((dist < m["mask"]["size"]) | (i < m["mask"]["keep_first"]))
        return _attend(q, k, v, m["scale"], seen, h.new_zeros(H)).flatten(1)

    def mlstm(self, h, p, m):
        T, H, D, E, cap = len(h), m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k, v = (self.times(h, p + n, H * d).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
        q = q * D ** -0.5
        take, keep = (cap * torch.tanh(self.times(h, p + n, H, f"{p}{n}.b") / cap) for n in ("i", "f"))
        keep = -_softplus(-keep)
        S, n, top, out = h.new_zeros(H, D, E), h.new_zeros(H, D), h.new_zeros(H), []
        for t in range(T):
            new = torch.maximum(keep[t] + top, take[t])
            a, b = torch.exp(keep[t] + top - new), torch.exp(take[t] - new)
            S = a.view(H, 1, 1) * S + (b.view(H, 1) * k[t]).unsqueeze(-1) * v[t].unsqueeze(1)
            n = a.view(H, 1) * n + b.view(H, 1) * k[t]
            top = new
            low = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
            out.append((q[t].unsqueeze(1) @ S).squeeze(1) / low.view(H, 1))
        return _rms(torch.stack(out), self.eps).flatten(1) * self.ones(p + "norm", H * E)

    # -- Darolix
    def run_darolix(self, ids):
        c, out = self.c, []
        width = c["width"]
        for x in self.embedded(ids):
            pos = torch.arange(len(x), dtype=torch.float64, device=x.device).view(-1, 1)
            angle = pos * 10000.0 ** (-2.0 * torch.arange(width // 2, dtype=torch.float64, device=x.device) / width)
            x = x * c["embedding"]["scale"] + torch.stack([torch.sin(angle), torch.cos(angle)], -1).flatten(1)
            for i, layer in enumerate(c["layers"]):
                p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
                h = _rms(x, self.eps, self.ones(p + "norm1", width))
                if layer["type"] == "mamba2":
                    y = self.mamba2(h, p + "mix.", m)
                else:
                    y = 0.5 * (_rms(self.tempered(h, p + "mix.left.", m["left"]), self.eps, self.ones(p + "mix.left.out", width))
                               + _rms(self.gated_linear(h, p + "mix.right.", m["right"]), self.eps, self.ones(p + "mix.right.out", width)))
                if mlp is not None:
                    n, top, ff = mlp["router"]["experts"], mlp["router"]["top"], mlp["expert"]["ff"]
                    total = n + mlp["router"]["identity"]
                    s = torch.softmax(self.times(h, p + "mlp.router", total), -1)
                    chosen = (s + self.w(p + "mlp.correction", total)).topk(top).indices
                    share = s.gather(1, chosen)
                    share = share / (share.sum(-1, keepdim=True) + 1e-20)
                    y = y + self.experts(h, p + "mlp.", total, chosen, share, lambda q, rows, weights: weights * (
                        self.gated_ff(rows, q, ff) if int(q.rsplit("e", 1)[1][:-1]) < n else rows))
                x = x + y
            out.append(x)
        return out

    def mamba2(self, h, p, m):
        T, H, E, N, G = len(h), m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * E
        z, xbc, dt = self.times(h, p + "in", 2 * inner + 2 * G * N + H).split([inner, inner + 2 * G * N, H], -1)
        xbc = _silu(_conv(xbc, self.w(p + "conv", inner + 2 * G * N, m["conv"])) + self.w(p + "conv.b", inner + 2 * G * N))
        x, B, C = xbc.split([inner, G * N, G * N], -1)
        x, (B, C) = x.view(T, H, E), (b.view(T, G, N).repeat_interleave(H // G, 1) for b in (B, C))
        dt = _softplus(dt + self.w(p + "dt_bias", H)).unsqueeze(-1)
        keep = torch.exp(-torch.exp(self.w(p + "A_log", H)).view(1, H, 1) * dt)
        y = _linear_state(C, B, dt * x, keep) + self.ones(p + "D", H).view(1, H, 1) * x
        y = (y.reshape(T, inner) * _silu(z)).view(T, m["norm_groups"], -1)
        return self.times(_rms(y, self.eps).reshape(T, inner) * self.ones(p + "norm", inner), p + "o", self.c["width"])

    def tempered(self, h, p, m):
        T, H, G, D = len(h), m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (self.times(h, p + n, a * D).view(T, a, D) for n, a in (("q", H), ("k", G), ("v", G)))
        at = torch.arange(1, T + 1, device=h.device) // m["q_temp"]["every"]
        q = _rms(q, self.eps) * (1.0 + m["q_temp"]["coef"] * torch.log(at.double() + 1.0)).view(T, 1, 1)
        return self.times(_attend(q, _rms(k, self.eps), v, m["scale"], cap=m["softcap"]).flatten(1), p + "o", self.c["width"])

    def gated_linear(self, h, p, m):
        T, H, D, E = len(h), m["heads"], m["dim"], m["vdim"]
        q, k, v = (self.times(h, p + n, H * d).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
        z = self.times(self.times(h, p + "a1", 16), p + "a2", H * D, p + "a2.b")
        keep = torch.exp(-_softplus(-z) / m["tau"]).view(T, H, D)
        o = _rms(_linear_state(q * D ** -0.5, k, v, keep), self.eps, self.ones(p + "norm", E)).flatten(1)
        return self.times(o * _silu(self.times(h, p + "g", H * E)), p + "o", self.c["width"])

    # -- Vulosun
    def run_vulosun(self, ids):
        c, out = self.c, []
        for x in self.embedded(ids):
            held = {}
            for i, layer in enumerate(c["layers"]):
                p, m, mlp = f"l{i}.", layer["mixer"], layer["mlp"]
                h = self.layer_norm(x, p + "norm1")
                if layer["type"] == "parallel":
                    y = m["left_scale"] * self.head_normed(h, p + "mix.left.", m["left"]) + m["right_scale"] * self.lightning(h, p + "mix.right.", m["right"])
                elif layer["type"] == "attention":
                    y = self.row_normed(h, p + "mix.", m)
                else:
                    if m.get("kv_from") is None:
                        held[i] = self.two_keys(h, p + "mix.", m)
                    y = self.differential(h, p + "mix.", m, *held[m.get("kv_from", i)])
                x = x + self.layer_norm(y, p + "norm1b")
                h, ff = self.layer_norm(x, p + "norm2"), p + "mlp."
                y = self.gated_ff(h, ff, mlp["ff"]) if mlp["kind"] == "dense" else self.grouped_experts(h, ff, mlp)
                x = x + self.layer_norm(y, p + "norm2b")
            out.append(x)
        return out

    def grouped_experts(self, h, p, mlp):
        r, T = mlp["router"], len(h)

        def expert(q, rows, weights=1.0):
            return weights * self.times(torch.relu(self.times(rows, q + "up", mlp["expert"]["ff"])) ** 2, q + "down", h.shape[1])
        s = torch.sigmoid(self.times(h, p + "router", r["experts"]))
        groups = s.view(T, r["groups"]["count"], -1)
        kept = groups.topk(2).values.sum(-1).topk(r["groups"]["keep"]).indices
        allowed = torch.zeros(groups.shape[:2], dtype=torch.bool, device=h.device).scatter(1, kept, True)
        best, chosen = groups.masked_fill(~allowed.unsqueeze(-1), -math.inf).view(T, -1).topk(r["top"])
        return self.experts(h, p, r["experts"], chosen, r["scale"] * best, expert) + expert(p + "shared.", h)

    def row_normed(self, h, p, m):
        T, H, G, D = len(h), m["heads"], m["kv_heads"], m["dim"]
        q, k = (_turn(_rms(self.times(h, p + n, a * D), self.eps, self.ones(f"{p}{n}.norm", a * D)).view(T, a, D), m["rot"], True)
                for n, a in (("q", H), ("k", G)))
        o = _attend(q, k, self.times(h, p + "v", G * D).view(T, G, D), m["scale"])
        return self.times((o * torch.sigmoid(self.times(h, p + "g", H)).unsqueeze(-1)).flatten(1), p + "o", self.c["width"])

    def head_normed(self, h, p, m):
        T, H, G, D = len(h), m["heads"], m["kv_heads"], m["dim"]
        q, k = (_turn(_rms(self.times(h, p + n, a * D).view(T, a, D), self.eps, self.ones(f"{p}{n}.norm", D)), m["rot"])
                for n, a in (("q", H), ("k", G)))
        o = _attend(q, k, self.times(h, p + "v", G * D).view(T, G, D), m["scale"], sink=self.w(p + "sink", H))
        return self.times(o.flatten(1), p + "o", self.c["width"])

    def two_keys(self, h, p, m):
        T, G, D, E = len(h), m["kv_heads"], m["dim"], m["vdim"]
        k = _turn(self.times(h, p + "k", G * 2 * D, p + "k.b").view(T, 2 * G, D), m["rot"], True)
        return k.view(T, G, 2, D), self.times(h, p + "v", G * E, p + "v.b").view(T, G, E)

    def differential(self, h, p, m, k, v):
        T, H, D, E = len(h), m["heads"], m["dim"], m["vdim"]
        q = _turn(self.times(h, p + "q", H * 2 * D, p + "q.b").view(T, 2 * H, D), m["rot"], True).view(T, H, 2, D)
        i = torch.arange(T, device=h.device)
        chunk = i // m["mask"]["size"]
        seen = (i.view(-1, 1) >= i) & (chunk.view(-1, 1) == chunk)
        a, b = (_attend(q[:, :, j], k[:, :, j], v, m["scale"], seen) for j in (0, 1))
        l1, l2 = (torch.exp((self.w(p + "lq" + n, D) * self.w(p + "lk" + n, D)).sum()) for n in "12")
        o = _rms(a - (l1 - l2 + m["diff"]) * b, self.eps) * (1.0 - m["diff"])
        return self.times((o * torch.sigmoid(self.times(h, p + "g", H)).unsqueeze(-1)).flatten(1), p + "o", self.c["width"])

    def lightning(self, h, p, m):
        T, H, D, E = len(h), m["heads"], m["dim"], m["vdim"]
        q, k, v = (_silu(self.times(h, p + n, H * d)).view(T, H, d) for n, d in (("q", D), ("k", D), ("v", E)))
        keep = torch.tensor(m["decay"], dtype=torch.float64, device=h.device).view(1, H, 1).expand(T, H, 1)
        o = _rms(_linear_state(q, k, v, keep).flatten(1), self.eps, self.ones(p + "norm", H * E))
        return self.times(o * torch.sigmoid(self.times(h, p + "g", H * E)), p + "o", self.c["width"])
