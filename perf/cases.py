"""What the speed of this library is measured on: steps of whole models through Engine.step, and the sampler.

The models are the ones that bench.py measures, with their layer sizes and random weights: the dense decoder (Llama-3.2-1B whole; eight layers of
the Llama-3.1-8B and Qwen3-14B sizes, whole vocabularies), and the Nipulorn design with four layers of 2,048 or 4,096 channels and the Batodra and
Zogurax designs with eight.  (Random layers pass rounding errors on, with a little gain each: at 32 of them the logits in bfloat16 are 4 % from those in 64 bits,
and two correct implementations as far from each other, at eight 2 %.)  A design whose experts are chosen
by a learned router (Zasidra, Peponex, Zisedra) is left out: two correct implementations may choose another expert where two scores lie closer
than bfloat16 resolves, after which their logits have nothing to do with each other.  Zogurax's experts are chosen by a table over token ids.

A case is one of four kinds of work:

  prompt   new sequences, their whole prompts in one step, the logits of each sequence's last token; the sequences are given up again
  decode   sequences that are in the cache already, a few single-token steps with given tokens, the logits of every step; the pass starts by
           forgetting what the last one added
  request  new sequences: their prompts in one step, then single-token steps, the logits of every step; the sequences are given up again
  sample   drawing a token for each row of a batch of logits

A model stays loaded for the cases and passes that share it, as in a server; tokens are new for every seed."""
import importlib
import math

import numpy as np
import torch

llogos = importlib.import_module("daisi-llogos_amd")

# ---------------------------------------------------------------------------------------------------------------------------------------
# models
# ---------------------------------------------------------------------------------------------------------------------------------------

_LAYERS = 8
_LLAMA_ROPE = {"rope_type": "llama3", "factor": 8.0, "low_freq_factor": 1.0, "high_freq_factor": 4.0, "original_max_position_embeddings": 8192}
_LLAMA_8B = {
    "architectures": ["LlamaForCausalLM"], "vocab_size": 128256, "hidden_size": 4096, "intermediate_size": 14336,
    "num_hidden_layers": _LAYERS, "num_attention_heads": 32, "num_key_value_heads": 8, "head_dim": 128, "rms_norm_eps": 1e-5,
    "rope_theta": 500000.0, "max_position_embeddings": 131072, "rope_scaling": _LLAMA_ROPE, "attention_bias": False,
    "tie_word_embeddings": False, "torch_dtype": "bfloat16", "eos_token_id": 128001,
}
_DENSE = {
    "llama-3.1-8b": _LLAMA_8B,
    "llama-3.2-1b": dict(_LLAMA_8B, hidden_size=2048, intermediate_size=8192, num_hidden_layers=16, head_dim=64, tie_word_embeddings=True,
                         rope_scaling=dict(_LLAMA_ROPE, factor=32.0)),
    "qwen3-14b": {
        "architectures": ["Qwen3ForCausalLM"], "vocab_size": 151936, "hidden_size": 5120, "intermediate_size": 17408,
        "num_hidden_layers": _LAYERS, "num_attention_heads": 40, "num_key_value_heads": 8, "head_dim": 128, "rms_norm_eps": 1e-6,
        "rope_theta": 1000000.0, "max_position_embeddings": 40960, "attention_bias": False, "tie_word_embeddings": False,
        "torch_dtype": "bfloat16", "eos_token_id": 151645,
    },
}
_DESIGNS = ("nipulorn", "batodra", "zogurax")
_FEED_FORWARD = {2048: 8192, 4096: 14336}       # of the dense decoder of the same width
_VOCAB = 32000


def _nipulorn(width):
    """Three layers of a matrix-state recurrence and one of latent attention; two matrices a feed-forward instead of three, half as wide again."""
    ff = {"kind": "dense", "ff": _FEED_FORWARD[width] * 3 // 2}
    wkv = {"type": "wkv", "mixer": {"heads": width // 64, "dim": 64, "decay_rank": 64}, "mlp": ff}
    lat = {"type": "latent_attention", "mlp": ff,
           "mixer": {"heads": width // 128, "dim": 128, "rot_dim": 64, "vdim": 128, "q_rank": 3 * width // 8, "kv_rank": 512, "scale": 192 ** -0.5,
                     "rot": {"base": 10000.0, "dims": 64, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
    return {"architecture": "Nipulorn", "vocab": _VOCAB, "width": width, "embedding": {"scale": 1.0}, "logit_scale": 1.0, "norm": {"eps": 1e-5},
            "canon": {"taps": 4}, "layers": [wkv, wkv, wkv, lat], "torch_dtype": "bfloat16"}


def _batodra(width):
    """A gated linear recurrence, window attention that keeps the first tokens, a recurrence, differential attention, in turn."""
    heads = width // 128
    kv = max(1, heads // 4)
    ff = {"kind": "dense", "ff": _FEED_FORWARD[width] * 3 // 2}
    rec = {"type": "rglru", "mixer": {"width": width, "blocks": width // 256, "conv": 4}, "mlp": ff}
    win = {"type": "attention_2", "mlp": ff,
           "mixer": {"heads": heads, "kv_heads": kv, "dim": 128, "vdim": 128, "scale": 0.125, "mask": {"size": 1024, "keep_first": 4},
                     "rot": {"base": 500000.0, "dims": 128, "scaling": {"factor": 8.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
    dif = {"type": "attention", "mlp": ff,
           "mixer": {"heads": heads, "kv_heads": kv, "dim": 64, "vdim": 128, "scale": 0.125, "diff": 0.5, "rot": {"base": 500000.0, "dims": 64}}}
    return {"architecture": "Batodra", "vocab": _VOCAB, "width": width, "norm": {"eps": 1e-5}, "postln_alpha": 2.0,
            "layers": [(rec, win, rec, dif)[i % 4] for i in range(_LAYERS)], "torch_dtype": "bfloat16"}


def _zogurax(width):
    """Two attention forms in turn, 16 experts of which a token takes 2 beside a shared one, the second and third layer gone through twice."""
    heads, ff = width // 128, _FEED_FORWARD[width] // 2
    moe = {"kind": "moe", "router": {"experts": 16, "top": 2}, "expert": {"ff": ff}, "shared": {"ff": ff}}
    mixer = {"heads": heads, "kv_heads": max(1, heads // 4), "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "softcap": 50.0,
             "q_temp": {"coef": 0.3, "every": 128}}
    first, second = {"type": "attention", "mixer": dict(mixer, conv=4), "mlp": moe}, {"type": "attention_2", "mixer": mixer, "mlp": moe}
    return {"architecture": "Zogurax", "vocab": _VOCAB, "width": width, "norm": {"eps": 1e-5}, "loop": {"start": 1, "stop": 3, "times": 2},
            "layers": [second if i % 2 == 0 else first for i in range(_LAYERS - 2)], "torch_dtype": "bfloat16"}


def _config(case):
    if case["model"] in _DENSE:
        return dict(_DENSE[case["model"]], torch_dtype=case["dtype"])
    return {"nipulorn": _nipulorn, "batodra": _batodra, "zogurax": _zogurax}[case["model"]](case["width"])


def _vocab(case):
    return _DENSE[case["model"]]["vocab_size"] if case["model"] in _DENSE else _VOCAB


# ---------------------------------------------------------------------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------------------------------------------------------------------

def _dense(name, model, kind, sequences, longest, shortest, steps=0, dtype="bfloat16"):
    return {"name": name, "kind": kind, "model": model, "dtype": dtype, "sequences": sequences, "longest": longest, "shortest": shortest, "steps": steps}


def _design(name, model, sequences, longest, shortest, steps, width=4096):
    return dict(_dense(name, model, "request", sequences, longest, shortest, steps), width=width)


def listed():
    return [
        # one user's chat with a small model: the smallest step there is, where launches and latency count
        _dense("1b-decode-1", "llama-3.2-1b", "decode", 1, 211, 211, 8),
        # few users on one GPU: the library's headline batch
        _dense("8b-decode-8", "llama-3.1-8b", "decode", 8, 700, 300, 8),
        # a server's full batch, contexts of every length
        _dense("8b-decode-64", "llama-3.1-8b", "decode", 64, 400, 30, 4),
        # long documents: the cache weighs as much as the matrices
        _dense("1b-decode-long", "llama-3.2-1b", "decode", 8, 8190, 4100, 4),
        # a handful of short chat turns that arrive together
        _dense("8b-prompts-short", "llama-3.1-8b", "prompt", 5, 130, 9),
        # the headline prompt
        _dense("8b-prompt-2048", "llama-3.1-8b", "prompt", 1, 2048, 2048),
        # a document into a larger model with per-head norms, an odd length
        _dense("14b-prompt-5003", "qwen3-14b", "prompt", 1, 5003, 5003),
        # the true 32-bit engine: replaying and checking a model in full precision
        _dense("1b-float32", "llama-3.2-1b", "request", 2, 515, 190, 8, "float32"),
        # the other designs: chats of a few users, a long one by itself, and short ones
        _design("nipulorn-8", "nipulorn", 8, 600, 250, 16),
        _design("batodra-1", "batodra", 1, 2500, 2500, 16),
        _design("zogurax-4", "zogurax", 4, 400, 130, 16),
        # drawing a token for a full batch with the usual settings
        {"name": "sample-64", "kind": "sample", "rows": 64, "vocab": 128256, "temperature": 0.7, "top_k": 40, "top_p": 0.9, "penalty": 1.1},
    ]


def _log(rng, low, high):
    """A whole number from low to high, spread evenly over its logarithm."""
    return int(min(high, max(low, round(math.exp(rng.uniform(math.log(low - 0.5), math.log(high + 0.5)))))))


def draw(rng):
    what = rng.choice(("decode", "decode", "decode", "prompt", "prompt", "prompt", "design", "design", "design", "float32", "sample"))
    if what == "sample":
        return {"kind": "sample", "rows": _log(rng, 1, 64), "vocab": rng.choice((32000, 128256, 151936)),
                "temperature": round(rng.uniform(0.3, 1.2), 2), "top_k": rng.choice((20, 40, 100)), "top_p": rng.choice((0.8, 0.9, 0.95, 1.0)),
                "penalty": rng.choice((1.0, 1.1))}
    if what == "design":
        sequences = _log(rng, 1, 8)
        model = rng.choice(_DESIGNS)
        # (the norm on a Nipulorn head's sums divides by next to nothing in a sequence's first tokens, where rounding then decides)
        least = 100 if model == "nipulorn" else 1
        longest = _log(rng, least, 4096 // sequences)
        case = _design(None, model, sequences, longest, _log(rng, least, longest), rng.randint(2, 16), rng.choice((2048, 4096)))
    elif what == "float32":
        sequences = _log(rng, 1, 8)
        longest = _log(rng, 1, 1024 // sequences)
        case = _dense(None, "llama-3.2-1b", "request", sequences, longest, _log(rng, 1, longest), rng.randint(2, 8), "float32")
    elif what == "decode":
        model = rng.choice(("llama-3.2-1b", "llama-3.1-8b", "qwen3-14b"))
        sequences = _log(rng, 1, 64)
        longest = _log(rng, 4, min(16000, {"llama-3.2-1b": 65000, "llama-3.1-8b": 24000, "qwen3-14b": 10000}[model] // sequences))
        case = _dense(None, model, "decode", sequences, longest, _log(rng, 2, longest), rng.randint(2, 8))
    else:
        model = rng.choice(("llama-3.2-1b", "llama-3.1-8b", "qwen3-14b"))
        sequences = _log(rng, 1, 8)
        longest = _log(rng, 2, {"llama-3.2-1b": 12000, "llama-3.1-8b": 6000, "qwen3-14b": 4500}[model] // sequences)
        case = _dense(None, model, "prompt", sequences, longest, _log(rng, 1, longest))
    del case["name"]
    return case


def _lengths(case):
    """Tokens of each sequence: the longest first, the last the shortest, the others at odd places between."""
    n, a, b = case["sequences"], case["longest"], case["shortest"]
    if n == 1:
        return [a]
    return [a] + [b + (a - b) * ((7 * i) % n) // n for i in range(1, n - 1)] + [b]


# ---------------------------------------------------------------------------------------------------------------------------------------
# inputs and passes
# ---------------------------------------------------------------------------------------------------------------------------------------

_loaded = {}            # the one model that is loaded: its key -> engine


def _engine(case):
    lens = _lengths(case)
    key = (case["model"], case["dtype"], case.get("width"))
    # room for the sequences of four states, rounded up so that a model serves cases of several sizes
    slots = 4 * case["sequences"] if case["kind"] == "decode" else case["sequences"]
    tokens = sum(n + case["steps"] + 64 for n in lens) * (4 if case["kind"] == "decode" else 1)
    engine = _loaded.get(key)
    if engine is None or engine.cache.slots.n_slots < slots or min(engine.cache.free_pages()) * 64 < tokens // 4:
        _loaded.clear()
        del engine
        torch.cuda.empty_cache()
        engine = _loaded[key] = llogos.Engine.from_config(_config(case), seed=11, dtype=case["dtype"], max_tokens=max(16384, tokens), n_slots=max(32, slots))
    return engine


class _Sequences:
    """Slots of an engine, given back when the state that holds them goes."""

    def __init__(self, engine, count):
        self.engine, self.slots = engine, [engine.alloc_slot() for _ in range(count)]

    def __del__(self):
        for s in self.slots:
            self.engine.free_slot(s)


def _tokens(case, seed):
    """Of each sequence: its prompt or context, and one more token for every single-token step."""
    rng = np.random.default_rng([seed, 77])
    return [rng.integers(0, _vocab(case), size=n + case["steps"]).tolist() for n in _lengths(case)]


def prepare(case, seed):
    if case["kind"] == "sample":
        g = torch.Generator(device="cuda").manual_seed(seed)
        rows = case["rows"]
        rng = np.random.default_rng([seed, 78])
        params = llogos.GenerationParams(temperature=case["temperature"], top_k=case["top_k"], top_p=case["top_p"],
                                         repetition_penalty=case["penalty"], seed=seed)
        # logits as a trained model gives them: most of the mass on few tokens
        logits = torch.randn(rows, case["vocab"], device="cuda", generator=g) * 3.0
        return {"sampler": llogos.Sampler(params), "logits": logits, "requests": list(range(rows)), "indices": [int(i) for i in rng.integers(0, 200, size=rows)],
                "histories": [rng.integers(0, case["vocab"], size=int(n)).tolist() for n in rng.integers(20, 300, size=rows)]}
    engine = _engine(case)
    lens, tokens = _lengths(case), _tokens(case, seed)
    state = {"kind": case["kind"], "engine": engine, "lens": lens,
             "prompts": [t[:n] for t, n in zip(tokens, lens)],
             "next": [[[t[n + s]] for t, n in zip(tokens, lens)] for s in range(case["steps"])]}
    if case["kind"] == "decode":
        state["sequences"] = _Sequences(engine, len(lens))
        entries = list(zip(state["sequences"].slots, state["prompts"]))
        while entries:                               # contexts go in a few thousand tokens at a time
            n, some = 0, []
            while entries and (not some or n + len(entries[0][1]) <= 16384):
                n += len(entries[0][1])
                some.append(entries.pop(0))
            engine.step(some, want=None)
    return state


def run(state):
    if "sampler" in state:
        return state["sampler"].sample(state["logits"], state["requests"], state["indices"], state["histories"])
    engine = state["engine"]
    if state["kind"] == "decode":
        slots = state["sequences"].slots
        for s, n in zip(slots, state["lens"]):
            engine.cache.truncate(s, n)
        return [engine.step(list(zip(slots, tokens)), want="last") for tokens in state["next"]]
    slots = [engine.alloc_slot() for _ in state["prompts"]]
    try:
        out = [engine.step(list(zip(slots, state["prompts"])), want="last")]
        for tokens in state["next"]:
            out.append(engine.step(list(zip(slots, tokens)), want="last"))
    finally:
        for s in slots:
            engine.free_slot(s)
    return out


# ---------------------------------------------------------------------------------------------------------------------------------------
# what a pass cannot do without, and how exact it can be
# ---------------------------------------------------------------------------------------------------------------------------------------

def _layer_costs(case):
    """Of every layer run: (matrix elements all of which a step reads, matrix elements a token is multiplied with, [experts, chosen, elements
    of one] or None, key and value elements a position, flops a (query, key) pair, most keys a query sees, elements of state a sequence)."""
    cfg = _config(case)
    if case["model"] in _DENSE:
        h, i = cfg["hidden_size"], cfg["intermediate_size"]
        q, kv = cfg["num_attention_heads"] * cfg["head_dim"], cfg["num_key_value_heads"] * cfg["head_dim"]
        n = h * (q + 2 * kv) + q * h + 3 * h * i
        return [(n, n, None, 2 * kv, 4 * q, math.inf, 0)] * cfg["num_hidden_layers"]
    w, out = cfg["width"], []
    for layer in cfg["layers"]:
        m, f = layer["mixer"], layer["mlp"]
        if layer["type"] == "wkv":
            c = m["heads"] * m["dim"]
            costs = [5 * w * c + m["decay_rank"] * (w + c), None, 0, 0, 0, c * m["dim"] + 3 * w]
        elif layer["type"] == "latent_attention":
            hd, r = m["heads"], m["kv_rank"]
            n = w * m["q_rank"] + m["q_rank"] * hd * (m["dim"] + m["rot_dim"]) + w * (r + m["rot_dim"]) + hd * r * (m["dim"] + m["vdim"]) + hd * m["vdim"] * w
            costs = [n, None, r + m["rot_dim"], 2 * hd * (m["dim"] + m["rot_dim"] + m["vdim"]), math.inf, 2 * w]
        elif layer["type"] == "rglru":
            c = m["width"]
            costs = [3 * w * c + 2 * c * c // m["blocks"], None, 0, 0, 0, 4 * c]
        else:
            maps = 2 if "diff" in m else 1
            q, k, v = m["heads"] * maps * m["dim"], m["kv_heads"] * maps * m["dim"], m["kv_heads"] * m["vdim"]
            o = m["heads"] * m["vdim"]
            keys = m["mask"]["size"] + m["mask"]["keep_first"] if "mask" in m else math.inf
            costs = [w * (q + k + v + o), None, k + v, 2 * (q + maps * o), keys, 0]
        if f["kind"] == "moe":
            one = 2 * w * f["expert"]["ff"]
            costs[0] += 2 * w * f["shared"]["ff"]
            costs[1] = (f["router"]["experts"], f["router"]["top"], one)
            per_token = costs[0] + f["router"]["top"] * one
        else:
            costs[0] += 2 * w * f["ff"]
            per_token = costs[0]
        out.append((costs[0], per_token) + tuple(costs[1:]))
    loop = cfg.get("loop")
    if loop:                                           # runs of the looped layers, each pass opened by a product of [x ; x0]
        runs = out[loop["start"]:loop["stop"]] * loop["times"]
        enter = [(2 * w * w, 2 * w * w, None, 0, 0, 0, 0)] * loop["times"]
        out = out[:loop["start"]] + runs + enter + out[loop["stop"]:]
    return out


def work(case):
    if case["kind"] == "sample":
        n = case["rows"] * case["vocab"]
        return {"bytes": 4 * n, "flops": 2 * n}
    layers, lens, size = _layer_costs(case), _lengths(case), 4 if case["dtype"] == "float32" else 2
    head = (_DENSE[case["model"]]["hidden_size"] if case["model"] in _DENSE else case["width"]) * _vocab(case)
    total = {"bytes": 0.0, "flops": 0.0}

    def step(before, new):
        """`new` tokens for each of the sequences that hold `before`."""
        tokens, rows = sum(new), len(new)
        total["bytes"] += size * head + 4 * rows * _vocab(case)
        total["flops"] += 2 * head * rows
        for matrices, per_token, experts, kv, pair, most, state in layers:
            total["bytes"] += size * matrices
            if experts:                                 # experts that at least one token names, on average
                n, top, one = experts
                total["bytes"] += size * one * n * (1 - (1 - top / n) ** tokens)
            total["flops"] += 2 * per_token * tokens
            for b, c in zip(before, new):
                total["bytes"] += size * kv * (min(b, most) + c) + 8 * state
                total["flops"] += pair * sum(min(b + i + 1, most) for i in (range(c) if most < math.inf else ())) if most < math.inf else \
                    pair * (c * b + c * (c + 1) / 2)
    if case["kind"] != "decode":
        step([0] * len(lens), lens)
    for s in range(case["steps"]):
        step([n + s for n in lens], [1] * len(lens))
    return total


def tolerance(case):
    if case["kind"] == "sample":
        return "exact"                                  # token ids
    # measured against 64 bits: 1.0e-6 to 2.0e-6 in 32 bits (single logits up to 1.1e-5 of the root mean square)
    if case["dtype"] == "float32":
        return {"rel": 8e-6, "max": 5e-5}
    # bfloat16, where every layer rounds what it hands on to 8 bits: 0.005 to 0.006 with Zogurax's plain sum of both sublayers, 0.007 to 0.013
    # with the norms of Nipulorn and Batodra, 0.012 to 0.023 with the dense decoder (single logits up to 0.13)
    return {"rel": 0.02, "max": 0.2} if case["model"] == "zogurax" else {"rel": 0.03, "max": 0.5}


# ---------------------------------------------------------------------------------------------------------------------------------------
# the same passes in 64 bits: whole sequences, no cache, plain torch
# ---------------------------------------------------------------------------------------------------------------------------------------

_RANGES = {"norm": (0.9, 1.1), "offset": (-0.1, 0.1), "unit": (0.0, 0.8), "decay": (-6.0, -0.5), "sink": (0.0, 4.0), "shape": (-1.5, 0.5),
           "taps": (-0.5, 0.5), "bonus": (-0.5, 1.5)}


class _Weights:
    """The random weights of a model: element i of a tensor depends on the seed, the tensor's name and i alone (an integer hash; uniform in
    the kind's range, or N(0, 0.02) from two uniforms), rounded to the type the model is stored in."""

    def __init__(self, dtype):
        self.dtype = getattr(torch, dtype)

    @staticmethod
    def _mix(x):
        x = (x ^ (x >> 16)) * 0x7FEB352D & 0xFFFFFFFF
        x = (x ^ (x >> 15)) * 0x846CA68B & 0xFFFFFFFF
        return x ^ (x >> 16)

    def _hash(self, name, first, count):
        import hashlib
        digest = hashlib.sha256(f"11:{name}".encode()).digest()
        a, b = int.from_bytes(digest[:4], "little"), int.from_bytes(digest[4:8], "little")
        i = torch.arange(first, first + count, dtype=torch.int64, device="cuda")
        return self._mix(self._mix((i + a) & 0xFFFFFFFF) ^ b)

    def stored(self, name, *shape, kind="matrix"):
        n = math.prod(shape)
        out = torch.empty(n, dtype=self.dtype, device="cuda")
        for first in range(0, n, 1 << 26):
            count = min(1 << 26, n - first)
            h = self._hash(name, first, count)
            u = (h >> 8).double()
            if kind in _RANGES:
                low, high = _RANGES[kind]
                values = low + u * ((high - low) / (1 << 24))
            else:
                turn = (self._mix(h ^ 0x9E3779B9) >> 8).double() * (1.0 / (1 << 24))
                values = torch.sqrt(-2.0 * torch.log((u + 1.0) * (1.0 / (1 << 24)))) * torch.cos((2.0 * math.pi) * turn) * 0.02
            out[first:first + count] = values.to(self.dtype)
        return out.view(shape)

    def __call__(self, name, *shape, kind="matrix"):
        return self.stored(name, *shape, kind=kind).double()

    def choices(self, name, rows, top, n):
        """Every row names `top` neighbouring numbers below n, from a start of its own."""
        start = self._hash(name, 0, rows) % n
        return (start[:, None] + torch.arange(top, device="cuda")[None, :]) % n


def _unit(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _frequencies(dims, base, scaling):
    """(turns a position, stretch of cos and sin): plain, with the Llama-3 rule, or with the YaRN rule."""
    f = torch.tensor([base ** (-2.0 * i / dims) for i in range(dims // 2)], dtype=torch.float64, device="cuda")
    if not scaling:
        return f, 1.0
    if scaling.get("rope_type") == "llama3":
        low, high = scaling["low_freq_factor"], scaling["high_freq_factor"]
        kept = ((scaling["original_max_position_embeddings"] * f / (2 * math.pi) - low) / (high - low)).clamp(0, 1)
        return f * ((1 - kept) / scaling["factor"] + kept), 1.0
    at = lambda turns: dims * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(base))
    low, high = max(math.floor(at(scaling["fast"])), 0), min(math.ceil(at(scaling["slow"])), dims - 1)
    ramp = ((torch.arange(dims // 2, device="cuda").double() - low) / max(high - low, 0.001)).clamp(0, 1)
    return f / scaling["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0


def _turn(x, f, stretch, pairs="halves"):
    """x [T, heads, D] of positions 0, 1, ...: the first 2 len(f) dimensions turned, i with i + len(f), or neighbours."""
    angle = torch.arange(x.shape[0], device="cuda").double()[:, None] * f[None, :]
    c, s = (angle.cos() * stretch)[:, None, :], (angle.sin() * stretch)[:, None, :]
    n, out = len(f), x.clone()
    first, second = (slice(0, n), slice(n, 2 * n)) if pairs == "halves" else (slice(0, 2 * n, 2), slice(1, 2 * n, 2))
    a, b = x[..., first], x[..., second]
    out[..., first], out[..., second] = a * c - b * s, b * c + a * s
    return out


def _attend(q, k, v, scale, window=0, keep=0, cap=0.0, sink=None):
    """q [T, H, D], k [T, G, D], v [T, G, E] of one sequence -> [T, H, E]; `sink`: a score a head that joins the denominator alone."""
    T, H, D = q.shape
    G, E = v.shape[1:]
    q, k, v = q.view(T, G, H // G, D).permute(1, 2, 0, 3), k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    out = torch.empty(T, H, E, dtype=torch.float64, device="cuda")
    rows = max(16, min(T, (1 << 27) // (H * T)))
    for a in range(0, T, rows):
        b = min(T, a + rows)
        s = torch.matmul(q[:, :, a:b].reshape(G, -1, D), k[:, :, :b]).view(G, H // G, b - a, b) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        i, j = torch.arange(a, b, device="cuda")[:, None], torch.arange(b, device="cuda")[None, :]
        seen = j <= i
        if window:
            seen = seen & ((i - j < window) | (j < keep))
        s = s.masked_fill(~seen, -math.inf)
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            z = sink.view(G, H // G, 1, 1)
            top = torch.maximum(top, z)
        e = torch.exp(s - top)
        den = e.sum(-1, keepdim=True) + (torch.exp(z - top) if sink is not None else 0.0)
        o = torch.matmul(e.view(G, -1, b), v[:, :b]).view(G, H // G, b - a, E) / den
        out[a:b] = o.permute(2, 0, 1, 3).reshape(b - a, H, E)
    return out


def _each(spans, f, *rows):
    """f over the rows of each sequence."""
    return torch.cat([f(*(r[a:b] for r in rows)) for a, b in spans])


def _convolve(x, taps):
    """Causal, a channel at a time: the last column of taps [channels, n] weighs the present row."""
    n = taps.shape[1]
    full = torch.cat([x.new_zeros(n - 1, x.shape[1]), x])
    return sum(taps[:, j] * full[j:j + x.shape[0]] for j in range(n))


def _before(x):
    return torch.cat([torch.zeros_like(x[:1]), x[:-1]])


def _exact_dense(cfg, W, ids, spans, rows):
    H, G, D, h, i, eps = (cfg[k] for k in ("num_attention_heads", "num_key_value_heads", "head_dim", "hidden_size", "intermediate_size", "rms_norm_eps"))
    f, stretch = _frequencies(D, cfg["rope_theta"], cfg.get("rope_scaling"))
    per_head = cfg["architectures"][0].startswith("Qwen3")
    table = W.stored("model.embed_tokens.weight", cfg["vocab_size"], h)
    x = table[ids].double()
    for n in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{n}."
        y = _unit(x, eps) * W(p + "input_layernorm.weight", h, kind="norm")
        q, k, v = (y @ W(p + f"self_attn.{c}_proj.weight", m * D, h).T for c, m in (("q", H), ("k", G), ("v", G)))
        q, k, v = q.view(-1, H, D), k.view(-1, G, D), v.view(-1, G, D)
        if per_head:
            q, k = (_unit(t, eps) * W(p + f"self_attn.{c}_norm.weight", D, kind="norm") for t, c in ((q, "q"), (k, "k")))
        a = _each(spans, lambda q, k, v: _attend(_turn(q, f, stretch), _turn(k, f, stretch), v, D ** -0.5), q, k, v)
        x = x + a.reshape(-1, H * D) @ W(p + "self_attn.o_proj.weight", h, H * D).T
        y = _unit(x, eps) * W(p + "post_attention_layernorm.weight", h, kind="norm")
        g = torch.nn.functional.silu(y @ W(p + "mlp.gate_proj.weight", i, h).T)
        g *= y @ W(p + "mlp.up_proj.weight", i, h).T
        x = x + g @ W(p + "mlp.down_proj.weight", h, i).T
    x = _unit(x[rows], eps) * W("model.norm.weight", h, kind="norm")
    head = table if cfg["tie_word_embeddings"] else W.stored("lm_head.weight", cfg["vocab_size"], h)
    return x @ head.double().T


def _padded(spans, *rows):
    """[longest, sequences, ...] copies of the rows, zeros behind a sequence's end, and the way back."""
    longest = max(b - a for a, b in spans)
    place = torch.cat([torch.arange(b - a, device="cuda") * len(spans) + s for s, (a, b) in enumerate(spans)])
    out = []
    for r in rows:
        full = r.new_zeros((longest * len(spans),) + tuple(r.shape[1:]))
        full[place] = r
        out.append(full.view((longest, len(spans)) + tuple(r.shape[1:])))
    return out, lambda full: full.reshape((-1,) + tuple(full.shape[2:]))[place]


def _wkv(m, W, p, x, width, eps, spans):
    H, D, rank = m["heads"], m["dim"], m["decay_rank"]
    before = _each(spans, _before, x)
    mixed = {s: x + (before - x) * W(p + "mu." + s, width, kind="unit") for s in "rkvgw"}
    r, k, v = ((mixed[s] @ W(p + s, H * D, width).T).view(-1, H, D) for s in "rkv")
    gate = torch.nn.functional.silu(mixed["g"] @ W(p + "g", H * D, width).T)
    w = torch.tanh(mixed["w"] @ W(p + "w1", rank, width).T) @ W(p + "w2", H * D, rank).T + W(p + "w0", H * D, kind="decay")
    decay = torch.exp(-torch.exp(w)).view(-1, H, D)
    bonus = W(p + "u", H, D, kind="bonus")
    (r, k, v, decay), back = _padded(spans, r, k, v, decay)
    S = torch.zeros(len(spans), H, D, D, dtype=torch.float64, device="cuda")
    out = torch.empty_like(r)
    own = (r * bonus * k).sum(-1, keepdim=True) * v
    for t in range(r.shape[0]):
        out[t] = torch.matmul(r[t].unsqueeze(-2), S).squeeze(-2) + own[t]
        S = decay[t].unsqueeze(-1) * S + k[t].unsqueeze(-1) * v[t].unsqueeze(-2)
    o = _unit(back(out), eps).reshape(-1, H * D) * W(p + "norm", H * D, kind="norm") * gate
    return o @ W(p + "o", width, H * D).T


def _latent(m, W, p, x, width, eps, spans):
    H, D, R, E, rank, q_rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"], m["q_rank"]
    f, stretch = _frequencies(m["rot"]["dims"], m["rot"]["base"], m["rot"].get("scaling"))
    c = _unit(x @ W(p + "dq", q_rank, width).T, eps) * W(p + "dq.norm", q_rank, kind="norm")
    q = (c @ W(p + "uq", H * (D + R), q_rank).T).view(-1, H, D + R)
    kv = x @ W(p + "dkv", rank + R, width).T
    c = _unit(kv[:, :rank], eps) * W(p + "dkv.norm", rank, kind="norm")
    k, v = (c @ W(p + "uk", H * D, rank).T).view(-1, H, D), (c @ W(p + "uv", H * E, rank).T).view(-1, H, E)
    sink = W(p + "sink", H, kind="sink")

    def one(q, k, k_turned, v):
        q = torch.cat([q[..., :D], _turn(q[..., D:], f, stretch, "neighbours")], -1)
        k = torch.cat([k, _turn(k_turned[:, None], f, stretch, "neighbours").expand(-1, H, -1)], -1)
        return _attend(q, k, v, m["scale"], sink=sink)
    return _each(spans, one, q, k, kv[:, rank:], v).reshape(-1, H * E) @ W(p + "o", width, H * E).T


def _exact_nipulorn(cfg, W, ids, spans, rows):
    w, eps = cfg["width"], cfg["norm"]["eps"]
    table = W("embed", cfg["vocab"], w)
    x = table[ids]
    norm = lambda x, name: _unit(x, eps) * (1.0 + W(name, w, kind="offset"))
    with_past = lambda x, name: (lambda taps: _each(spans, lambda r: r + _convolve(r, taps), x))(W(name, w, cfg["canon"]["taps"], kind="taps"))
    for n, layer in enumerate(cfg["layers"]):
        p = f"l{n}."
        y = with_past(norm(x, p + "norm1"), p + "canon1")
        x = x + norm((_wkv if layer["type"] == "wkv" else _latent)(layer["mixer"], W, p + "mix.", y, w, eps, spans), p + "norm1b")
        y = with_past(norm(x, p + "norm2"), p + "canon2")
        ff = layer["mlp"]["ff"]
        z = y @ W(p + "mlp.up", ff, w).T
        act = W(p + "mlp.act", 2, kind="shape")
        up, down = torch.nn.functional.softplus(act[0]), 0.5 + torch.nn.functional.softplus(act[1])
        low = z.clamp(max=0.0)
        z = torch.where(z > 0, up * z * z, down * (torch.expm1(low) - low)) + 0.5 * z
        x = x + norm(z @ W(p + "mlp.down", w, ff).T, p + "norm2b")
    return norm(x[rows], "final.norm") @ table.T


def _rglru(m, W, p, x, width, spans):
    C, blocks = m["width"], m["blocks"]
    size = C // blocks
    y = torch.nn.functional.gelu(x @ W(p + "y", C, width).T + W(p + "y.b", C), approximate="tanh")
    u = x @ W(p + "x", C, width).T + W(p + "x.b", C)
    taps = W(p + "conv", C, m["conv"], kind="taps")
    u = _each(spans, lambda r: _convolve(r, taps), u) + W(p + "conv.b", C)
    part = u.view(-1, blocks, size).transpose(0, 1).contiguous()
    r, i = (torch.sigmoid(torch.matmul(part, W(p + n, blocks, size, size).transpose(1, 2).contiguous()) + W(p + n + ".b", blocks, size)[:, None])
            .transpose(0, 1).reshape(-1, C) for n in ("ra", "ri"))
    a = torch.exp(-8.0 * r * torch.nn.functional.softplus(W(p + "lam", C, kind="bonus")))
    (a, new), back = _padded(spans, a, torch.sqrt(1.0 - a * a) * i * u)
    S, out = torch.zeros_like(new[0]), torch.empty_like(new)
    for t in range(new.shape[0]):
        S = a[t] * S + new[t]
        out[t] = S
    return (back(out) * y) @ W(p + "o", width, C).T


def _batodra_attention(m, W, p, x, width, eps, spans):
    H, G, D, E = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    f, stretch = _frequencies(m["rot"]["dims"], m["rot"]["base"], m["rot"].get("scaling"))
    maps = 2 if "diff" in m else 1
    q, k = ((x @ W(p + c, n * maps * D, width).T).view(-1, n * maps, D) for c, n in (("q", H), ("k", G)))
    v = (x @ W(p + "v", G * E, width).T).view(-1, G, E)
    if maps == 1:
        mask = m.get("mask") or {}
        one = lambda q, k, v: _attend(_unit(_turn(q, f, stretch), eps), _unit(_turn(k, f, stretch), eps), v, m["scale"],
                                      mask.get("size", 0), mask.get("keep_first", 0))
        o = _each(spans, one, q, k, v)
    else:
        q, k = (_unit(t, eps) * W(p + c, D, kind="norm") for t, c in ((q, "q.norm"), (k, "k.norm")))

        def one(q, k, v):
            q, k = _turn(q, f, stretch).view(-1, H, 2, D), _turn(k, f, stretch).view(-1, G, 2, D)
            weight = torch.exp(l[0] @ l[1]) - torch.exp(l[2] @ l[3]) + m["diff"]
            return _attend(q[:, :, 0], k[:, :, 0], v, m["scale"]) - weight * _attend(q[:, :, 1], k[:, :, 1], v, m["scale"])
        l = [W(p + n, D) for n in ("lq1", "lk1", "lq2", "lk2")]
        o = _unit(_each(spans, one, q, k, v), eps) * (1.0 - m["diff"])
    return o.reshape(-1, H * E) @ W(p + "o", width, H * E).T


def _exact_batodra(cfg, W, ids, spans, rows):
    w, eps, alpha = cfg["width"], cfg["norm"]["eps"], cfg["postln_alpha"]
    x = W("embed", cfg["vocab"], w)[ids]
    norm = lambda x, name: _unit(x, eps) * W(name, w, kind="norm")
    for n, layer in enumerate(cfg["layers"]):
        p, m = f"l{n}.", layer["mixer"]
        a = _rglru(m, W, p + "mix.", x, w, spans) if layer["type"] == "rglru" else _batodra_attention(m, W, p + "mix.", x, w, eps, spans)
        x = norm(alpha * x + a, p + "norm1")
        ff = layer["mlp"]["ff"]
        x = norm(alpha * x + torch.relu(x @ W(p + "mlp.up", ff, w).T).square() @ W(p + "mlp.down", w, ff).T, p + "norm2")
    return norm(x[rows], "final.norm") @ W("head", cfg["vocab"], w).T


def _zogurax_attention(kind, m, W, p, x, width, eps, spans):
    H, G, D, E = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    sizes = {"q": H * D, "k": G * D, "v": G * E}
    t = {c: x @ W(p + c, n, width).T for c, n in sizes.items()}
    if kind == "attention_2":
        t = {c: r + W(p + c + ".b", sizes[c]) for c, r in t.items()}
    else:
        for c, n in sizes.items():
            taps = W(p + c + ".conv", n, m["conv"], kind="taps")
            t[c] = _each(spans, lambda r: _convolve(r, taps), t[c])
        for c in "qk":
            t[c] = _unit(t[c], eps) * W(p + c + ".norm", sizes[c], kind="norm")
    sink = torch.zeros(H, dtype=torch.float64, device="cuda") if kind == "attention_2" else None

    def one(q, k, v):
        block = torch.div(torch.arange(q.shape[0], device="cuda") + 1, m["q_temp"]["every"], rounding_mode="floor")
        q = q * (1.0 + m["q_temp"]["coef"] * torch.log(block + 1.0))[:, None]
        return _attend(q.view(-1, H, D), k.view(-1, G, D), v.view(-1, G, E), m["scale"], cap=m["softcap"], sink=sink)
    a = _each(spans, one, t["q"], t["k"], t["v"])
    if kind == "attention":
        a = a * torch.sigmoid(x @ W(p + "g", H, width).T)[:, :, None]
    out = a.reshape(-1, H * E) @ W(p + "o", width, H * E).T
    return out + W(p + "o.b", width) if kind == "attention_2" else out


def _exact_zogurax(cfg, W, ids, spans, rows):
    w, eps, loop = cfg["width"], cfg["norm"]["eps"], cfg["loop"]
    position = torch.cat([torch.arange(b - a, device="cuda") for a, b in spans]).double()
    angle = position[:, None] * torch.tensor([10000.0 ** (-2.0 * i / w) for i in range(w // 2)], dtype=torch.float64, device="cuda")
    x = first = W("embed", cfg["vocab"], w)[ids] + torch.stack([angle.sin(), angle.cos()], -1).reshape(-1, w)

    def norm(x, name):
        x = x - x.mean(-1, keepdim=True)
        return _unit(x, eps) * W(name, w, kind="norm")
    inside = range(loop["start"], loop["stop"])
    runs = [(i, None) for i in range(loop["start"])] + [(i, t if i == loop["start"] else None) for t in range(loop["times"]) for i in inside]
    for n, opens in runs + [(i, None) for i in range(loop["stop"], len(cfg["layers"]))]:
        layer, p = cfg["layers"][n], f"l{n}."
        if opens is not None:
            x = torch.cat([x, first], 1) @ W("loop.in", w, 2 * w).T + W("loop.step", loop["times"], w)[opens]
        y = norm(x, p + "norm1")
        x = x + _zogurax_attention(layer["type"], layer["mixer"], W, p + "mix.", y, w, eps, spans)
        f = layer["mlp"]
        ff, top, n_experts = f["expert"]["ff"], f["router"]["top"], f["router"]["experts"]
        chosen = W.choices(p + "mlp.table", cfg["vocab"], top, n_experts)[ids]
        expert = lambda y, name, ff: torch.relu(y @ W(name + "up", ff, w).T).square() @ W(name + "down", w, ff).T
        for e in range(n_experts):
            mine = (chosen == e).any(-1).nonzero().flatten()
            if len(mine):
                x = x.index_add(0, mine, expert(y[mine], p + f"mlp.e{e}.", ff) / top)
        x = x + expert(y, p + "mlp.shared.", f["shared"]["ff"]) * torch.sigmoid(y @ W(p + "mlp.shared.sg", 1, w).T)
    return norm(x[rows], "final.norm") @ W("head", cfg["vocab"], w).T


def exact(case, seed):
    if case["kind"] == "sample":
        return None                                     # token ids, no computed numbers
    tokens = _tokens(case, seed)
    ends = np.cumsum([len(t) for t in tokens]).tolist()
    spans = [(e - len(t), e) for t, e in zip(tokens, ends)]
    firsts = [a + n - (0 if case["kind"] == "decode" else 1) for (a, _), n in zip(spans, _lengths(case))]
    steps = case["steps"] + (0 if case["kind"] == "decode" else 1)
    rows = torch.tensor([f + s for s in range(steps) for f in firsts], device="cuda")
    ids = torch.tensor([i for t in tokens for i in t], device="cuda")
    forward = {"nipulorn": _exact_nipulorn, "batodra": _exact_batodra, "zogurax": _exact_zogurax}.get(case["model"], _exact_dense)
    with torch.no_grad():
        logits = forward(_config(case), _Weights(_config(case)["torch_dtype"]), ids, spans, rows)
    return list(logits.view(steps, len(tokens), -1))
