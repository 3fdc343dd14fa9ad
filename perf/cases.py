"""The calls whose speed counts, with their inputs, their results in 64 bits and what they cannot do without.

A case is one model at given sizes and one way of using its engine:

  prompts   new sequences, their prompts whole in one step or in chunks of every sequence, the logits of
            every prompt's last token, the sequences closed: what a request's first token costs
  decode    sequences that stand in the cache already, one more token each, greedy selection started on the
            logits, the sequences rewound: a turn of the generation loop (models without a fixed-size state)
  request   new sequences, their prompts in one step, then a given continuation token by token with the
            logits of every step kept, the sequences closed: a whole request, scored instead of sampled

Models have the layer sizes of GPT-2's published models or of the family workloads of the repository's
benchmark; weights are drawn by the families' own initialisation on the GPU, tokens uniformly.
"""

import math

import numpy as np
import torch

import burn_transformers_amd as bt

GPT2_SIZES = {"xl": (48, 1600, 25), "medium": (24, 1024, 16), "small": (12, 768, 12)}      # layers, width, heads
VOCAB = 32000                                # of the families beside GPT-2
LAYERS = 12
FAMILIES = ("salopel", "kodatar", "rotutar", "gavasun", "loselix", "rirovik")
REWINDABLE = ("gpt2", "loselix")             # every key kept and no state of fixed size: decode cases can rewind


# --- the cases ---------------------------------------------------------------------------------

def listed():
    """Latency of the smallest call to the widest batch and the longest prompt, each family once."""
    def gpt2(name, size, dtype, use, batch, low, high, chunk=0, steps=0):
        return {"name": name, "family": "gpt2", "size": size, "dtype": dtype, "use": use, "batch": batch, "low": low,
                "high": high, "chunk": chunk, "steps": steps}

    def family(name, width, use, batch, low, high, chunk=0, steps=0):
        return {"name": f"{name}_{use}", "family": name, "size": str(width), "dtype": "bf16", "use": use, "batch": batch,
                "low": low, "high": high, "chunk": chunk, "steps": steps}

    return [
        # one user at the start of a conversation with a small model: launches and latency alone
        gpt2("gpt2_small_decode_b1", "small", "bf16", "decode", 1, 37, 37),
        # the repository's headline: eight conversations of a few hundred tokens each, one decode step
        gpt2("gpt2_xl_decode_b8", "xl", "bf16", "decode", 8, 512, 1000),
        # a full server: sixty-four conversations of unequal length
        gpt2("gpt2_xl_decode_b64", "xl", "bf16", "decode", 64, 130, 900),
        # the benchmark's prefill: two prompts of the model's whole context
        gpt2("gpt2_xl_prompts", "xl", "bf16", "prompts", 2, 1024, 1024),
        # admission of unequal prompts in chunks, as a server does it to bound a step's time
        gpt2("gpt2_medium_chunks", "medium", "bf16", "prompts", 8, 64, 768, chunk=256),
        # full precision: prompts of every length and a few tokens behind each
        gpt2("gpt2_small_fp32_request", "small", "fp32", "request", 4, 3, 1000, steps=4),
        # scans over long prompts (a state per channel, a state per head) beside latent attention
        family("salopel", 1024, "prompts", 2, 1024, 1024),
        # experts, rotary attention in chunks: many short prompts at once
        family("kodatar", 1024, "prompts", 16, 5, 200),
        # matrix states with a decay per key channel, window attention, experts with a gate
        family("rotutar", 1024, "prompts", 2, 1024, 1024),
        # a delta rule with one decay a head: unequal prompts and the first tokens behind them
        family("gavasun", 1024, "request", 4, 90, 1000, steps=8),
        # differential and sigmoid attention: eight conversations, one decode step
        family("loselix", 1024, "decode", 8, 300, 1000),
        # latent attention at the larger width: short prompts, then mostly decode steps
        family("rirovik", 2048, "request", 8, 20, 150, steps=16),
    ]


def _log_uniform(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the same ranges: half GPT-2, half the other families."""
    family = "gpt2" if rng.random() < 0.5 else rng.choice(FAMILIES)
    dtype = "fp32" if rng.random() < 0.2 else "bf16"
    uses = ["prompts", "request"] + (["decode", "decode"] if family in REWINDABLE else [])
    use = rng.choice(uses)
    if family == "gpt2":
        size = rng.choice(["small", "medium", "xl"] if dtype == "bf16" else ["small", "medium"])
    else:
        size = rng.choice(["1024", "1024", "2048"] if dtype == "bf16" else ["1024"])
    small = size in ("small", "medium", "1024")
    steps = chunk = 0
    if use == "decode":
        batch = _log_uniform(rng, 1, 64 if family == "gpt2" and dtype == "bf16" else 16)
        low = _log_uniform(rng, 8, 900)
        high = rng.randint(low, 1000)
    else:
        budget = _log_uniform(rng, 16, (2048 if small else 1024) if dtype == "bf16" else 1024)      # prompt tokens in all
        batch = _log_uniform(rng, 1, 16)
        mean = max(2, min(1000, budget // batch))
        low = rng.randint(1, mean)
        high = min(1000, 2 * mean - low)
        if use == "request":
            steps = rng.randint(1, 8)
        elif family == "gpt2" and high > 300 and rng.random() < 0.3:
            chunk = rng.choice([128, 200, 256])
    return {"family": family, "size": size, "dtype": dtype, "use": use, "batch": batch, "low": low, "high": high,
            "chunk": chunk, "steps": steps}


def _lengths(case):
    """Tokens every sequence brings: spread over low..high, the same for every seed."""
    low, high = case["low"], case["high"]
    return [high - (i * 61803 % 100000) * (high - low) // 99999 for i in range(case["batch"])]


# --- models ------------------------------------------------------------------------------------

def _config(case):
    """config.json of the case's model: the layer sizes of the repository's benchmark."""
    family = case["family"]
    if family == "gpt2":
        layers, width, heads = GPT2_SIZES[case["size"]]
        return {"architectures": ["GPT2LMHeadModel"], "model_type": "gpt2", "n_layer": layers, "n_embd": width, "n_head": heads,
                "n_inner": 4 * width, "vocab_size": 50257, "n_positions": 1024, "activation_function": "gelu_new",
                "layer_norm_epsilon": 1e-5}
    width = int(case["size"])
    heads, eps = max(4, width // 128), {"eps": 1e-5}
    third = LAYERS // 3
    if family == "salopel":
        attention = {"type": "latent_attention", "mlp": {"kind": "dense", "ff": 4 * width},
                     "mixer": {"heads": min(16, width // 64), "dim": 128, "vdim": 64, "q_rank": 3 * width // 8 // 8 * 8,
                               "kv_rank": 128, "scale": 128 ** -0.5}}
        per_head = {"type": "mamba2", "mlp": None, "mixer": {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 1,
                                                             "norm_groups": 1, "conv": 4}}
        per_channel = {"type": "mamba1", "mlp": None, "mixer": {"inner": 2 * width, "state": 16, "dt_rank": width // 16, "conv": 4}}
        group = [attention, per_head, per_channel, attention]
        return {"architecture": "Salopel", "vocab": VOCAB, "width": width, "residual_mult": 0.5, "norm": eps,
                "layers": [dict(group[i % 4]) for i in range(LAYERS)]}
    if family == "kodatar":
        layer = {"type": "attention",
                 "mixer": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 64, "scale": 128 ** -0.5,
                           "rot": {"dims": 128, "base": 500000.0,
                                   "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}}, "mask": {"size": 512}},
                 "mlp": {"kind": "moe", "expert": {"ff": width}, "shared": {"ff": 2 * width},
                         "router": {"experts": 8, "top": 2, "identity": 1, "groups": {"count": 3, "keep": 2}}}}
        return {"architecture": "Kodatar", "vocab": VOCAB, "width": width, "embedding": {"scale": 1.0}, "logit_scale": 1.0,
                "norm": eps, "loop": {"start": 0, "stop": third, "times": 2}, "layers": [dict(layer) for _ in range(LAYERS - third)]}
    if family == "rotutar":
        forget = {"heads": heads, "dim": 128, "vdim": 128}
        pair = {"left": {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                         "rot": {"dims": 128, "base": 10000.0}, "mask": {"size": 512}},
                "right": {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4, "rank": 64},
                "left_scale": 1.0, "right_scale": 1.0}
        experts = {"kind": "moe", "expert": {"ff": width, "limit": 7.0},
                   "router": {"experts": 8, "top": 2, "groups": {"count": 4, "keep": 2}}}
        group = [{"type": "hgrn2", "mixer": forget, "mlp": {"kind": "dense", "ff": 4 * width}},
                 {"type": "hgrn2", "mixer": forget, "mlp": experts}, {"type": "parallel", "mixer": pair, "mlp": experts},
                 {"type": "hgrn2", "mixer": forget, "mlp": experts}]
        return {"architecture": "Rotutar", "vocab": VOCAB, "width": width, "logit_softcap": 30.0, "norm": {"eps": 1e-5, "groups": 2},
                "layers": [dict(group[i % 4]) for i in range(LAYERS)]}
    if family == "loselix":
        shared = {"heads": heads, "kv_heads": heads // 4, "vdim": 128}
        pair = ("attention", {**shared, "dim": 64, "scale": 64 ** -0.5, "rot": {"dims": 64, "base": 500000.0}, "softcap": 50.0, "diff": 0.3})
        gated = ("attention_2", {**shared, "dim": 128, "scale": 128 ** -0.5, "rot": {"dims": 64, "base": 500000.0}})
        sigmoid = ("attention_3", {**shared, "dim": 128, "scale": 128 ** -0.5, "q_temp": {"coef": 0.1, "every": 512}})
        group = [pair, gated, gated, sigmoid]
        return {"architecture": "Loselix", "vocab": VOCAB, "width": width, "norm": eps, "loop": {"start": 0, "stop": third, "times": 2},
                "layers": [{"type": group[i % 4][0], "mixer": dict(group[i % 4][1]), "mlp": {"kind": "dense", "ff": 4 * width}}
                           for i in range(LAYERS - third)]}
    experts = {"kind": "moe", "expert": {"ff": width}, "router": {"experts": 8, "top": 2}, "shared": {"ff": width}}
    latent = {"heads": min(heads, 16), "dim": 128, "rot_dim": 32, "vdim": 128, "q_rank": 3 * width // 8, "kv_rank": 96,
              "scale": 160 ** -0.5}
    if family == "gavasun":
        slowed = {"factor": 4.0, "original": 2048, "fast": 16.0, "slow": 2.0}
        attention = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "conv": 4,
                     "rot": {"dims": 64, "base": 500000.0, "scaling": slowed}, "mask": {"size": 512}}
        delta = {"heads": heads, "kv_heads": heads // 2, "dim": 128, "vdim": 128, "conv": 4}
        latent = dict(latent, rot={"dims": 32, "base": 10000.0, "scaling": slowed}, mask={"size": 512})
        group = [{"type": "attention", "mixer": attention, "mlp": {"kind": "dense", "ff": 4 * width}},
                 {"type": "delta", "mixer": delta, "mlp": experts}, {"type": "latent_attention", "mixer": latent, "mlp": experts},
                 {"type": "delta", "mixer": delta, "mlp": experts}]
        return {"architecture": "Gavasun", "vocab": VOCAB, "width": width, "embedding": {"scale": 1.0}, "norm": eps, "loop": None,
                "layers": [dict(group[i % 4]) for i in range(LAYERS)]}
    attention = {"heads": heads, "kv_heads": heads // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5,
                 "mask": {"size": 512, "keep_first": 64}}
    whole = dict(latent, rot={"dims": 32, "base": 500000.0})
    window = dict(whole, mask={"size": 512})
    group = [("attention", attention), ("latent_attention_2", whole), ("latent_attention", window), ("latent_attention", window)]
    return {"architecture": "Rirovik", "vocab": VOCAB, "width": width, "embedding": {"scale": 1.0}, "norm": eps,
            "layers": [{"type": group[i % 4][0], "mixer": dict(group[i % 4][1], **({"kv_from": i - 1} if i % 4 == 3 else {})),
                        "mlp": experts} for i in range(LAYERS)]}


def _vocab(config):
    return config.get("vocab") or config["vocab_size"]


def _decide(tensors, generator):
    """Gives routers something to go by: every token's embedding carries two experts' directions, which the routers
    read, so that a token's experts are chosen by a margin as trained routers choose them.  Random routers leave
    many tokens' choices to rounding, and whoever rounds otherwise has another result."""
    routers = [name for name in tensors if name.endswith(".router")]
    if not routers:
        return
    count, width = tensors[routers[0]].shape
    directions = torch.linalg.qr(torch.randn((width, count), generator=generator))[0].T
    token = torch.arange(tensors["embed"].shape[0])
    first = token % count
    second = (first + 1 + token // count % (count - 1)) % count
    tensors["embed"] += 40.0 * directions[first] + 32.0 * directions[second]
    for name in routers:
        tensors[name] = 0.15 * directions + 0.1 * width ** -0.5 * torch.randn((count, width), generator=generator)
    if "loop.in" in tensors:                                 # a pass starts near the mean of the stream and the embedding
        tensors["loop.in"] += 0.5 * torch.eye(width).repeat(1, 2)


def _tensors(case, seed):
    """A checkpoint's tensors as the family initialises them, drawn on the GPU; stored in the case's type."""
    config = _config(case)
    family = bt.resolve_family(config)
    generator = torch.Generator(device="cuda:0").manual_seed(1000003 * seed + 17)
    with torch.device("cuda:0"):
        tensors = family.init(family.config_class.from_dict(config), generator)
        _decide(tensors, generator)
    return {name: t.to(torch.bfloat16) for name, t in tensors.items()} if case["dtype"] == "bf16" else tensors


def _tokens(case, seed):
    """(prompts, continuations): token ids of every sequence; the continuation is what follows a prompt."""
    rng = np.random.default_rng([seed, 5])
    vocab, after = _vocab(_config(case)), {"prompts": 0, "decode": 1, "request": case["steps"]}[case["use"]]
    rows = [rng.integers(0, vocab, n + after).tolist() for n in _lengths(case)]
    return [row[:len(row) - after] for row in rows], [row[len(row) - after:] for row in rows]


def prepare(case, seed):
    """The model, an engine with room for the sequences, and the tokens; for a decode step the sequences too."""
    prompts, after = _tokens(case, seed)
    model = bt.model_from_tensors(_config(case), _tensors(case, seed), dtype="bfloat16" if case["dtype"] == "bf16" else "float32")
    room = sum((len(p) + len(a) + 63) // 64 * 64 for p, a in zip(prompts, after))
    engine = bt.Engine(model, max_tokens=room, max_slots=max(8, len(prompts)))
    state = {"case": case, "engine": engine, "prompts": prompts, "after": after}
    if case["use"] == "decode":
        state["slots"] = [engine.open() for _ in prompts]
        for begin in range(0, len(prompts), 8):
            group = slice(begin, begin + 8)
            engine.step(list(zip(state["slots"][group], prompts[group])), want=[[] for _ in prompts[group]])
        state["sampler"] = bt.Sampler(bt.GenerationConfig(), len(prompts), engine.device)
    return state


def run(state):
    case, engine, prompts, after = state["case"], state["engine"], state["prompts"], state["after"]
    if case["use"] == "decode":
        slots, sampler = state["slots"], state["sampler"]
        logits = engine.step(list(zip(slots, after)))
        sampler.launch(logits, range(len(slots)))
        for slot, prompt in zip(slots, prompts):
            engine.truncate(slot, len(prompt))
        return {"logits": logits, "logp": sampler.logp[:len(slots)]}       # (of the chosen token: ties change nothing)
    slots = [engine.open() for _ in prompts]
    try:
        if case["use"] == "request":
            rows = [engine.step(list(zip(slots, prompts))).clone()]
            for step in range(case["steps"]):
                rows.append(engine.step([(slot, [tokens[step]]) for slot, tokens in zip(slots, after)]).clone())
            return rows
        if not case["chunk"]:
            return engine.step(list(zip(slots, prompts)))
        logits = torch.empty((len(prompts), engine.model.vocab_size), dtype=torch.float32, device=engine.device)
        for chunk in range(0, max(len(p) for p in prompts), case["chunk"]):
            rows = [i for i, p in enumerate(prompts) if len(p) > chunk]
            last = [i for i in rows if len(prompts[i]) <= chunk + case["chunk"]]
            pieces = [prompts[i][chunk:chunk + case["chunk"]] for i in rows]
            part = engine.step([(slots[i], piece) for i, piece in zip(rows, pieces)],
                               want=[[len(piece) - 1] if i in last else [] for i, piece in zip(rows, pieces)])
            for place, i in enumerate(last):
                logits[i] = part[place]
        return logits
    finally:
        for slot in slots:
            engine.close(slot)


# --- what a pass cannot do without -------------------------------------------------------------

def _runs(config):
    """Layers in the order they run."""
    count, loop = config.get("n_layer") or len(config["layers"]), config.get("loop")
    if not loop:
        return list(range(count))
    stretch = list(range(loop["start"], loop["stop"]))
    return list(range(loop["start"])) + stretch * loop["times"] + list(range(loop["stop"], count))


def _mixing(config, index, lengths, before):
    """(flops, bytes in elements of the cache) of layer ``index``'s mixing of tokens, for sequences that bring
    ``lengths`` tokens behind ``before`` in the cache."""
    if "n_layer" in config:
        heads, dim, kv, window, state = config["n_head"], 2 * config["n_embd"] // config["n_head"], 2 * config["n_embd"], 0, 0
    else:
        layer = config["layers"][index]
        m, kind, state = layer["mixer"], layer["type"], 0
        if kind == "mamba1":
            return 6.0 * sum(lengths) * m["inner"] * m["state"], 4.0 * len(lengths) * m["inner"] * m["state"]
        if kind == "mamba2":
            size = m["heads"] * m["vdim"] * m["state"]
            return 6.0 * sum(lengths) * size, 4.0 * len(lengths) * size
        if kind in ("hgrn2", "delta"):
            size = m["heads"] * m["dim"] * m["vdim"]
            return (5.0 if kind == "hgrn2" else 7.0) * sum(lengths) * size, 4.0 * len(lengths) * size
        if kind == "parallel":
            state, m = m["right"]["heads"] * m["right"]["dim"] * m["right"]["vdim"], m["left"]
        heads, dim = m["heads"], m["dim"] * (2 if "diff" in m else 1) + m.get("rot_dim", 0) + m.get("vdim", m["dim"])
        kv = m["kv_rank"] + m.get("rot_dim", 0) if "kv_rank" in m else m["kv_heads"] * dim
        window = (m.get("mask") or {}).get("size", 0)
    pairs = read = 0
    for n, past in zip(lengths, before):
        positions = np.arange(past, past + n)
        seen = np.minimum(positions + 1, window) if window else positions + 1
        pairs += int(seen.sum())
        read += (min(past, window) if window else past) + n
    return 2.0 * pairs * heads * dim + 7.0 * sum(lengths) * state, read * kv + 4.0 * len(lengths) * state


def work(case):
    config = _config(case)
    family = bt.resolve_family(config)
    specs = family.contract(family.config_class.from_dict(config)).tensors
    element = 2 if case["dtype"] == "bf16" else 4
    lengths = _lengths(case)
    if case["use"] == "decode":
        steps = [([1] * len(lengths), lengths, len(lengths))]
    elif case["use"] == "request":
        steps = [(lengths, [0] * len(lengths), len(lengths))]
        steps += [([1] * len(lengths), [n + s for n in lengths], len(lengths)) for s in range(case["steps"])]
    else:
        size = case["chunk"] or max(lengths)
        steps = []
        for begin in range(0, max(lengths), size):
            live = [n for n in lengths if n > begin]
            steps.append(([min(size, n - begin) for n in live], [begin] * len(live), sum(n <= begin + size for n in live)))
    order, matrices, experts, other = _runs(config), {}, {}, 0.0
    for spec in specs:
        size = float(np.prod([64 if isinstance(extent, str) else extent for extent in spec.shape]))
        if spec.name in ("embed", "wpe.weight"):
            continue
        layer = spec.name.split(".")[1] if spec.name.startswith("h.") else spec.name.split(".")[0][1:]
        if spec.name in ("wte.weight", "head"):
            other += size
        elif layer.isdigit():
            held = experts if ".mlp.e" in spec.name else matrices
            held[int(layer)] = held.get(int(layer), 0.0) + size
    if not any(spec.name in ("wte.weight", "head") for spec in specs):          # the readout is tied to the table
        other = float(_vocab(config)) * config["width"]
    flops = nbytes = 0.0
    for counts, before, rows in steps:
        tokens = sum(counts)
        flops += 2.0 * rows * other
        nbytes += other * element + rows * 4.0 * _vocab(config)
        for index in set(order):                             # weights are read once a step, however often a layer runs
            nbytes += element * matrices.get(index, 0.0)
            if index in experts:
                router = config["layers"][index]["mlp"]["router"]
                nbytes += element * experts[index] * min(1.0, tokens * router["top"] / router["experts"])
        for index in order:
            share = 1.0
            if index in experts:
                router = config["layers"][index]["mlp"]["router"]
                share = router["top"] / router["experts"]
            mixing, cached = _mixing(config, index, counts, before)
            flops += 2.0 * tokens * (matrices.get(index, 0.0) + share * experts.get(index, 0.0)) + mixing
            nbytes += element * cached
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    """Relative error of the logits, about four times what is measured against 64 bits: rounding values to bfloat16
    between kernels adds up over the layers to 1.4e-3 (Kodatar), 3.5e-3 to 5.2e-3 (GPT-2, Gavasun, Loselix, Rirovik),
    5.5e-3 to 11e-3 (Salopel and Rotutar, with norms of the sublayers' outputs); sums in 32 bits to 0.3e-6 to 2.1e-6."""
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 0.03 if case["family"] in ("salopel", "rotutar") else 0.018}


# --- the same in 64 bits -----------------------------------------------------------------------

def _rms(x, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, weight, bias, eps):
    x = x - x.mean(-1, keepdim=True)
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * weight + bias


def _silu(x):
    return x * torch.sigmoid(x)


def _softplus(x):
    return torch.where(x > 30.0, x, torch.log1p(torch.exp(x.clamp(max=30.0))))


def _frequencies(rot):
    """(f [dims / 2], amplitude) of a rotation, long waves slowed in one of two ways."""
    dims, base, scaling = rot["dims"], rot["base"], rot.get("scaling")
    f = [base ** (-2.0 * i / dims) for i in range(dims // 2)]
    amplitude = 1.0
    if scaling and "high" in scaling:                        # blended by wavelength
        for i, plain in enumerate(f):
            turns = scaling["original"] * plain / (2.0 * math.pi)
            t = min(1.0, max(0.0, (turns - scaling["low"]) / (scaling["high"] - scaling["low"])))
            f[i] = (1.0 - t) * plain / scaling["factor"] + t * plain
    elif scaling:                                            # blended by a ramp over the pair's number
        pair_of = lambda turns: dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))
        lo, hi = max(math.floor(pair_of(scaling["fast"])), 0), min(math.ceil(pair_of(scaling["slow"])), dims - 1)
        for i, plain in enumerate(f):
            t = min(1.0, max(0.0, (i - lo) / max(hi - lo, 0.001)))
            f[i] = plain / scaling["factor"] * t + plain * (1.0 - t)
        amplitude = 0.1 * math.log(scaling["factor"]) + 1.0
    return f, amplitude


def _turn(x, positions, rot, neighbours):
    """x [N, heads, n]: pairs (2i, 2i + 1) or (i, i + dims / 2) turned by position times f_i."""
    if not rot:
        return x
    dims = rot["dims"]
    f, amplitude = _frequencies(rot)
    angle = positions.double()[:, None] * torch.tensor(f, dtype=torch.float64, device=x.device)[None]
    cos, sin = (torch.cos(angle) * amplitude)[:, None], (torch.sin(angle) * amplitude)[:, None]
    first = slice(0, dims, 2) if neighbours else slice(0, dims // 2)
    second = slice(1, dims, 2) if neighbours else slice(dims // 2, dims)
    u, v, out = x[..., first], x[..., second], x.clone()
    out[..., first], out[..., second] = u * cos - v * sin, v * cos + u * sin
    return out


class _Plain:
    """Whole sequences without a cache, the tokens of all of them packed into rows [N, ...]; ``w`` in 64 bits."""

    def __init__(self, config, w, sequences):
        self.config, self.w = config, w
        self.device = next(iter(w.values())).device
        self.lengths = [len(s) for s in sequences]
        self.offsets = np.concatenate([[0], np.cumsum(self.lengths)]).tolist()
        self.ids = torch.tensor([t for s in sequences for t in s], device=self.device)
        self.positions = torch.cat([torch.arange(n, device=self.device) for n in self.lengths])
        self.eps = config["norm"]["eps"] if "norm" in config else config["layer_norm_epsilon"]

    def lin(self, x, name):
        y = x @ self.w[name].T
        return y + self.w[name + ".b"] if name + ".b" in self.w else y

    def attend(self, q, k, v, scale, mask=None, weigh=None):
        """q [N, H, D], k [N, G, D], v [N, G, V] -> [N, H, V]; ``mask``: (window, chunk, kept first positions)."""
        window, chunk, keep = mask or (0, 0, 0)
        group, out = q.shape[1] // k.shape[1], []
        for a, b in zip(self.offsets, self.offsets[1:]):
            p = torch.arange(b - a, device=self.device)
            i, j = p[:, None], p[None]
            seen = j <= i
            if window:
                seen = seen & ((i - j < window) | (j < keep))
            if chunk:
                seen = seen & (i // chunk == j // chunk)
            spread = lambda x: x[a:b].transpose(0, 1).repeat_interleave(group, 0).contiguous()
            scores = q[a:b].transpose(0, 1).contiguous() @ spread(k).transpose(1, 2).contiguous() * scale
            weights = weigh(scores, seen) if weigh else torch.softmax(scores.masked_fill(~seen, -math.inf), -1)
            out.append((weights @ spread(v)).transpose(0, 1))
        return torch.cat(out)

    def conv(self, x, taps):
        """Per channel over the sequence's own tokens, the last tap on the current one."""
        count = taps.shape[1]
        y = x * taps[:, count - 1]
        for back in range(1, count):
            earlier = torch.zeros_like(x)
            earlier[back:] = x[:-back] if back < len(x) else 0
            y = y + torch.where((self.positions >= back)[:, None], earlier, torch.zeros_like(x)) * taps[:, count - 1 - back]
        return y

    def scan(self, state, step, *rows):
        """``step(state, *row of every sequence) -> (state, output)`` token by token; rows [N, ...] -> [N, ...]."""
        longest, count = max(self.lengths), len(self.lengths)
        place = torch.stack([torch.arange(longest, device=self.device).clamp(max=n - 1) + a
                             for a, n in zip(self.offsets, self.lengths)], 1)                    # [T, sequences]
        padded = [row[place] for row in rows]
        S, out = state.expand(count, *state.shape).clone(), []
        for t in range(longest):
            S, y = step(S, *(row[t] for row in padded))
            out.append(y)
        out = torch.stack(out)
        return torch.cat([out[:n, s] for s, n in enumerate(self.lengths)])

    # mixers
    def heads(self, x, count):
        return x.view(x.shape[0], count, -1)

    def gpt2_attention(self, h, p):
        q, k, v = (self.heads(x, self.config["n_head"]) for x in
                   (h @ self.w[p + "c_attn.weight"] + self.w[p + "c_attn.bias"]).chunk(3, -1))
        return self.attend(q, k, v, q.shape[-1] ** -0.5).flatten(1) @ self.w[p + "c_proj.weight"] + self.w[p + "c_proj.bias"]

    def latent(self, h, p, m, neighbours_rot, latents=None, layer=None, window=0):
        """Latent attention of three families: an optional turned key part, a gate, a borrowed latent."""
        w, H, D, R, rank = self.w, m["heads"], m["dim"], m.get("rot_dim", 0), m["kv_rank"]
        rot = dict(neighbours_rot, dims=R) if R else None
        q = self.heads((_rms(h @ w[p + "dq"].T, self.eps) * w[p + "dq.norm"]) @ w[p + "uq"].T, H)
        if m.get("kv_from") is not None:
            c, r = latents[m["kv_from"]]
        else:
            down = h @ w[p + "dkv"].T
            c = _rms(down[:, :rank], self.eps) * w[p + "dkv.norm"]
            r = _turn(down[:, None, rank:], self.positions, rot, True)
            if latents is not None:
                latents[layer] = c, r
        k, v = self.heads(c @ w[p + "uk"].T, H), self.heads(c @ w[p + "uv"].T, H)
        if R:
            q = torch.cat([q[..., :D], _turn(q[..., D:], self.positions, rot, True)], -1)
            k = torch.cat([k, r.expand(-1, H, -1)], -1)
        return self.attend(q, k, v, m["scale"], (window, 0, 0))

    def mamba1(self, h, p, m):
        w, inner, rank, state = self.w, m["inner"], m["dt_rank"], m["state"]
        x, z = (h @ w[p + "in"].T).split(inner, -1)
        x = _silu(self.conv(x, w[p + "conv"]) + w[p + "conv.b"])
        low, B, C = (x @ w[p + "x"].T).split([rank, state, state], -1)
        dt = _softplus(low @ w[p + "dt"].T + w[p + "dt.b"])
        A = -torch.exp(w[p + "A_log"])

        def step(S, dt, x, B, C):
            S = torch.exp(dt[..., None] * A) * S + (dt * x)[..., None] * B[:, None]
            return S, (S * C[:, None]).sum(-1)
        y = self.scan(h.new_zeros(inner, state), step, dt, x, B, C) + w[p + "D"] * x
        return (y * _silu(z)) @ w[p + "o"].T

    def mamba2(self, h, p, m):
        w, H, V, state = self.w, m["heads"], m["vdim"], m["state"]
        inner = H * V
        z, xbc, dt = (h @ w[p + "in"].T).split([inner, inner + 2 * state, H], -1)
        xbc = _silu(self.conv(xbc, w[p + "conv"]) + w[p + "conv.b"])
        x, B, C = xbc.split([inner, state, state], -1)
        x, dt = self.heads(x, H), _softplus(dt + w[p + "dt_bias"])
        decay = torch.exp(-torch.exp(w[p + "A_log"]) * dt)

        def step(S, decay, write, B, C):
            S = decay[..., None, None] * S + write[..., None] * B[:, None, None]
            return S, (S * C[:, None, None]).sum(-1)
        y = self.scan(h.new_zeros(H, V, state), step, decay, dt[..., None] * x, B, C) + w[p + "D"][:, None] * x
        return (_rms(y.flatten(1) * _silu(z), self.eps) * w[p + "norm"]) @ w[p + "o"].T

    def hgrn2(self, h, p, m):
        w, H = self.w, m["heads"]
        q, v = self.heads(_silu(h @ w[p + "q"].T), H), self.heads(h @ w[p + "v"].T, H)
        f = self.heads(w[p + "lower"] + (1.0 - w[p + "lower"]) * torch.sigmoid(h @ w[p + "f"].T + w[p + "f.b"]), H)

        def step(S, f, q, v):
            S = f[..., None] * S + (1.0 - f)[..., None] * v[:, :, None]
            return S, (S * q[..., None]).sum(-2)
        out = self.scan(h.new_zeros(H, m["dim"], m["vdim"]), step, f, q, v)
        return (_rms(out, self.eps) * w[p + "norm"]).flatten(1) @ w[p + "o"].T

    def delta(self, h, p, m, decay, gate):
        w, H, G = self.w, m["heads"], m["kv_heads"]
        q, k = (self.heads(_silu(self.conv(h @ w[p + n].T, w[p + n + ".conv"])), G) for n in "qk")
        v = self.heads(_silu(self.conv(h @ w[p + "v"].T, w[p + "v.conv"])), H)
        unit = lambda x: (x * torch.rsqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
        q, k, beta = unit(q) * m["dim"] ** -0.5, unit(k), torch.sigmoid(h @ w[p + "b"].T)

        def step(S, decay, q, k, v, beta):
            S = decay[..., None] * S
            u = beta[..., None] * (v - (S * k[..., None]).sum(-2))
            S = S + k[..., None] * u[:, :, None]
            return S, (S * q[..., None]).sum(-2)
        out = self.scan(h.new_zeros(H, m["dim"], m["vdim"]), step, decay, q, k, v, beta)
        return (_rms(out, self.eps) * w[p + "norm"] * gate).flatten(1) @ w[p + "o"].T

    def mixer(self, h, layer, index, latents):
        w, m, family, p, eps = self.w, layer["mixer"], self.config["architecture"], f"l{index}.mix.", self.eps
        pos, kind, size = self.positions, layer["type"], (layer["mixer"].get("mask") or {}).get("size", 0)
        H, G = m.get("heads"), m.get("kv_heads")
        if kind == "mamba1":
            return self.mamba1(h, p, m)
        if kind == "mamba2":
            return self.mamba2(h, p, m)
        if kind == "hgrn2":
            return self.hgrn2(h, p, m)
        if kind == "delta":
            decay = torch.exp(-torch.exp(w[p + "A_log"]) * _softplus(h @ w[p + "a"].T + w[p + "dt_bias"]))
            return self.delta(h, p, m, decay[..., None], self.heads(_silu(h @ w[p + "g"].T), H))
        if kind == "parallel":
            left, right, a, b = m["left"], m["right"], p + "left.", p + "right."
            H, G = left["heads"], left["kv_heads"]
            q = _turn(self.heads(_rms(h @ w[a + "q"].T, eps) * w[a + "q.norm"], H), pos, left["rot"], True)
            k = _turn(self.heads(_rms(h @ w[a + "k"].T, eps) * w[a + "k.norm"], G), pos, left["rot"], True)
            sink = w[a + "sink"][:, None, None]

            def weigh(scores, seen):
                scores = torch.cat([scores.masked_fill(~seen, -math.inf), sink.expand(-1, scores.shape[1], 1)], -1)
                return torch.softmax(scores, -1)[..., :-1].contiguous()
            y = self.attend(q, k, self.heads(h @ w[a + "v"].T, G), left["scale"], (left["mask"]["size"], 0, 0), weigh)
            low = (h @ w[b + "a1"].T) @ w[b + "a2"].T + w[b + "dt_bias"]
            decay = torch.exp(-torch.exp(w[b + "A_log"])[:, None] * self.heads(_softplus(low), right["heads"]))
            gate = self.heads(torch.sigmoid((h @ w[b + "g1"].T) @ w[b + "g2"].T), right["heads"])
            return m["left_scale"] * (y.flatten(1) @ w[a + "o"].T) + m["right_scale"] * self.delta(h, b, right, decay, gate)
        if "kv_rank" in m:
            y = self.latent(h, p, m, m.get("rot"), latents, index, size)
            if p + "g" in w:
                gate = torch.sigmoid(h @ w[p + "g"].T)
                y = y * (gate[..., None] if gate.shape[1] == H else self.heads(gate, H))
            return y.flatten(1) @ w[p + "o"].T
        if family == "Kodatar":
            q = _turn(_rms(self.heads(h @ w[p + "q"].T, H), eps) * w[p + "q.norm"], pos, m["rot"], False)
            k = _turn(_rms(self.heads(h @ w[p + "k"].T, G), eps) * w[p + "k.norm"], pos, m["rot"], False)
            y = self.attend(q, k, self.heads(h @ w[p + "v"].T, G), m["scale"], (0, size, 0))
        elif family == "Gavasun":
            q, k, v = (self.conv(self.lin(h, p + n), w[p + n + ".conv"]) for n in "qkv")
            q = _turn(self.heads(_rms(q, eps) * w[p + "q.norm"], H), pos, m["rot"], False)
            k = _turn(self.heads(_rms(k, eps) * w[p + "k.norm"], G), pos, m["rot"], False)
            y = self.attend(q, k, self.heads(v, G), m["scale"], (0, size, 0))
        elif family == "Rirovik":
            q, k = _rms(self.heads(self.lin(h, p + "q"), H), eps), _rms(self.heads(self.lin(h, p + "k"), G), eps)
            y = self.attend(q, k, self.heads(self.lin(h, p + "v"), G), m["scale"], (size, 0, m["mask"]["keep_first"]))
            return (y.flatten(1) * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T
        elif kind == "attention":                            # Loselix: the difference of two maps
            q = self.heads(_turn(self.heads(h @ w[p + "q"].T, 2 * H), pos, m["rot"], False).flatten(1), H)
            k = self.heads(_turn(self.heads(h @ w[p + "k"].T, 2 * G), pos, m["rot"], False).flatten(1), G)
            v, D, cap = self.heads(h @ w[p + "v"].T, G), m["dim"], m["softcap"]

            def weigh(scores, seen):
                return torch.softmax((cap * torch.tanh(scores / cap)).masked_fill(~seen, -math.inf), -1)
            maps = [self.attend(q[..., i * D:(i + 1) * D], k[..., i * D:(i + 1) * D], v, m["scale"], None, weigh) for i in (0, 1)]
            lam = torch.exp((w[p + "lq1"] * w[p + "lk1"]).sum()) - torch.exp((w[p + "lq2"] * w[p + "lk2"]).sum()) + m["diff"]
            y = _rms(maps[0] - lam * maps[1], eps) * (1.0 - m["diff"])
        elif kind == "attention_2":                          # a gate a head
            q = _turn(self.heads(h @ w[p + "q"].T, H), pos, m["rot"], False)
            k = _turn(self.heads(h @ w[p + "k"].T, G), pos, m["rot"], False)
            y = self.attend(q, k, self.heads(h @ w[p + "v"].T, G), m["scale"]) * torch.sigmoid(h @ w[p + "g"].T)[..., None]
        else:                                                # sigmoid weights on keys that are their own values
            rows = h @ w[p + "k"].T
            q = self.heads(_rms(h @ w[p + "q"].T, eps) * w[p + "q.norm"], H)
            k = self.heads(_rms(rows, eps) * w[p + "k.norm"], G)
            grow = 1.0 + m["q_temp"]["coef"] * torch.log(((pos + 1) // m["q_temp"]["every"]).double() + 1.0)
            bias = w[p + "pb"][:, None, None]
            y = self.attend(q * grow[:, None, None], k, self.heads(rows, G), m["scale"], None,
                            lambda scores, seen: torch.sigmoid(scores + bias) * seen)
            return (y.flatten(1) * torch.sigmoid(h @ w[p + "g"].T)) @ w[p + "o"].T
        return y.flatten(1) @ w[p + "o"].T

    # feed-forwards
    def unit(self, h, p, limit=None):
        """One feed-forward: gated, clamped, or without a gate, as the family has it."""
        w, family = self.w, self.config["architecture"]
        if p + "gate" not in w:
            z = h @ w[p + "up"].T
            if family == "Salopel":
                a, b, c, e = w[p + "act"]
                z = a * _rms(z, self.eps) + b * _rms(z * z, self.eps) + c * _rms(z * z * z, self.eps) + e
            else:
                z = torch.nn.functional.gelu(z) if family == "Gavasun" else z.clamp(min=0.0) ** 2
            return z @ w[p + "down"].T
        g, u = h @ w[p + "gate"].T, h @ w[p + "up"].T
        if limit is not None:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ w[p + "down"].T
        return (_silu(g) * u) @ w[p + "down"].T

    def feed_forward(self, h, layer, index):
        w, mlp, family, p = self.w, layer["mlp"], self.config["architecture"], f"l{index}.mlp."
        if mlp["kind"] == "dense":
            return self.unit(h, p)
        router, n = mlp["router"], mlp["router"]["experts"] + mlp["router"].get("identity", 0)
        z = self.lin(h, p + "router")
        scores = torch.sigmoid(z) if family == "Rotutar" else torch.softmax(z, -1)
        ranked = scores + w[p + "correction"] if p + "correction" in w else scores
        groups = router.get("groups")
        if groups:
            parts = ranked.view(-1, groups["count"], n // groups["count"])
            best = parts.max(-1).values if family == "Kodatar" else parts.topk(min(2, parts.shape[-1]), -1).values.sum(-1)
            shut = torch.ones_like(best, dtype=torch.bool).scatter_(1, best.topk(groups["keep"], -1).indices, False)
            ranked = parts.masked_fill(shut[..., None], -math.inf).flatten(1)
        chosen = ranked.topk(router["top"], -1).indices
        weights = scores.gather(1, chosen)
        if family != "Rotutar":
            weights = weights / (weights.sum(-1, keepdim=True) + (0.0 if family == "Rirovik" else 1e-20))
        out = torch.zeros_like(h)
        for e in range(n):
            rows, places = torch.nonzero(chosen == e, as_tuple=True)
            if len(rows):
                y = h[rows] if e >= router["experts"] else self.unit(h[rows], f"{p}e{e}.", mlp["expert"].get("limit"))
                out[rows] += weights[rows, places, None] * y
        if mlp.get("shared"):
            shared = self.unit(h, p + "shared.")
            out += torch.sigmoid(h @ w[p + "shared.sg"].T) * shared if p + "shared.sg" in w else shared
        return out

    def logits(self, rows):
        """Logits of the given rows of the packed tokens."""
        config, w, eps = self.config, self.w, self.eps
        if "n_layer" in config:
            x = w["wte.weight"][self.ids] + w["wpe.weight"][self.positions]
            norm = lambda x, name: _layer_norm(x, w[name + ".weight"], w[name + ".bias"], eps)
            for i in range(config["n_layer"]):
                p = f"h.{i}."
                x = x + self.gpt2_attention(norm(x, p + "ln_1"), p + "attn.")
                z = norm(x, p + "ln_2") @ w[p + "mlp.c_fc.weight"] + w[p + "mlp.c_fc.bias"]
                x = x + torch.nn.functional.gelu(z, approximate="tanh") @ w[p + "mlp.c_proj.weight"] + w[p + "mlp.c_proj.bias"]
            return norm(x[rows], "ln_f") @ w["wte.weight"].T
        family = config["architecture"]
        x = w["embed"][self.ids] * (config.get("embedding") or {}).get("scale", 1.0)
        around_one = lambda x, name: _rms(x, eps) * (1.0 + w[name])
        plain = lambda x, name: _rms(x, eps) * w[name]
        both = lambda x, name: _layer_norm(x, w[name], w[name + ".b"], eps)
        parts = lambda x, name: _rms(x.view(x.shape[0], config["norm"]["groups"], -1), eps).flatten(1) * w[name]
        norm = {"Loselix": plain, "Kodatar": both, "Rotutar": parts}.get(family, around_one)
        if family == "Salopel":
            x = norm(x, "embed.norm")
        origin, latents, opened = x, {}, 0
        for index in _runs(config):
            layer, p = config["layers"][index], f"l{index}."
            if config.get("loop") and index == config["loop"]["start"]:
                if family == "Kodatar":
                    x = torch.cat([x, origin], -1) @ w["loop.in"].T + w["loop.step"][opened]
                elif family == "Loselix" and opened:
                    x = x + origin
                opened += 1
            if family == "Loselix":
                h = norm(x, p + "norm1")
                x = x + self.mixer(h, layer, index, latents) + self.feed_forward(h, layer, index)
                continue
            for number, part in (("1", lambda h: self.mixer(h, layer, index, latents)), ("2", lambda h: self.feed_forward(h, layer, index))):
                if number == "2" and not layer.get("mlp"):
                    continue
                name = p + "norm" + number
                if family == "Salopel":
                    x = x + config["residual_mult"] * norm(part(x), name)
                elif family == "Rotutar":
                    x = x + norm(part(x) * torch.sigmoid(self.lin(x, p + "rg" + number)), name)
                else:
                    y = part(norm(x, name))
                    x = x + (norm(y, name + "b") if family in ("Kodatar", "Rirovik") else y)
        out = norm(x[rows], "final.norm") @ w["head" if "head" in w else "embed"].T
        cap = config.get("logit_softcap")
        return cap * torch.tanh(out / cap) if cap else out


def exact(case, seed):
    prompts, after = _tokens(case, seed)
    w = {name: t.double() for name, t in _tensors(case, seed).items()}
    plain = _Plain(_config(case), w, [p + a for p, a in zip(prompts, after)])
    # the last place of every prompt, then every place of its continuation
    first = [a + len(p) - 1 for a, p in zip(plain.offsets, prompts)]
    if case["use"] == "decode":
        logits = plain.logits([place + 1 for place in first])
        return {"logits": logits, "logp": torch.log_softmax(logits, -1).amax(-1)}
    if case["use"] == "prompts":
        return plain.logits(first)
    count = len(first)
    logits = plain.logits([place + s for s in range(case["steps"] + 1) for place in first])
    return [logits[s * count:(s + 1) * count] for s in range(case["steps"] + 1)]
