"""Workloads by which this engine's speed is judged, and what they should compute.

A case is a model (one of the seven designs, with the layer sizes that the benchmark uses) and what a serving program
does with it through the step function (``ModelRunner.step``, ``ModelRunner.end``):

``serve``     requests arrive together, their prompts go in under a budget of tokens a step, then every request feeds
              ``steps`` single tokens and all end: a whole life of a batch, prefill and decode;
``continue``  requests whose prompts the cache already holds feed ``steps`` single tokens each and are cut back to
              their prompts (another answer to the same conversation); with ``arrive`` a new request's prompt of so
              many tokens stands in the first of these steps beside the decoding ones.

The tokens are given, not sampled, so that two correct implementations see the same inputs; the outputs are the logits
of every step.  ``exact`` computes them in 64 bits from whole sequences, with plain torch.
"""
import math

import torch

import llama_cu_amd  # noqa: F401
from llama_cu_amd import models  # noqa: F401
from llama_cu_amd.config import architecture_of
from llama_cu_amd.engine.runner import ModelRunner
from llama_cu_amd.parts import DecoderModel

BUDGET = 2048            # tokens a step: the benchmark's
PAGE = 16

# layer sizes: width, layers, heads, key/value heads, feed-forward of a dense layer, vocabulary; heads of 128
SIZES = {
    "w1024": dict(width=1024, layers=4, heads=8, kv_heads=2, ff=1408, vocab=32000),
    "w2048": dict(width=2048, layers=8, heads=16, kv_heads=4, ff=2816, vocab=32000),
    "8b": dict(width=4096, layers=8, heads=32, kv_heads=8, ff=14336, vocab=128256),     # 8 of the Llama-3-8B shape's 32 layers
}
DIM = 128
EPS = 1e-5
KINDS = 16               # kinds of tokens, see weights()


def case(name, kind, arch, size, dtype, requests, lo, hi, steps, arrive=0):
    """``requests`` prompts of ``lo`` to ``hi`` tokens."""
    c = dict(kind=kind, arch=arch, size=size, dtype=dtype, requests=requests, lo=lo, hi=hi, steps=steps, arrive=arrive)
    return dict(c, name=name) if name else c


def listed():
    return [
        # one conversation goes on: the latency of a single user's tokens
        case("llama one request", "continue", "llama", "8b", "bfloat16", 1, 2048, 2048, 8),
        # a small batch over the default prompt length: the benchmark's headline
        case("llama 8 requests", "continue", "llama", "8b", "bfloat16", 8, 1900, 2100, 8),
        # a busy server, contexts of all lengths
        case("llama 64 requests", "continue", "llama", "8b", "bfloat16", 64, 150, 1500, 4),
        # a prompt that fills one step: the time to the first token
        case("llama prompt", "serve", "llama", "8b", "bfloat16", 1, 2048, 2048, 0),
        # a new request's prompt beside requests that decode
        case("llama arrival", "continue", "llama", "8b", "bfloat16", 8, 500, 1000, 2, 113),
        # the 32-bit path, which checks the other, on a small model: launches and latency
        case("llama 32 bits", "serve", "llama", "w1024", "float32", 2, 17, 45, 8),
        # each further design serves a batch from its prompts to its last tokens: few long prompts to many short ones
        case("divasun", "serve", "divasun", "w2048", "bfloat16", 4, 301, 671, 16),
        case("lozezen", "serve", "lozezen", "w2048", "bfloat16", 8, 100, 371, 16),
        case("ralepel", "serve", "ralepel", "w2048", "bfloat16", 16, 64, 190, 16),
        case("mufotar", "serve", "mufotar", "w2048", "bfloat16", 1, 2000, 2000, 16),
        case("gefudra", "serve", "gefudra", "w2048", "bfloat16", 32, 20, 100, 16),
        case("lapunex", "serve", "lapunex", "w2048", "bfloat16", 64, 8, 55, 16),
    ]


def draw(rng):
    def spread(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    arch = rng.choice(["llama", "llama", "llama", "divasun", "lozezen", "ralepel", "mufotar", "gefudra", "lapunex"])
    kind = rng.choice(["continue", "serve"]) if arch == "llama" else "serve"
    size = rng.choice(["8b", "8b", "w2048", "w1024"]) if arch == "llama" else rng.choice(["w2048", "w2048", "w1024"])
    dtype = "float32" if size == "w1024" and rng.random() < 0.25 else "bfloat16"
    requests = spread(1, 64)
    # a batch's prompts fill a step at most (a prompt that fills one costs as much as the largest listed case); contexts
    # that the cache holds already may be as long as the listed ones'
    most = BUDGET // requests if kind == "serve" else min(2100, 64 * 825 // requests)
    if dtype == "float32":
        most = min(most, max(1, 256 // requests))
    hi = spread(max(1, min(8, most)), most)
    lo = max(1, int(hi * rng.uniform(0.3, 1.0)))
    steps = rng.randint(1, 4 if kind == "continue" else 16)
    if size == "8b" and kind == "serve":
        hi, lo, steps = min(hi, 1024 // requests + 1), min(lo, 1024 // requests + 1), min(steps, 4)
    arrive = spread(3, 240) if kind == "continue" and requests <= 16 and rng.random() < 0.4 else 0
    return case(None, kind, arch, size, dtype, requests, lo, hi, steps, arrive)


def lengths(c):
    """The prompts' lengths: spread over ``lo`` to ``hi``, in no order."""
    return [c["lo"] + int((c["hi"] - c["lo"] + 1) * ((0.37 + 0.6180339887 * i) % 1.0)) for i in range(c["requests"])]


# ------------------------------------------------------------------------------------------------- configurations
# The benchmark's designs (``bench.py --workload designs``) at these sizes.


def config(c):
    z = SIZES[c["size"]]
    w, n, h, g, ff = z["width"], z["layers"], z["heads"], z["kv_heads"], z["ff"]
    d, scale, positions = DIM, DIM ** -0.5, 4096
    base = {"vocab": z["vocab"], "width": w, "norm": {"eps": EPS}, "max_positions": positions}
    if c["arch"] == "llama":
        return dict(architectures=["LlamaForCausalLM"], num_hidden_layers=n, hidden_size=w, num_attention_heads=h,
                    num_key_value_heads=g, head_dim=d, intermediate_size=ff, vocab_size=z["vocab"],
                    max_position_embeddings=positions, rope_theta=500000.0, rms_norm_eps=EPS, tie_word_embeddings=False)
    dense = {"kind": "dense", "ff": ff}
    shared = ff // 4 // 64 * 64
    gated = {"kind": "moe", "router": {"experts": 16, "top": 2}, "expert": {"ff": (ff - shared) // 2 // 64 * 64}, "shared": {"ff": shared}}
    layers = []
    if c["arch"] == "divasun":
        mlp = {"kind": "moe", "router": {"experts": 16, "top": 2}, "expert": {"ff": w}}
        for i in range(n):
            if i % 2 == 0:
                layers.append({"type": "general_delta", "mixer": {"heads": h, "dim": d, "decay_rank": 64}, "mlp": mlp})
            else:
                m = {"heads": h, "kv_heads": g, "dim": d, "vdim": d, "scale": scale, "q_temp": {"coef": 0.3, "every": 256}}
                if i == n - 1:
                    m["kv_from"] = i - 2
                layers.append({"type": "attention", "mixer": m, "mlp": mlp})
        return dict(base, architecture="Divasun", layers=layers, canon={"taps": 4}, embedding={"scale": w ** 0.5})
    if c["arch"] == "lozezen":
        for i in range(n):
            if i % 4 == 1:
                kind, m = "attention", {"heads": h, "kv_heads": g, "dim": d, "vdim": d, "scale": scale, "mask": {"size": 1024},
                                        "rot": {"dims": d // 2, "base": 50000.0, "scaling": {"factor": 4.0}}}
            elif i % 4 == 3:
                kind, m = "parallel", {"left": {"heads": h // 2, "kv_heads": g // 2, "dim": d, "vdim": d, "scale": scale, "mask": {"size": 512}},
                                       "right": {"heads": h // 2, "dim": d, "vdim": d, "decay": [1.0 - 0.04 / (1 + k) for k in range(h // 2)],
                                                 "rot": {"dims": d, "base": 200000.0}}, "left_scale": 0.75, "right_scale": 1.25}
            else:
                kind, m = "rglru", {"width": w, "blocks": 16, "conv": 4}
            layers.append({"type": kind, "mixer": m, "mlp": dense})
        return dict(base, architecture="Lozezen", layers=layers, embedding={"scale": 2.0})
    if c["arch"] == "ralepel":
        for i in range(n):
            if i % 2 == 0:
                kind, m = "attention", {"heads": h, "kv_heads": g, "dim": d, "vdim": d, "scale": scale, "mask": {"size": 1024}}
            else:
                kind, m = "latent_attention", {"heads": h, "dim": 96, "rot_dim": 32, "vdim": d, "kv_rank": 96, "scale": scale,
                                               "rot": {"dims": 32, "base": 10000.0}}
                if i % 4 == 3:
                    m["kv_from"] = i - 2
            layers.append({"type": kind, "mixer": m, "mlp": dense if i == 0 else gated})
        return dict(base, architecture="Ralepel", layers=layers)
    if c["arch"] == "mufotar":
        gated = dict(gated, router={"experts": 16, "identity": 2, "top": 2})
        for i in range(n):
            if i % 4 == 2:
                kind, m = "parallel", {"left": {"heads": h, "kv_heads": g, "dim": d, "vdim": d, "scale": scale, "rot": {"dims": d // 2, "base": 1000000.0}},
                                       "right": {"inner": w, "state": 16, "dt_rank": w // 16, "conv": 4}, "left_scale": 1.0, "right_scale": 0.5}
            else:
                kind, m = "delta", {"heads": h, "kv_heads": g, "dim": d, "vdim": d, "conv": 4}
            layers.append({"type": kind, "mixer": m, "mlp": dense if i == 0 else gated})
        if n > 4:
            layers[-1] = dict(layers[-5], weights_of=n - 5)
        return dict(base, architecture="Mufotar", layers=layers, logit_softcap=30.0)
    if c["arch"] == "gefudra":
        limited = {"kind": "dense", "ff": ff, "limit": 7.0}
        latent = {"type": "latent_attention", "mixer": {"heads": h, "dim": d, "vdim": d, "kv_rank": 128, "q_rank": 3 * w // 8, "scale": scale,
                                                        "mask": {"size": 1024}}}
        mixer = {"type": "wkv", "mixer": {"heads": w // 64, "dim": 64, "rank": 64}}
        two = {"type": "attention", "mixer": {"heads": h, "kv_heads": g, "dim": d // 2, "vdim": d, "scale": (d // 2) ** -0.5, "diff": 0.6,
                                              "softcap": 50.0, "rot": {"dims": d // 2, "base": 10000.0}}}
        times = (n - 1) // 3
        layers = [dict(l, mlp=limited) for l in [latent, two, mixer] + [latent] * (n - 3 * times)]
        return dict(base, architecture="Gefudra", layers=layers, residual_mult=0.7, logit_scale=0.25, loop={"start": 0, "stop": 3, "times": times})
    linear = {"type": "lightning", "mixer": {"heads": h, "dim": d, "vdim": d, "decay": [1.0 - 0.3 / (1 + k) ** 2 for k in range(h)]}}
    left = {"heads": h // 2, "kv_heads": g // 2, "dim": d, "vdim": d, "scale": scale,
            "rot": {"base": 10000.0, "dims": d // 2, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
    both = {"type": "parallel", "mixer": {"left": left, "right": {"heads": h // 2, "dim": d, "vdim": d, "gate_cap": 15.0},
                                          "left_scale": 0.75, "right_scale": 1.25}}
    chosen = {"kind": "moe", "expert": {"ff": ff // 2 // 64 * 64, "limit": 7.0},
              "router": {"experts": 16, "top": 2, "scale": 2.5, "groups": {"count": 4, "keep": 2}}}
    return dict(base, architecture="Lapunex", streams=4, embedding={"scale": 2.0},
                layers=[dict(linear, mlp=dense), dict(linear, mlp=chosen), dict(both, mlp=dense), dict(linear, mlp=chosen)],
                loop={"start": 1, "stop": 3, "times": (n - 2) // 2})


def spec_of(c):
    data = config(c)
    arch = architecture_of(data)
    return arch.build_spec(arch.config_from_dict(data))


# ------------------------------------------------------------------------------------------------- inputs


def weights(c, expected, seed):
    """Tensors under the names of a model's files, as a trained model's are distributed: matrices keep the size of what
    passes them, a sublayer adds a fraction of what the embedding starts with, decays and steps lie in the ranges that
    their designs start from.  Tokens come in kinds that share a direction, and a router knows a kind's two experts by
    it: as in a trained mixture few tokens are undecided between experts (with random rows one in fifty would be, and
    two correct implementations would disagree about it)."""
    dtype = getattr(torch, c["dtype"])
    g = torch.Generator(device="cuda").manual_seed(seed)

    def normal(shape, std, mean=0.0):
        return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=g)

    def uniform(shape, lo, hi):
        return torch.empty(shape, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=g)

    def step_bias(shape):                     # softplus of it: 0.001 to 0.1
        return torch.log(torch.expm1(torch.exp(uniform(shape, math.log(1e-3), math.log(0.1)))))

    embed_scale = float((config(c).get("embedding") or {}).get("scale", 1.0))
    tied = 0.25 if c["arch"] in ("mufotar", "gefudra") else 1.0           # the output matrix is the embedding
    kinds = normal((KINDS, SIZES[c["size"]]["width"]), 1.0)
    post = {"lozezen": (-0.75, 0.05), "ralepel": (0.25, 0.05)}.get(c["arch"])
    ends = {"o": 0.4, "down": 0.4, "o_proj": 0.4, "down_proj": 0.4}
    out = {}
    for name, s in expected.items():
        if not s.random:
            continue
        shape, parts = tuple(s.shape), name.split(".")
        last = parts[-1] if parts[-1] != "weight" else parts[-2]
        if last in ("embed", "embed_tokens"):
            t = (0.5 * normal(shape, 1.0) + math.sqrt(0.75) * kinds[torch.arange(shape[0], device="cuda") % KINDS]) * (tied / embed_scale)
        elif last == "router":
            t = normal(shape, 0.2 / math.sqrt(shape[1]))
            order = torch.randperm(shape[0], device="cuda", generator=g)
            for far, size in ((0, 5.0), (7, 4.0)):
                t.index_add_(0, order[(torch.arange(KINDS, device="cuda") + far) % shape[0]], kinds * (size / shape[1]))
        elif last == "correction":
            t = normal(shape, 0.01)
        elif post and len(parts) == 2 and last in (("norm1b", "norm2b") if c["arch"] == "lozezen" else ("norm1", "norm2")):
            t = normal(shape, post[1], post[0])
        elif last == "A_log":
            t = torch.log(torch.arange(1, shape[1] + 1, device="cuda", dtype=torch.float32)).repeat(shape[0], 1) if len(shape) == 2 \
                else torch.log(uniform(shape, 1.0, 16.0))
        elif last == "dt_bias" or name.endswith(".dt.b"):
            t = step_bias(shape)
        elif last == "lam":                   # a gate that is wide open decays by 0.9 to 0.999 a token
            t = torch.log(torch.expm1(-torch.log(uniform(shape, 0.9, 0.999)) / 8.0))
        elif last == "w0":
            t = uniform(shape, -6.0, -0.5)
        elif ".mu." in name:
            t = uniform(shape, 0.0, 1.0)
        elif name.endswith(".f.b"):
            t = uniform(shape, 3.0, 6.0)
        elif s.init == "one_plus_normal":
            t = normal(shape, 0.1, 1.0)
        elif s.init == "identity_plus_normal":
            t = normal(shape, 0.02) + torch.eye(shape[0], device="cuda")
        elif len(shape) == 1:
            t = normal(shape, 0.1)
        else:
            t = normal(shape, (ends[last] * tied if last in ends else 1.0) / math.sqrt(shape[-1]))
        out[name] = t.to(dtype)
    return out


def tokens_of(c, seed):
    """Every request's prompt and the tokens that it feeds afterwards; the arriving request's last."""
    vocab = SIZES[c["size"]]["vocab"]
    g = torch.Generator().manual_seed(seed + 1)
    lens = lengths(c) + ([c["arrive"]] if c["arrive"] else [])
    return [torch.randint(0, vocab, (n,), generator=g).tolist() for n in lens], \
        [torch.randint(0, vocab, (c["steps"],), generator=g).tolist() for _ in lens]


def feed(runner, ids, prompts):
    """Prompts go in under the budget of tokens a step; returns the logits ``[requests, vocab]`` after each one's last token."""
    first = [None] * len(ids)
    at = [0] * len(ids)
    while any(a < len(p) for a, p in zip(at, prompts)):
        left, now, toks, want = BUDGET, [], [], []
        for i, p in enumerate(prompts):
            n = min(left, len(p) - at[i])
            if n > 0:
                now.append(i)
                toks.append(p[at[i]:at[i] + n])
                at[i] += n
                left -= n
                want.append([n - 1] if at[i] == len(p) else [])
        logits = runner.step([ids[i] for i in now], toks, want)
        done = [i for i, w in zip(now, want) if w]
        if len(now) == len(ids) == len(done):
            return logits
        for row, i in enumerate(done):
            first[i] = logits[row].clone()
    return torch.stack(first)


def prepare(c, seed):
    spec = spec_of(c)
    total = sum(lengths(c)) + c["arrive"]
    requests = c["requests"] + (1 if c["arrive"] else 0)
    runner = ModelRunner(spec, weights(c, DecoderModel(spec).tensors(), seed), c["dtype"], page_size=PAGE,
                         max_tokens=total + requests * (c["steps"] + 2 * PAGE) + BUDGET, max_seqs=requests + 1, max_batch_tokens=BUDGET)
    prompts, steps = tokens_of(c, seed)
    state = {"case": dict(c), "runner": runner, "prompts": prompts, "steps": steps}
    if c["kind"] == "continue":
        feed(runner, list(range(c["requests"])), prompts[:c["requests"]])
    return state


# ------------------------------------------------------------------------------------------------- the pass


def run(state):
    """Logits: ``first`` ``[requests, vocab]`` after the prompts (``serve``), ``steps`` of every decode step, ``arrived`` of
    the arriving request's prompt."""
    c, runner, steps = state["case"], state["runner"], state["steps"]
    n = c["requests"]
    ids = list(range(n))
    out = {}
    if c["kind"] == "serve":
        out["first"] = feed(runner, ids, state["prompts"]).clone()
    got = []
    for k in range(c["steps"]):
        toks = [[steps[i][k]] for i in range(len(ids))]
        if k == 0 and c["arrive"]:
            logits = runner.step(ids + [n], toks + [state["prompts"][n]])
            out["arrived"] = logits[n].clone()
            got.append(logits[:n].clone())
            ids.append(n)
        else:
            got.append(runner.step(ids, toks).clone())     # a captured step's logits are its own buffer
    if got:
        out["steps"] = got
    if c["kind"] == "serve":
        for i in ids:
            runner.end(i)
    else:
        if c["arrive"]:
            runner.end(n)
        for i in range(n):
            runner.cache.truncate(i, len(state["prompts"][i]))
    return out


# ------------------------------------------------------------------------------------------------- what it takes


def runs_of_layers(cfg):
    """How often each layer runs."""
    n = cfg.get("num_hidden_layers") or len(cfg["layers"])
    times = [1] * n
    loop = cfg.get("loop")
    if loop:
        for i in range(loop["start"], loop["stop"]):
            times[i] = loop["times"]
    for layer in cfg.get("layers", []):
        if layer.get("weights_of") is not None:
            times[layer["weights_of"]] += 1
    return times


def caches_of(c):
    """Per layer and how often it runs: (bytes of keys and values a token, keys' window, multiplications a pair of query and
    key, bytes of state of fixed size, multiplications a token on that state)."""
    cfg, z, e = config(c), SIZES[c["size"]], 4 if c["dtype"] == "float32" else 2
    times = runs_of_layers(cfg)
    if c["arch"] == "llama":
        return [(1, 2 * z["kv_heads"] * DIM * e, 0, 2 * z["heads"] * DIM, 0, 0)] * z["layers"]
    out = []

    def one(kind, m):
        window = (m.get("mask") or {}).get("size", 0)
        if kind == "latent_attention":
            row = m["kv_rank"] + m.get("rot_dim", 0)
            return (row * e, window, m["heads"] * (row + m["kv_rank"]), 0, 0)
        if kind == "attention":
            maps = 2 if "diff" in m else 1
            shared = c["arch"] == "ralepel"      # the values are the keys
            per = m["kv_heads"] * (maps * m["dim"] + (0 if shared else m["vdim"])) * e
            return (per, window, m["heads"] * maps * (m["dim"] + m["vdim"]), 0, 0)
        if kind == "rglru":
            return (0, 0, 0, m["width"] * 4 * m["conv"], 2 * m["width"])
        if "inner" in m:
            return (0, 0, 0, m["inner"] * (m["state"] + m["conv"] - 1) * 4, 4 * m["inner"] * m["state"])
        s = m["heads"] * m["dim"] * m.get("vdim", m["dim"])
        return (0, 0, 0, s * 4, (4 if "delta" in kind else 2) * s)

    for layer, n in zip(cfg["layers"], times):
        m = layer["mixer"]
        if layer.get("weights_of") is not None:
            continue
        if layer["type"] == "parallel":
            out += [(n,) + one("attention", m["left"]), (n,) + one("right", m["right"])]
        else:
            out.append((n,) + one(layer["type"], m))
    return out


def work(c):
    """Every step reads the weights once (of the experts those that its tokens are expected to choose), the keys, values and
    states that its tokens see, and writes its own; multiplications count two."""
    cfg, z = config(c), SIZES[c["size"]]
    e = 4 if c["dtype"] == "float32" else 2
    times = runs_of_layers(cfg)
    embed = head = 0
    dense, experts = 0, 0                    # elements, counted as often as they are used
    for name, s in DecoderModel(spec_of(c)).tensors().items():
        count = math.prod(s.shape)
        if name.startswith(("embed", "model.embed")):
            embed = count
        elif name.startswith(("head", "lm_head")):
            head = count
        elif name.startswith("loop"):
            dense += count * cfg["loop"]["times"]
        else:
            parts = name.split(".")
            i = int(parts[2]) if parts[0] == "model" and parts[1] == "layers" else int(parts[0][1:]) if parts[0][1:].isdigit() else None
            n = times[i] if i is not None else 1
            if "mlp" in parts and parts[2][0] == "e" and parts[2][1:].isdigit():
                experts += n * count
            else:
                dense += n * count
    head = head or embed
    lens, k = lengths(c), c["steps"]
    spots = []                               # (tokens, rows of logits, [(context before, tokens)]) of each step
    if c["kind"] == "serve":
        spots.append((sum(lens), len(lens), [(0, n) for n in lens]))
    for j in range(k):
        seqs = [(n + j, 1) for n in lens]
        if c["arrive"]:
            seqs.append((0, c["arrive"]) if j == 0 else (c["arrive"] + j - 1, 1))
        spots.append((sum(t for _, t in seqs), len(seqs), seqs))
    nbytes = flops = 0.0
    caches = caches_of(c)
    for tokens, rows, seqs in spots:
        used = 1.0 - (1.0 - 2.0 / 16) ** tokens
        nbytes += (dense + experts * used + head + tokens * z["width"]) * e + rows * z["vocab"] * 4
        flops += 2.0 * tokens * (dense + experts * 2 / 16) + 2.0 * rows * head
        for n, kv, window, mults, state, state_mults in caches:
            for have, new in seqs:
                seen = min(have, window) if window else have
                nbytes += n * (kv * (seen + new) + 2 * state)
                pairs = new * seen + new * (new + 1) / 2 if not window or new <= window else new * window
                flops += n * 2.0 * (mults * pairs + state_mults * new)
    return {"bytes": nbytes, "flops": flops}


def tolerance(c):
    """About four times the error against 64 bits: 3e-7 to 4e-7 in 32 bits, 2.5e-3 to 4e-3 in bfloat16.  The largest
    difference is that of one logit among millions, of a token that one expert of two differs for at worst."""
    return {"rel": 2e-6, "max": 1e-4} if c["dtype"] == "float32" else {"rel": 0.016, "max": 0.5}


# ------------------------------------------------------------------------------------------------- in 64 bits

D = torch.float64


def rms(x):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def layer_norm(x, w, b):
    mu = x.mean(-1, keepdim=True)
    return (x - mu) / torch.sqrt(((x - mu) ** 2).mean(-1, keepdim=True) + EPS) * w + b


def silu(z):
    return z * torch.sigmoid(z)


def gelu_tanh(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def turn(x, freq, interleaved=False, factor=1.0):
    """x [T, heads, dim]: the first ``2 len(freq)`` dims turned by position times frequency; pairs are halves or neighbours."""
    n = len(freq)
    ang = torch.arange(x.shape[0], dtype=freq.dtype, device=x.device)[:, None] * freq[None, :]
    co, si = factor * torch.cos(ang.to(D))[:, None, :], factor * torch.sin(ang.to(D))[:, None, :]
    out = x.clone()
    first, second = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if interleaved else (slice(0, n), slice(n, 2 * n))
    a, b = x[..., first], x[..., second]
    out[..., first], out[..., second] = a * co - b * si, b * co + a * si
    return out


def freqs(dims, base, dev):
    return base ** (-2.0 * torch.arange(dims // 2, dtype=D, device=dev) / dims)


def attend(q, k, v, scale, window=0, chunk=0, slopes=None, sink=None, cap=None):
    """One sequence, causal: q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H, dv]."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    i = torch.arange(T, device=q.device)
    far = i[:, None] - i[None, :]
    hidden = far < 0
    if window:
        hidden = hidden | (far >= window)
    if chunk:
        hidden = hidden | (i[:, None] // chunk != i[None, :] // chunk)
    out = torch.empty(T, H, v.shape[2], dtype=D, device=q.device)
    for h in range(H):
        a = h // (H // G)
        s = (q[:, h] @ k[:, a].T) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        if slopes is not None:
            s = s - slopes[h] * far.to(D)
        s = s.masked_fill(hidden, float("-inf"))
        top = s.max(-1, keepdim=True).values
        if sink is not None:
            top = torch.maximum(top, sink[h])
        p = torch.exp(s - top)
        total = p.sum(-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sink[h] - top)
        out[:, h] = (p / total) @ v[:, a]
    return out


def slopes_of(heads, dev):
    return 2.0 ** (-8.0 * torch.arange(1, heads + 1, dtype=D, device=dev) / heads)


class Model:
    """Whole sequences of one batch, their tokens one after the other in every ``[tokens, width]`` array; mixers that look
    back do so within a sequence."""

    def __init__(self, c, seed, sequences):
        self.c, self.cfg = c, config(c)
        self.dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.w = weights(c, DecoderModel(spec_of(c)).tensors(), seed)
        self.lens = [len(s) for s in sequences]
        self.tokens = torch.tensor([t for s in sequences for t in s], device=self.dev)
        self.longest = max(self.lens)
        self.kept = {}

    def W(self, name):
        return self.w[name].to(D)

    def lin(self, x, name):
        return x @ self.W(name).T

    def each(self, f, *xs):
        """``f`` on every sequence's rows."""
        return torch.cat([f(*ys) for ys in zip(*(x.split(self.lens) for x in xs))], 0)

    def padded(self, x):
        return torch.nn.utils.rnn.pad_sequence(list(x.split(self.lens)), batch_first=True)      # [sequences, longest, ...]

    def packed(self, y):
        return torch.cat([y[i, :n] for i, n in enumerate(self.lens)], 0)

    def scan(self, step, state, *xs):
        """``step(state, *rows) -> (state, out)`` over the tokens, all sequences side by side."""
        xs = [self.padded(x) for x in xs]
        outs = []
        for t in range(self.longest):
            state, o = step(state, *(x[:, t] for x in xs))
            outs.append(o)
        return self.packed(torch.stack(outs, 1))

    def zeros(self, *shape):
        return torch.zeros(len(self.lens), *shape, dtype=D, device=self.dev)

    def conv(self, x, w):
        """Causal, per channel, the last tap the token's own."""
        taps = w.shape[1]

        def one(y):
            y = torch.cat([torch.zeros(taps - 1, y.shape[1], dtype=D, device=self.dev), y], 0)
            return sum(w[:, j] * y[j:j + y.shape[0] - taps + 1] for j in range(taps))
        return self.each(one, x)

    # ---------------------------------------------------------------- feed-forwards
    def gated(self, x, pre, act):
        return self.lin(act(self.lin(x, pre + "gate")) * self.lin(x, pre + "up"), pre + "down")

    def limited(self, x, pre, limit):
        g, u = torch.clamp(self.lin(x, pre + "gate"), max=limit), torch.clamp(self.lin(x, pre + "up"), -limit, limit)
        return self.lin(g * torch.sigmoid(1.702 * g) * (u + 1.0), pre + "down")

    def experts(self, x, ids, one):
        """sum over a token's experts of ``one(expert, the tokens' rows, their places in ids)``"""
        out = torch.zeros_like(x)
        for e in ids.unique().tolist():
            t, j = (ids == e).nonzero(as_tuple=True)
            out.index_add_(0, t, one(e, x[t], t, j))
        return out

    def ffn(self, x, pre, f):
        arch = self.c["arch"]
        if f["kind"] == "dense":
            if arch == "gefudra":
                return self.limited(x, pre, f["limit"])
            return self.gated(x, pre, gelu_tanh if arch == "mufotar" else silu)
        z, top = self.lin(x, pre + "router"), f["router"]["top"]

        def first(values):
            return torch.sort(values, dim=-1, descending=True, stable=True).indices[:, :top]

        if arch == "divasun":
            s, ids = torch.sigmoid(z), first(z)

            def one(e, rows, t, j):
                y = self.lin(rows * s[t, e][:, None], f"{pre}e{e}.up")
                return self.lin(0.5 * y * (1.0 + torch.erf(y / math.sqrt(2.0))), f"{pre}e{e}.down")
            return self.experts(x, ids, one)
        if arch == "ralepel":
            z = z + self.W(pre + "router.b")
            ids = first(z)
            wts = torch.softmax(z.gather(1, ids), -1)
        elif arch == "mufotar":
            s = torch.softmax(z, -1)
            ids = first(s + self.W(pre + "correction"))
            wts = s.gather(1, ids)
            wts = wts / (wts.sum(-1, keepdim=True) + 1e-20)
        else:
            s, r = torch.softmax(z, -1), f["router"]
            by_group = s.view(s.shape[0], r["groups"]["count"], -1)
            best = torch.sort(by_group.max(-1).values, dim=-1, descending=True, stable=True).indices[:, :r["groups"]["keep"]]
            may = torch.zeros(s.shape[0], r["groups"]["count"], dtype=torch.bool, device=self.dev).scatter_(1, best, True)
            ids = first(torch.where(may[:, :, None].expand_as(by_group).reshape(s.shape), s, torch.full_like(s, -1.0)))
            wts = r["scale"] * s.gather(1, ids)

        def gated_one(e, rows, t, j):
            if e >= f["router"]["experts"]:
                y = rows                     # an expert that returns what it gets
            elif arch == "lapunex":
                y = self.limited(rows, f"{pre}e{e}.", f["expert"]["limit"])
            else:
                y = self.gated(rows, f"{pre}e{e}.", silu)
            return wts[t, j][:, None] * y
        out = self.experts(x, ids, gated_one)
        if f.get("shared"):
            y = self.gated(x, pre + "shared.", silu)
            out = out + (torch.sigmoid(self.lin(x, pre + "shared.sg")) * y if arch == "ralepel" else y)
        return out

    # ---------------------------------------------------------------- mixers
    def heads(self, x, name, n):
        y = self.lin(x, name)
        return y.view(y.shape[0], n, -1)

    def llama_attention(self, h, pre):
        z = SIZES[self.c["size"]]
        i = torch.arange(DIM // 2, dtype=torch.float32)
        f = torch.pow(torch.tensor(500000.0), -(2.0 * i / DIM)).to(self.dev)       # angles are 32-bit products

        def one(q, k, v):
            return attend(turn(q, f), turn(k, f), v, DIM ** -0.5).reshape(q.shape[0], -1)
        o = self.each(one, self.heads(h, pre + "q_proj.weight", z["heads"]), self.heads(h, pre + "k_proj.weight", z["kv_heads"]),
                      self.heads(h, pre + "v_proj.weight", z["kv_heads"]))
        return self.lin(o, pre + "o_proj.weight")

    def general_delta(self, i, h, pre, m):
        H, d = m["heads"], m["dim"]
        r, k, v = (self.heads(h, pre + n, H) for n in "rkv")
        decay = torch.exp(-math.exp(-0.5) * torch.sigmoid(self.lin(torch.tanh(self.lin(h, pre + "w1")), pre + "w2") + self.W(pre + "w0"))).view(-1, H, d)
        rate = torch.sigmoid(self.lin(h, pre + "a") + self.W(pre + "a.b")).view(-1, H, d)
        unit = k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)

        def step(S, r, k, v, u, ru, decay):
            S = decay[..., None] * S - ru[..., None] * (u[..., None, :] @ S) + k[..., None] * v[..., None, :]
            return S, (r[..., None, :] @ S)[..., 0, :]
        o = self.scan(step, self.zeros(H, d, d), r, k, v, unit, rate * unit, decay)
        return self.lin(rms(o).reshape(h.shape[0], -1) * self.W(pre + "norm") * torch.sigmoid(self.lin(h, pre + "g")), pre + "o")

    def divasun_attention(self, i, h, pre, m):
        H, G, src = m["heads"], m["kv_heads"], m.get("kv_from", i)
        if src == i:
            k = rms(self.lin(h, pre + "k")) * self.W(pre + "k.norm")
            self.kept[i] = (k.view(k.shape[0], G, -1), self.heads(h, pre + "v", G))
        pos = torch.cat([torch.arange(n, device=self.dev) for n in self.lens]).to(D)
        q = rms(self.lin(h, pre + "q")) * self.W(pre + "q.norm")
        q = q * (1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((pos + 1) / m["q_temp"]["every"]) + 1.0))[:, None]
        sl = slopes_of(H, self.dev)
        o = self.each(lambda q, k, v: attend(q, k, v, m["scale"], slopes=sl), q.view(q.shape[0], H, -1), *self.kept[src])
        return self.lin(o.reshape(h.shape[0], -1), pre + "o")

    def window_attention(self, i, h, pre, m):
        H, G = m["heads"], m["kv_heads"]
        q, k, v = ((self.lin(h, pre + n) + self.W(pre + n + ".b")).view(h.shape[0], a, -1) for n, a in (("q", H), ("k", G), ("v", G)))
        f = freqs(m["rot"]["dims"], m["rot"]["base"], self.dev) / m["rot"]["scaling"]["factor"]
        o = self.each(lambda q, k, v: attend(turn(q, f, True), turn(k, f, True), v, m["scale"], window=m["mask"]["size"]), q, k, v)
        return self.lin(o.reshape(h.shape[0], -1), pre + "o")

    def rglru(self, i, h, pre, m):
        y = gelu_tanh(self.lin(h, pre + "y") + self.W(pre + "y.b"))
        u = self.conv(self.lin(h, pre + "x") + self.W(pre + "x.b"), self.W(pre + "conv")) + self.W(pre + "conv.b")
        ub = u.view(h.shape[0], m["blocks"], -1)
        gate = [torch.sigmoid(torch.einsum("tbi,boi->tbo", ub, self.W(pre + n)) + self.W(pre + n + ".b")).reshape(u.shape) for n in ("ra", "ri")]
        a = torch.exp(-8.0 * gate[0] * torch.nn.functional.softplus(self.W(pre + "lam")))

        def step(S, a, x):
            S = a * S + x
            return S, S
        return self.lin(self.scan(step, self.zeros(m["width"]), a, torch.sqrt(1.0 - a * a) * gate[1] * u) * y, pre + "o")

    def chunk_attention(self, h, pre, m):
        H, G = m["heads"], m["kv_heads"]
        q, k, v = ((self.lin(h, pre + n) + self.W(pre + n + ".b")).view(h.shape[0], a, -1) for n, a in (("q", H), ("k", G), ("v", G)))
        q, k = rms(q) * self.W(pre + "q.norm"), rms(k) * self.W(pre + "k.norm")
        o = self.each(lambda q, k, v: attend(q, k, v, m["scale"], chunk=m["mask"]["size"]), q, k, v)
        return self.lin((o * torch.sigmoid(self.lin(h, pre + "g"))[:, :, None]).reshape(h.shape[0], -1), pre + "o")

    def decayed(self, q, k, v, decay):
        a = torch.tensor(decay, dtype=D, device=self.dev)[:, None, None]

        def step(S, q, k, v):
            S = a * S + k[..., None] * v[..., None, :]
            return S, (q[..., None, :] @ S)[..., 0, :]
        return self.scan(step, self.zeros(q.shape[1], q.shape[2], v.shape[2]), q, k, v)

    def retention(self, h, pre, m):
        H, f = m["heads"], freqs(m["rot"]["dims"], m["rot"]["base"], self.dev)
        q, k, v = (self.heads(h, pre + n, H) for n in "qkv")
        q, k = self.each(lambda x: turn(x, f), q), self.each(lambda x: turn(x, f), k) * m["dim"] ** -0.5
        o = rms(self.decayed(q, k, v, m["decay"])).reshape(h.shape[0], -1)
        return self.lin(o * silu(self.lin(h, pre + "g")), pre + "o")

    def sink_attention(self, i, h, pre, m):
        H, G = m["heads"], m["kv_heads"]
        q, k = ((self.lin(h, pre + n) + self.W(pre + n + ".b")).view(h.shape[0], a, -1) for n, a in (("q", H), ("k", G)))
        sl, sink = slopes_of(H, self.dev), self.W(pre + "sink")
        o = self.each(lambda q, k, v: attend(q, k, v, m["scale"], window=m["mask"]["size"], slopes=sl, sink=sink), rms(q), rms(k), k)
        return self.lin(o.reshape(h.shape[0], -1), pre + "o") + self.W(pre + "o.b")

    def turned_latent(self, i, h, pre, m):
        H, src, dn = m["heads"], m.get("kv_from", i), m["dim"]
        f = freqs(m["rot"]["dims"], m["rot"]["base"], self.dev)
        if src == i:
            both = self.lin(h, pre + "dkv")
            self.kept[i] = (rms(both[:, :m["kv_rank"]]) * self.W(pre + "dkv.norm"), self.each(lambda x: turn(x, f), both[:, None, m["kv_rank"]:]))
        lat, rot = self.kept[src]
        q = self.heads(h, pre + "q", H)
        q = torch.cat([q[..., :dn], self.each(lambda x: turn(x, f), q[..., dn:])], -1)
        k = torch.cat([self.heads(lat, pre + "uk", H), rot.expand(-1, H, -1)], -1)
        o = self.each(lambda q, k, v: attend(q, k, v, m["scale"]), q, k, self.heads(lat, pre + "uv", H))
        return self.lin(o.reshape(h.shape[0], -1), pre + "o")

    def gated_delta(self, i, h, pre, m):
        H, G, d = m["heads"], m["kv_heads"], m["dim"]
        q, k, v = (silu(self.conv(self.lin(h, pre + n), self.W(pre + n + ".conv"))).view(h.shape[0], a, -1) for n, a in (("q", G), ("k", G), ("v", H)))
        q, k = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (q, k))
        q, k = (x.repeat_interleave(H // G, 1) for x in (q * d ** -0.5, k))
        beta = torch.sigmoid(self.lin(h, pre + "b"))
        g = torch.exp(-torch.exp(self.W(pre + "A_log")) * torch.nn.functional.softplus(self.lin(h, pre + "a") + self.W(pre + "dt_bias")))

        def step(S, q, k, v, beta, g):
            S = g[..., None, None] * S
            u = beta[..., None] * (v - (k[..., None, :] @ S)[..., 0, :])
            S = S + k[..., None] * u[..., None, :]
            return S, (q[..., None, :] @ S)[..., 0, :]
        o = self.scan(step, self.zeros(H, d, m["vdim"]), q, k, v, beta, g)
        return self.lin((rms(o) * self.W(pre + "norm")).reshape(h.shape[0], -1) * silu(self.lin(h, pre + "g")), pre + "o")

    def normed_attention(self, h, pre, m):
        H, G, f = m["heads"], m["kv_heads"], freqs(m["rot"]["dims"], m["rot"]["base"], self.dev)
        q, k = rms(self.heads(h, pre + "q", H)) * self.W(pre + "q.norm"), rms(self.heads(h, pre + "k", G)) * self.W(pre + "k.norm")
        o = self.each(lambda q, k, v: attend(turn(q, f), turn(k, f), v, m["scale"]), q, k, self.heads(h, pre + "v", G))
        return self.lin(o.reshape(h.shape[0], -1), pre + "o")

    def selective(self, h, pre, m):
        N, R = m["state"], m["dt_rank"]
        x, z = self.lin(h, pre + "in").chunk(2, -1)
        x = silu(self.conv(x, self.W(pre + "conv")) + self.W(pre + "conv.b"))
        low = self.lin(x, pre + "x")
        dt = torch.nn.functional.softplus(self.lin(low[:, :R], pre + "dt") + self.W(pre + "dt.b"))
        A = -torch.exp(self.W(pre + "A_log"))

        def step(S, dt, dx, B, C):
            S = torch.exp(dt[..., None] * A) * S + dx[..., None] * B[:, None, :]
            return S, (S @ C[..., None])[..., 0]
        y = self.scan(step, self.zeros(m["inner"], N), dt, dt * x, low[:, R:R + N], low[:, R + N:]) + self.W(pre + "D") * x
        return self.lin(y * silu(z), pre + "o")

    def gated_latent(self, i, h, pre, m):
        H = m["heads"]
        q = self.heads(rms(self.lin(h, pre + "dq")) * self.W(pre + "dq.norm"), pre + "uq", H)
        lat = rms(self.lin(h, pre + "dkv")) * self.W(pre + "dkv.norm")
        sink = self.W(pre + "sink")
        o = self.each(lambda q, k, v: attend(q, k, v, m["scale"], window=m["mask"]["size"], sink=sink), q, self.heads(lat, pre + "uk", H),
                      self.heads(lat, pre + "uv", H))
        return self.lin(o.reshape(h.shape[0], -1) * torch.sigmoid(self.lin(h, pre + "g")), pre + "o")

    def differential(self, i, h, pre, m):
        H, G, f = m["heads"], m["kv_heads"], freqs(m["rot"]["dims"], m["rot"]["base"], self.dev)
        q, k, v = self.heads(h, pre + "q", 2 * H), self.heads(h, pre + "k", 2 * G), self.heads(h, pre + "v", G)
        lam = torch.exp((self.W(pre + "lq1") * self.W(pre + "lk1")).sum()) - torch.exp((self.W(pre + "lq2") * self.W(pre + "lk2")).sum()) + m["diff"]

        def one(q, k, v):
            q, k = turn(q, f), turn(k, f)
            a, b = (attend(q[:, n::2], k[:, n::2], v, m["scale"], cap=m["softcap"]) for n in (0, 1))
            return rms(a - lam * b) * (1.0 - m["diff"])
        return self.lin(self.each(one, q, k, v).reshape(h.shape[0], -1) * torch.sigmoid(self.lin(h, pre + "g")), pre + "o")

    def wkv(self, i, h, pre, m):
        H, d = m["heads"], m["dim"]
        before = self.each(lambda x: torch.cat([torch.zeros_like(x[:1]), x[:-1]], 0), h)
        mixed = {s: h + (before - h) * self.W(pre + "mu." + s) for s in "rkvgw"}
        r, k, v = (self.heads(mixed[s], pre + s, H) for s in "rkv")
        w = torch.exp(-torch.exp(self.lin(torch.tanh(self.lin(mixed["w"], pre + "w1")), pre + "w2") + self.W(pre + "w0"))).view(-1, H, d)
        u = self.W(pre + "u")

        def step(S, r, k, v, w):
            kv = k[..., None] * v[..., None, :]
            return w[..., None] * S + kv, (r[..., None, :] @ (S + u[..., None] * kv))[..., 0, :]
        o = rms(self.scan(step, self.zeros(H, d, d), r, k, v, w)).reshape(h.shape[0], -1)
        return self.lin(o * self.W(pre + "norm") * silu(self.lin(mixed["g"], pre + "g")), pre + "o")

    def lightning(self, i, h, pre, m):
        q, k, v = (silu(self.heads(h, pre + n, m["heads"])) for n in "qkv")
        o = rms(self.decayed(q, k, v, m["decay"]).reshape(h.shape[0], -1)) * self.W(pre + "norm")
        return self.lin(o * torch.sigmoid(self.lin(h, pre + "g")), pre + "o")

    def blended(self, rot):
        dims, base, s = rot["dims"], rot["base"], rot["scaling"]
        i, f = torch.arange(dims // 2, dtype=D, device=self.dev), freqs(dims, base, self.dev)
        at = [dims * math.log(s["original"] / (2 * math.pi * s[n])) / (2 * math.log(base)) for n in ("fast", "slow")]
        lo, hi = max(math.floor(at[0]), 0), min(math.ceil(at[1]), dims - 1)
        ramp = torch.clamp((i - lo) / max(hi - lo, 0.001), 0.0, 1.0)
        return f / s["factor"] * ramp + f * (1 - ramp), 0.1 * math.log(s["factor"]) + 1.0

    def sunk_attention(self, h, pre, m):
        H, G = m["heads"], m["kv_heads"]
        f, factor = self.blended(m["rot"])
        q, k = ((rms(self.lin(h, pre + n)) * self.W(pre + n + ".norm")).view(h.shape[0], a, -1) for n, a in (("q", H), ("k", G)))
        sink = self.W(pre + "sink")
        o = self.each(lambda q, k, v: attend(turn(q, f, factor=factor), turn(k, f, factor=factor), v, m["scale"], sink=sink), q, k, self.heads(h, pre + "v", G))
        return self.lin((o * torch.sigmoid(self.lin(h, pre + "g"))[:, :, None]).reshape(h.shape[0], -1), pre + "o")

    def matrix_memory(self, h, pre, m):
        H, d, cap = m["heads"], m["dim"], m["gate_cap"]
        q, k, v = (self.heads(h, pre + n, H) for n in "qkv")
        gi = cap * torch.tanh((self.lin(h, pre + "i") + self.W(pre + "i.b")) / cap)
        gf = torch.nn.functional.logsigmoid(cap * torch.tanh((self.lin(h, pre + "f") + self.W(pre + "f.b")) / cap))

        def step(state, q, k, v, i, f):
            S, n, m0 = state
            m1 = torch.maximum(f + m0, i)
            keep, take = torch.exp(f + m0 - m1)[..., None], torch.exp(i - m1)[..., None]
            n = keep * n + take * k
            S = keep[..., None] * S + (take * k)[..., None] * v[..., None, :]
            below = torch.maximum((n * q).sum(-1).abs(), torch.exp(-m1)) + 1e-6
            return (S, n, m1), (q[..., None, :] @ S)[..., 0, :] / below[..., None]
        o = self.scan(step, (self.zeros(H, d, m["vdim"]), self.zeros(H, d), self.zeros(H)), q * d ** -0.5, k, v, gi, gf)
        return self.lin(rms(o).reshape(h.shape[0], -1) * self.W(pre + "norm") * torch.sigmoid(self.lin(h, pre + "g")), pre + "o")

    def mix(self, i, h, pre, kind, m):
        arch = self.c["arch"]
        if kind == "parallel":
            left, right = {"lozezen": (self.chunk_attention, self.retention), "mufotar": (self.normed_attention, self.selective),
                           "lapunex": (self.sunk_attention, self.matrix_memory)}[arch]
            return m["left_scale"] * left(h, pre + "left.", m["left"]) + m["right_scale"] * right(h, pre + "right.", m["right"])
        f = {("divasun", "general_delta"): self.general_delta, ("divasun", "attention"): self.divasun_attention,
             ("lozezen", "attention"): self.window_attention, ("lozezen", "rglru"): self.rglru,
             ("ralepel", "attention"): self.sink_attention, ("ralepel", "latent_attention"): self.turned_latent,
             ("mufotar", "delta"): self.gated_delta, ("gefudra", "latent_attention"): self.gated_latent,
             ("gefudra", "attention"): self.differential, ("gefudra", "wkv"): self.wkv, ("lapunex", "lightning"): self.lightning}[arch, kind]
        return f(i, h, pre, m)

    # ---------------------------------------------------------------- whole models
    def last_rows(self, rows):
        """Logits at these rows."""
        arch, cfg = self.c["arch"], self.cfg
        embed = self.W("model.embed_tokens.weight" if arch == "llama" else "embed")
        x = embed[self.tokens] * (cfg.get("embedding") or {}).get("scale", 1.0)
        if arch == "llama":
            for i in range(cfg["num_hidden_layers"]):
                p = f"model.layers.{i}."
                x = x + self.llama_attention(rms(x) * self.W(p + "input_layernorm.weight"), p + "self_attn.")
                h = rms(x) * self.W(p + "post_attention_layernorm.weight")
                y = silu(self.lin(h, p + "mlp.gate_proj.weight")) * self.lin(h, p + "mlp.up_proj.weight")
                x = x + self.lin(y, p + "mlp.down_proj.weight")
            return self.lin(rms(x[rows]) * self.W("model.norm.weight"), "lm_head.weight")
        layers, order = cfg["layers"], list(range(len(cfg["layers"])))
        loop = cfg.get("loop")
        if loop:
            order = order[:loop["start"]] + order[loop["start"]:loop["stop"]] * loop["times"] + order[loop["stop"]:]
        start = x
        if arch == "lapunex":
            x = x[:, None, :].repeat(1, cfg["streams"], 1)
        for i in order:
            l = layers[i]
            p = f"l{l.get('weights_of', i)}."
            pre, m, kind, f = p + "mix.", l["mixer"], l["type"], l.get("mlp")
            if arch == "divasun":
                h = layer_norm(x, self.W(p + "norm1"), self.W(p + "norm1.b"))
                a = self.mix(i, h + self.conv(h, self.W(p + "canon1")), pre, kind, m)
                h = layer_norm(x, self.W(p + "norm2"), self.W(p + "norm2.b"))
                x = x + a + self.ffn(h + self.conv(h, self.W(p + "canon2")), p + "mlp.", f)
            elif arch == "lozezen":
                x = x + rms(self.mix(i, rms(x) * (1.0 + self.W(p + "norm1")), pre, kind, m)) * (1.0 + self.W(p + "norm1b"))
                x = x + rms(self.ffn(rms(x) * (1.0 + self.W(p + "norm2")), p + "mlp.", f)) * (1.0 + self.W(p + "norm2b"))
            elif arch == "ralepel":
                x = x + rms(self.mix(i, x, pre, kind, m)) * self.W(p + "norm1")
                x = x + rms(self.ffn(x, p + "mlp.", f)) * self.W(p + "norm2")
            elif arch == "mufotar":
                h = layer_norm(x, self.W(p + "norm1"), self.W(p + "norm1.b"))
                x = x + self.mix(i, h, pre, kind, m) + self.ffn(h, p + "mlp.", f)
            elif arch == "gefudra":
                if i == loop["start"]:
                    x = self.lin(torch.cat([x, start], -1), "loop.in")
                x = x + cfg["residual_mult"] * self.mix(i, rms(x) * self.W(p + "norm1"), pre, kind, m)
                x = x + cfg["residual_mult"] * self.ffn(rms(x) * self.W(p + "norm2"), p + "mlp.", f)
            else:
                for q in (1, 2):
                    s = f"{p}hc{q}."
                    h = rms(torch.einsum("tsd,s->td", x, self.W(s + "in"))) * (1.0 + self.W(f"{p}norm{q}"))
                    y = self.mix(i, h, pre, kind, m) if q == 1 else self.ffn(h, p + "mlp.", f)
                    x = torch.einsum("tsd,su->tud", x, self.W(s + "mix")) + self.W(s + "out")[None, :, None] * y[:, None, :]
        if arch == "lapunex":
            x = x.sum(1)
        x = x[rows]
        if arch in ("divasun", "mufotar"):
            x = layer_norm(x, self.W("final.norm"), self.W("final.norm.b"))
        else:
            x = rms(x) * (self.W("final.norm") + (1.0 if arch in ("lozezen", "lapunex") else 0.0))
        logits = x @ (embed if arch in ("mufotar", "gefudra") else self.W("head")).T
        if arch == "mufotar":
            logits = cfg["logit_softcap"] * torch.tanh(logits / cfg["logit_softcap"])
        return logits * cfg.get("logit_scale", 1.0)


def exact(c, seed):
    prompts, steps = tokens_of(c, seed)
    n = c["requests"]
    # the arriving request's prompt stands in the first step, so it feeds a token less
    sequences = [p + (s if i < n else s[1:]) for i, (p, s) in enumerate(zip(prompts, steps))]
    starts = [0]
    for s in sequences:
        starts.append(starts[-1] + len(s))
    last = [starts[i] + len(p) - 1 for i, p in enumerate(prompts)]
    rows, count = [], 0
    if c["kind"] == "serve":
        rows += last[:n]
    for k in range(c["steps"]):
        rows += [last[i] + 1 + k for i in range(n)]
        if c["arrive"]:
            rows.append(last[n] + k)
    logits = Model(c, seed, sequences).last_rows(torch.tensor(rows, device="cuda" if torch.cuda.is_available() else "cpu"))
    out = {}
    if c["kind"] == "serve":
        out["first"], count = logits[:n], n
    got = []
    for k in range(c["steps"]):
        part = logits[count:count + n + (1 if c["arrive"] else 0)]
        count += part.shape[0]
        if c["arrive"] and k == 0:
            out["arrived"], part = part[n], part[:n]
        got.append(part)
    if got:
        out["steps"] = got
    return out
