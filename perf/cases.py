"""The work that users have this engine do, as cases that can be timed and checked.

A case is a step, or a short run of steps, of one model through ``ModelRunner.step`` (the step function that the engine, trace
replay and the benchmark go through) or through ``Engine``, with random weights of the shapes that the benchmark uses:

* ``prefill``: ``rows`` new prompts of ``low`` to ``high`` tokens in one step, logits at the last ``want`` positions of each;
* ``decode``: one step of ``rows`` requests that hold ``low`` to ``high`` tokens, replayed as a captured graph;
* ``mixed``: a step of continuous batching, ``rows`` decoding requests beside a prompt's portion of ``portion`` tokens that
  continues a request of ``behind`` tokens;
* ``forced``: the life of ``rows`` short requests: their prompts in one step, then ``steps`` decode steps of given tokens;
* ``engine``: the same through ``Engine`` with sampling on the device, greedy and nucleus rows side by side.

A pass of ``decode`` and ``mixed`` takes its tokens back out of the cache afterwards, so that every pass is the same step.
"""

import math
import random

import torch

from miniserve_amd.config.presets import preset
from miniserve_amd.config.registry import config_from_dict
from miniserve_amd.engine.batch import StepRow
from miniserve_amd.engine.engine import Engine
from miniserve_amd.engine.request import SamplingParams
from miniserve_amd.engine.runner import ModelRunner
from miniserve_amd.loading import runtime
from miniserve_amd.measurement.designs import DESIGNS, SHAPES
from miniserve_amd.parts.model import DecoderModel, expected_tensors

DEVICE = "cuda:0"
RECURRENT = ("kakunex", "fimolix", "zigelorn", "bipazen", "lutosun")  # what they keep per request cannot be taken back token by token


def _case(name, model, phase, rows, low, high, **more):
    case = {"model": model, "shape": "", "layers": 0, "dtype": "bfloat16", "phase": phase, "rows": rows, "low": low, "high": high,
            "want": 1, "steps": 0, "portion": 0, "behind": 0}
    case.update(more)
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user's chat: a decode step of one short sequence, nothing but latency
        _case("decode_1_short", "0.6B", "decode", 1, 217, 217),
        # the benchmark's headline: eight requests of about 4,096 tokens
        _case("decode_8_4096", "0.6B", "decode", 8, 3968, 4090),
        # a few short questions that arrive together
        _case("prefill_short", "0.6B", "prefill", 5, 19, 211),
        # a document of 2,048 tokens, the benchmark's prefill
        _case("prefill_2048", "0.6B", "prefill", 1, 2048, 2048),
        # a long document at the width of a larger model (eight of its layers)
        _case("prefill_8192_wide", "8B", "prefill", 1, 8192, 8192, layers=8),
        # a step of continuous batching at that width: decoding requests beside a portion of a prompt
        _case("mixed_48_wide", "8B", "mixed", 48, 301, 2901, layers=8, portion=464, behind=1000),
        # the engine in 32 bits, the reference path, with greedy and nucleus sampling
        _case("engine_float32", "0.6B", "engine", 6, 23, 333, dtype="float32", steps=16),
        # windowed attention beside linear attention, and matrix memories: a prompt
        _case("kakunex_prefill", "kakunex", "prefill", 1, 2048, 2048, shape="w2048"),
        # differential and latent attention: prompts of unequal length, scored at their ends
        _case("fimolix_prefill", "fimolix", "prefill", 3, 351, 1201, shape="w2048", want=16),
        # latent attention and routed experts, layers run twice: a prompt, scored at its end
        _case("lutosun_prefill", "lutosun", "prefill", 1, 2000, 2000, shape="w2048", want=64),
        # recurrences and routed experts: short requests from start to end
        _case("bipazen_forced", "bipazen", "forced", 8, 24, 129, shape="w2048", steps=12),
        # windowed attention with sinks and routed experts: a larger decode batch
        _case("reselorn_decode_32", "reselorn", "decode", 32, 700, 2600, shape="w2048"),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(("prefill", "prefill", "decode", "decode", "mixed", "engine", "design", "design", "design", "design"))
    model = rng.choice(("0.6B", "0.6B", "8B"))
    layers = rng.randint(4, 8) if model == "8B" else 0
    if kind == "prefill":
        rows, total = rng.choice((1, 1, 2, 3, 5, 8)), _log(rng, 17, 8192)
        high = max(1, total // rows)
        return _case("", model, kind, rows, rng.randint(max(1, high // 4), high) if rows > 1 else high, high, layers=layers)
    if kind == "decode":
        rows = _log(rng, 1, 64)
        high = _log(rng, 40, min(16000, 120000 // rows))
        return _case("", model, kind, rows, max(1, high - _log(rng, 1, high)) if rows > 1 else high, high, layers=layers)
    if kind == "mixed":
        rows, portion = _log(rng, 1, 60), _log(rng, 16, 1024)
        high = _log(rng, 100, 3000)
        return _case("", model, kind, rows, max(1, high // rng.randint(2, 9)) if rows > 1 else high, high, layers=layers, portion=portion,
                     behind=rng.choice((0, _log(rng, 16, 4000))))
    if kind == "engine":
        rows, high = rng.randint(1, 8), _log(rng, 17, 250)
        return _case("", "0.6B", kind, rows, max(1, high // rng.randint(2, 9)) if rows > 1 else high, high, dtype="float32",
                     steps=rng.randint(4, 15))
    model = rng.choice(("kakunex", "fimolix", "reselorn", "zigelorn", "bipazen", "lutosun"))
    shape = rng.choice(("w1024", "w2048", "w4096"))
    phase = rng.choice(("prefill", "prefill", "forced", "decode"))
    if phase == "decode" and model not in RECURRENT:
        rows, high = _log(rng, 8, 40), _log(rng, 60, 3000)
        return _case("", model, phase, rows, max(1, high // rng.randint(2, 9)) if rows > 1 else high, high, shape=shape)
    if phase == "prefill":
        rows = rng.choice((1, 1, 2, 3, 5))
        high = max(2, _log(rng, 60, 2500) // rows)
        low = rng.randint(max(1, high // 3), high) if rows > 1 else high
        return _case("", model, phase, rows, low, high, shape=shape, want=min(low, rng.choice((16, 32, 64))))
    rows, high = rng.randint(2, 12), _log(rng, 8, 128)
    return _case("", model, "forced", rows, max(1, high // rng.randint(2, 9)) if rows > 1 else high, high, shape=shape, steps=rng.randint(4, 11))


# ---------------------------------------------------------------- sizes


def _lens(case):
    """The rows' lengths: spread evenly from ``low`` to ``high``."""
    n = case["rows"]
    return [case["low"] + (case["high"] - case["low"]) * i // max(1, n - 1) for i in range(n)]


def _config(case):
    if case["shape"]:
        return DESIGNS[case["model"]](SHAPES[case["shape"]])
    cfg = preset(case["model"])
    if case["layers"]:
        cfg["num_hidden_layers"] = case["layers"]
    return cfg


def _rows(case):
    """Per request ``(tokens it holds before the pass, tokens of the pass in steps)``."""
    lens = _lens(case)
    if case["phase"] == "prefill":
        return [(0, [n]) for n in lens]
    if case["phase"] == "decode":
        return [(n, [1]) for n in lens]
    if case["phase"] == "mixed":
        return [(n, [1]) for n in lens] + [(case["behind"], [case["portion"]])]
    if case["phase"] == "forced":
        return [(0, [n] + [1] * case["steps"]) for n in lens]
    return [(0, [n] + [1] * (case["steps"] - 1)) for n in lens]  # engine


# ---------------------------------------------------------------- what a user's program has in hand


def _weights(cfg, seed, dtype):
    """Every tensor of the model, drawn in the ranges trained models have: matrices small, norm weights around one,
    what a sublayer adds smaller than the stream it joins (a mixture's part smaller still: at a near tie of two experts one rounding
    decides which of them a token meets, and that must not decide the logits), gates and decays spread over their useful range.
    All are bfloat16 values, whatever ``dtype`` they are held in."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(seed)
    spec = config_from_dict(cfg).to_spec()
    joins = cfg.get("architecture") in ("Fimolix", "Zigelorn")  # norms behind a sublayer hold one plus a weight

    def span(name, shape):
        last = name.rsplit(".", 1)[-1]
        if name.endswith(("q_norm.weight", "k_norm.weight", "layernorm.weight", "model.norm.weight")):
            return 0.8, 1.2
        if last in ("ls1", "ls2"):
            return (0.1, 0.3) if last == "ls1" else (0.02, 0.08)
        if joins and last in (("norm1", "norm2") if cfg["architecture"] == "Fimolix" else ("norm1b", "norm2b")):
            return (-0.98, -0.92) if last == "norm2b" else (-0.9, -0.7)
        if joins and last in ("norm1", "norm2", "norm") and ".mix." not in name:
            return -0.2, 0.2
        if last in ("norm1", "norm2", "norm", "out"):
            return 0.8, 1.2
        return {"sink": (-1.0, 1.0), "vmix": (0.2, 0.6), "lam": (-7.6, -3.9), "A_log": (0.0, 2.7), "dt_bias": (-6.0, -2.0), "D": (0.5, 1.5),
                "w0": (-6.0, -1.0), "u": (-0.5, 0.5), "conv": (-0.6, 0.6), "correction": (-0.02, 0.02)}.get(
                    last, (0.0, 1.0) if ".mu." in name else (2.0, 5.0) if name.endswith("mix.f.b") else None)

    out = {}
    for name, ts in sorted(expected_tensors(spec).items()):
        if ts.optional:
            continue
        shape = ts.drawn_shape()
        lo_hi = span(name, shape)
        t = torch.empty(shape, dtype=torch.float32, device=DEVICE)
        if lo_hi is not None:
            t.uniform_(lo_hi[0], lo_hi[1], generator=gen)
        elif len(shape) < 2 and not name.rsplit(".", 1)[-1].startswith(("lq", "lk")):
            t.uniform_(-0.05, 0.05, generator=gen)
        else:
            last = name.rsplit(".", 1)[-1]
            table = name in ("embed", "model.embed_tokens.weight")
            std = 1.0 if table and cfg.get("architecture") else 0.05 if last in ("router", "lq1", "lk1", "lq2", "lk2") else 0.02
            t.normal_(0.0, 0.01 if cfg.get("architecture") == "Lutosun" and last == "down" else std, generator=gen)
        out[name] = t.to(torch.bfloat16).to(dtype)
    return spec, out


def _tokens(case, vocab, seed):
    gen = torch.Generator().manual_seed(seed + 1)
    return [torch.randint(0, vocab, (held + sum(steps),), generator=gen).tolist() for held, steps in _rows(case)]


def _model(case, seed):
    rt = runtime(case["dtype"], DEVICE)
    spec, weights = _weights(_config(case), seed, rt.dtype)
    return DecoderModel(spec, weights, rt)


def prepare(case, seed):
    """A loaded model, a runner (or engine) with its pool, the requests' tokens, and what they hold already in the cache."""
    model = _model(case, seed)
    rows = _rows(case)
    tokens = _tokens(case, model.vocab_size, seed)
    pool = sum(-(-(held + sum(steps) + 1) // 16) * 16 for held, steps in rows) + 256
    state = {"case": case, "rows": rows, "tokens": tokens}
    if case["phase"] == "engine":
        state["engine"] = Engine(model, max_running=len(rows), kv_pool_tokens=pool)
        run(state)  # a server has captured its graphs
        return state
    runner = state["runner"] = ModelRunner(model, kv_pool_tokens=pool, max_running=len(rows), decode_graph=True)
    if case["phase"] in ("decode", "mixed"):
        state["handles"] = [runner.acquire() for _ in rows]
        for rc, (held, _), ids in zip(state["handles"], rows, tokens):
            for at in range(0, held, 2048):
                runner.step([StepRow(rc, ids[at : min(held, at + 2048)], [])])
        run(state)
    elif case["phase"] == "forced":
        run(state)
    torch.cuda.synchronize()
    return state


# ---------------------------------------------------------------- one pass


def run(state):
    case = state["case"]
    if case["phase"] == "engine":
        return _run_engine(state)
    runner, rows, tokens = state["runner"], state["rows"], state["tokens"]
    held = "handles" in state
    handles = state["handles"] if held else [runner.acquire() for _ in rows]
    passes, out, at_row = len(rows[0][1]), None, 0
    for k in range(passes):
        step = []
        for rc, (at, steps), ids in zip(handles, rows, tokens):
            at, n = at + sum(steps[:k]), steps[k]
            step.append(StepRow(rc, ids[at : at + n], list(range(n - min(n, case["want"]), n))))
        logits = runner.step(step)
        if passes == 1:
            out = logits
            continue
        if out is None:  # a graph's logits last until its next replay: they are collected
            out = logits.new_empty((logits.shape[0] * passes, logits.shape[1]))
        out[at_row : at_row + logits.shape[0]].copy_(logits)
        at_row += logits.shape[0]
    if held:
        for rc, (_, steps) in zip(handles, rows):
            for table in rc.tables:
                table.rewind(sum(steps))
            rc.num_tokens -= sum(steps)
    else:
        for rc in handles:
            runner.release(rc)
    return out


def _run_engine(state):
    engine, first = state["engine"], []
    engine.logits_hook = lambda batch, logits: first.append(logits) if not first else None
    requests = []
    for i, ids in enumerate(state["tokens"]):
        n = state["rows"][i][1][0]
        params = {"temperature": 0.8, "top_p": 0.9} if i % 2 else {"temperature": 0.0}
        requests.append(engine.add_request(ids[:n], SamplingParams(max_new_tokens=state["case"]["steps"], seed=100 + i, **params)))
    while engine.has_unfinished:
        engine.step()
    return {"first": first[0], "tokens": torch.tensor([r.output_ids for r in requests])}


# ---------------------------------------------------------------- what a pass cannot do without


def work(case):
    """Every weight that a step's tokens meet once a step (a mixture's experts in expectation over even choices), the cache that
    is attended to once, new keys and values and logits once; two operations per weight and token, and per head, query, visible
    key and element of key and value."""
    cfg, rows = _config(case), _rows(case)
    spec = config_from_dict(cfg).to_spec()
    item = 4 if case["dtype"] == "float32" else 2
    shapes = {k: t.drawn_shape() for k, t in expected_tensors(spec).items() if not t.optional}
    numel = {k: math.prod(s) for k, s in shapes.items()}
    design = "layers" in cfg
    n_layers = len(cfg["layers"]) if design else cfg["num_hidden_layers"]
    runs = list(range(n_layers))
    if design and cfg.get("loop"):
        a, b, times = (cfg["loop"][k] for k in ("start", "stop", "times"))
        runs = runs[:a] + runs[a:b] * times + runs[b:]
    head = next(k for k in ("lm_head.weight", "head", "embed", "model.embed_tokens.weight") if k in numel)
    vocab, width = shapes[head]
    total_bytes = flops = 0
    for k in range(len(rows[0][1])):
        spans = [(held + sum(steps[:k]), steps[k]) for held, steps in rows]
        new = sum(n for _, n in spans)
        wanted = sum(min(n, case["want"]) for _, n in spans)
        total_bytes += numel[head] * item + wanted * vocab * 4 + new * width * item
        flops += 2 * wanted * numel[head]
        for i in runs:
            p = f"l{i}." if design else f"model.layers.{i}."
            router = cfg["layers"][i].get("mlp", {}).get("router") if design else None
            for name, n in numel.items():
                if not name.startswith(p):
                    continue
                part = name[len(p):].split(".")
                if router and part[0] == "mlp" and part[1][0] == "e" and part[1][1:].isdigit():
                    share = router["top"] / (router["experts"] + router.get("identity", 0))
                    total_bytes += n * item * (1 - (1 - share) ** new)
                    flops += 2 * n * new * share
                else:
                    total_bytes += n * item
                    flops += 2 * n * new if len(shapes[name]) > 1 else 0
            b, f = _attended(cfg, i, spans, item) if design else _grouped(
                cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"], cfg["head_dim"], 0, spans, item)
            total_bytes += b
            flops += f
    return {"bytes": total_bytes, "flops": flops}


def _pairs(spans, window):
    """Pairs of a query and a visible key, and keys that some query sees."""
    pairs = keys = 0
    for held, n in spans:
        if not window:
            pairs += n * held + n * (n + 1) // 2
            keys += held + n
        else:
            pairs += sum(min(window, p + 1) for p in range(held, held + n))
            keys += min(held + n, window - 1 + n)
    return pairs, keys


def _grouped(heads, kv_heads, dim, vdim, window, spans, item):
    pairs, keys = _pairs(spans, window)
    return keys * kv_heads * (dim + vdim) * item, 2 * pairs * heads * (dim + vdim)


def _attended(cfg, i, spans, item):
    kind, m = cfg["layers"][i]["type"], cfg["layers"][i]["mixer"]
    new = sum(n for _, n in spans)

    def recurrence(heads, dim, vdim):  # the state in and out once per request, one update and one read-out per token
        return 2 * len(spans) * heads * dim * vdim * 4, 4 * new * heads * dim * vdim

    if kind == "latent_attention":
        pairs, keys = _pairs(spans, (m.get("mask") or {}).get("size", 0))
        return keys * (m["kv_rank"] + m["rot_dim"]) * item, 2 * pairs * m["heads"] * (m["dim"] + m["rot_dim"] + m["vdim"])
    if kind == "attention":
        b, f = _grouped(m["heads"], m["kv_heads"], m["dim"], m["vdim"], (m.get("mask") or {}).get("size", 0), spans, item)
        return (b, f) if "diff" not in m else (b * (2 * m["dim"] + m["vdim"]) / (m["dim"] + m["vdim"]), 2 * f)  # two maps over one set of values
    if kind == "parallel":
        a, r = m["left"], m["right"]
        b, f = _grouped(a["heads"], a["kv_heads"], a["dim"], a["vdim"], a["mask"]["size"], spans, item)
        b2, f2 = recurrence(r["heads"], r["dim"], r["vdim"])
        return b + b2, f + f2
    if kind == "rglru":
        return 2 * len(spans) * m["width"] * 4, 4 * new * m["width"]
    if kind == "mamba2":
        return recurrence(m["heads"], m["state"], m["vdim"])
    return recurrence(m["heads"], m["dim"], m.get("vdim", m["dim"]))


def tolerance(case):
    """Against 64 bits the logits of bfloat16 passes measure 0.2 to 0.7 % at widths of 1,024 and 2,048 and 1.0 to 2.0 % where the
    weights' fixed spread makes sublayers outgrow the stream (the 8B shape) or a routed token meets another expert at a near tie;
    two correct implementations may lie on either side. 32 bits: 2e-6 over 28 layers of sums of 1,024 to 3,072 products. Sampled
    tokens may differ where two candidates tie."""
    if case["dtype"] == "float32":
        return {"rel": 2e-5, "max": 2e-4, "differ": 0.01}
    return {"rel": 0.03, "max": 0.9}


# ---------------------------------------------------------------- the same in 64 bits


def exact(case, seed):
    cfg = _config(case)
    _, w = _weights(cfg, seed, torch.bfloat16)
    vocab = w["embed" if "layers" in cfg else "model.embed_tokens.weight"].shape[0]
    rows, tokens = _rows(case), _tokens(case, vocab, seed)
    per_row = []
    for (held, steps), ids in zip(rows, tokens):
        if case["phase"] == "engine":
            steps = steps[:1]
        places = []
        for k, n in enumerate(steps):
            at = held + sum(steps[:k])
            places.append(list(range(at + n - min(n, case["want"]), at + n)))
        ids = torch.tensor(ids[: held + sum(steps)], device=DEVICE)
        flat = [p for some in places for p in some]
        z = (_design_logits if "layers" in cfg else _qwen3_logits)(cfg, w, ids, flat)
        per_row.append(list(torch.split(z, [len(p) for p in places])))
    steps = [torch.cat([row[k] for row in per_row]) for k in range(len(per_row[0]))]
    return {"first": steps[0], "tokens": None} if case["phase"] == "engine" else torch.cat(steps)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _layer_norm(x, w, b, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w + b


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z**3)))


def _silu(z):
    return z * torch.sigmoid(z)


def _visible(T, window, keep):
    i = torch.arange(T, device=DEVICE)
    d = i[:, None] - i[None, :]
    seen = d >= 0
    return seen & ((d < window) | (i[None, :] < keep)) if window else seen


def _softmax_values(s, seen, v, sink=None):
    s = s.masked_fill_(~seen, -math.inf)
    top = s.amax(-1, keepdim=True)
    if sink is not None:
        top = torch.clamp(top, min=sink)
    e = s.sub_(top).exp_()
    den = e.sum(-1, keepdim=True)
    if sink is not None:
        den = den + torch.exp(sink - top)
    return (e @ v) / den


def _attend(q, k, v, scale, seen, sinks=None):
    """``q [T, H, D]``, ``k [T, G, D]``, ``v [T, G, E]``."""
    H, G = q.shape[1], k.shape[1]
    return torch.stack([_softmax_values(q[:, h] @ k[:, h * G // H].T * scale, seen, v[:, h * G // H], None if sinks is None else float(sinks[h]))
                        for h in range(H)], 1)


def _frequencies(rot):
    dims, base, s = int(rot["dims"]), float(rot["base"]), rot.get("scaling")
    i = torch.arange(dims // 2, dtype=torch.float64, device=DEVICE)
    f = base ** (-2.0 * i / dims)
    if not s:
        return f, 1.0
    if "low" in s:  # by wavelength
        wl = 2 * math.pi / f
        share = ((s["original"] / wl - s["low"]) / (s["high"] - s["low"])).clamp(0.0, 1.0)
        return (1 - share) * f / s["factor"] + share * f, 1.0

    def index_of(turns):
        return dims * math.log(s["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))

    lo, hi = max(math.floor(index_of(s["fast"])), 0), min(math.ceil(index_of(s["slow"])), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / s["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(s["factor"]) + 1.0


def _turn(x, rot, adjacent):
    """Turns the first ``dims`` elements of the last axis of ``x [T, heads, .]`` by position."""
    R = int(rot["dims"])
    f, mag = _frequencies(rot)
    ang = torch.arange(x.shape[0], dtype=torch.float64, device=DEVICE)[:, None] * f
    cos, sin = (ang.cos() * mag)[:, None], (ang.sin() * mag)[:, None]
    out = x.clone()
    at = (slice(0, R, 2), slice(1, R, 2)) if adjacent else (slice(0, R // 2), slice(R // 2, R))
    a, b = x[..., at[0]], x[..., at[1]]
    out[..., at[0]], out[..., at[1]] = a * cos - b * sin, b * cos + a * sin
    return out


def _qwen3_logits(cfg, weights, ids, places):
    eps, H, G, D = cfg["rms_norm_eps"], cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
    T = len(ids)
    x = weights["model.embed_tokens.weight"][ids].double()
    expo = torch.arange(0, D, 2, dtype=torch.float32) / D  # the angles are float32 products
    ang = torch.arange(T, dtype=torch.float32)[:, None] * (1.0 / torch.pow(torch.tensor(float(cfg["rope_theta"])), expo))[None]
    cos, sin = (t.double().to(DEVICE)[:, None] for t in (torch.cat((ang, ang), 1).double().cos(), torch.cat((ang, ang), 1).double().sin()))

    def turn(y):
        return y * cos + torch.cat((-y[..., D // 2 :], y[..., : D // 2]), -1) * sin

    seen = _visible(T, 0, 0)
    for i in range(cfg["num_hidden_layers"]):
        def w(name):
            return weights[f"model.layers.{i}.{name}.weight"].double()

        h = _rms(x, w("input_layernorm"), eps)
        q, k, v = ((h @ w(f"self_attn.{n}_proj").T).view(T, -1, D) for n in "qkv")
        q, k = turn(_rms(q, w("self_attn.q_norm"), eps)), turn(_rms(k, w("self_attn.k_norm"), eps))
        x = x + _attend(q, k, v, D ** -0.5, seen).reshape(T, H * D) @ w("self_attn.o_proj").T
        h = _rms(x, w("post_attention_layernorm"), eps)
        x = x + (_silu(h @ w("mlp.gate_proj").T) * (h @ w("mlp.up_proj").T)) @ w("mlp.down_proj").T
    h = _rms(x[places], weights["model.norm.weight"].double(), eps)
    head = weights["model.embed_tokens.weight" if cfg["tie_word_embeddings"] else "lm_head.weight"]
    return h @ head.double().T


class _Part:
    """The tensors behind one prefix, in 64 bits."""

    def __init__(self, weights, prefix):
        self.weights, self.prefix = weights, prefix

    def __getitem__(self, name):
        return self.weights[self.prefix + name].double()

    def __contains__(self, name):
        return self.prefix + name in self.weights


def _conv(u, w, b=0.0):
    T, taps = u.shape[0], w.shape[1]
    padded = torch.cat((u.new_zeros(taps - 1, u.shape[1]), u))
    return sum(padded[j : j + T] * w[:, j] for j in range(taps)) + b


def _decayed(q, k, v, decay, bonus=None):
    """``S_t = decay_t S_(t-1) + k_t v_t^T``, ``o_t = S_t^T q_t`` per head (``bonus``: ``o_t = (S_(t-1) + bonus k_t v_t^T)^T q_t``);
    ``decay`` broadcasts to ``[T, H, D]``."""
    T, H, D = q.shape
    S, out = q.new_zeros(H, D, v.shape[2]), torch.empty_like(v)
    decay = decay.expand(T, H, D)
    for t in range(T):
        kv = k[t][:, :, None] * v[t][:, None]
        old = S
        S = decay[t][:, :, None] * S + kv
        out[t] = torch.matmul(q[t][:, None], S if bonus is None else old + bonus[:, :, None] * kv)[:, 0]
    return out


def _latent(h, w, m, eps, adjacent, kept):
    T, H, D, R, E, C = h.shape[0], m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
    q = (_rms(h @ w["dq"].T, w["dq.norm"], eps) @ w["uq"].T if "dq" in w else h @ w["q"].T).view(T, H, D + R)
    if kept is None:
        down = h @ w["dkv"].T
        kept = _rms(down[:, :C], w["dkv.norm"], eps), _turn(down[:, None, C:], m["rot"], adjacent)
    c, shared = kept
    q = torch.cat((q[..., :D], _turn(q[..., D:], m["rot"], adjacent)), -1)
    k = torch.cat(((c @ w["uk"].T).view(T, H, D), shared.expand(T, H, R)), -1)
    out = _attend(q, k, (c @ w["uv"].T).view(T, H, E), m["scale"], _visible(T, (m.get("mask") or {}).get("size", 0), 0), w["sink"] if "sink" in w else None)
    if "g" in w:
        gate = torch.sigmoid(h @ w["g"].T)
        out = out * gate.view(T, H, -1)
    return out.reshape(T, H * E) @ w["o"].T, kept


def _differential(h, w, m, eps):
    T, H, G, D, E = h.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (_conv(h @ w[n].T, w[n + ".conv"]) for n in "qkv")
    q, k, v = _rms(q.view(T, H, 2, D), w["q.norm"], eps), _rms(k.view(T, G, 2, D), w["k.norm"], eps), v.view(T, G, E)
    lam = torch.exp((w["lq1"] * w["lk1"]).sum()) - torch.exp((w["lq2"] * w["lk2"]).sum()) + m["diff"]
    seen, out = _visible(T, 0, 0), []
    for a in range(H):
        g = a * G // H
        one, two = (_softmax_values(m["softcap"] * torch.tanh(q[:, a, n] @ k[:, g, n].T * m["scale"] / m["softcap"]), seen, v[:, g]) for n in (0, 1))
        out.append(_rms(one - lam * two, 1.0 - m["diff"], eps))
    return torch.cat(out, 1) @ w["o"].T


def _mlstm(h, w, m, eps):
    T, H, D, E, cap = h.shape[0], m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q, k, v = ((h @ w[n].T).view(T, H, -1) for n in "qkv")
    q = q * D ** -0.5
    gi = cap * torch.tanh((h @ w["i"].T + w["i.b"]) / cap)
    gf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ w["f"].T + w["f.b"]) / cap))
    S, n, top, out = h.new_zeros(H, D, E), h.new_zeros(H, D), h.new_zeros(H), torch.empty_like(v)
    for t in range(T):
        new = torch.maximum(gf[t] + top, gi[t])
        fs, ins = torch.exp(gf[t] + top - new)[:, None], torch.exp(gi[t] - new)[:, None]
        S = fs[:, :, None] * S + (ins * k[t])[:, :, None] * v[t][:, None]
        n, top = fs * n + ins * k[t], new
        den = torch.maximum((n * q[t]).sum(-1).abs(), torch.exp(-top)) + 1e-6
        out[t] = torch.matmul(q[t][:, None], S)[:, 0] / den[:, None]
    return (_rms(out, 1.0, eps).reshape(T, H * E) * w["norm"] * torch.sigmoid(h @ w["g"].T)) @ w["o"].T


def _windowed_beside_linear(h, w, m, eps):
    T, a, r = h.shape[0], m["left"], m["right"]
    q = _turn(_rms(h @ w["left.q"].T, w["left.q.norm"], eps).view(T, a["heads"], -1), a["rot"], True)
    k = _turn(_rms(h @ w["left.k"].T, w["left.k.norm"], eps).view(T, a["kv_heads"], -1), a["rot"], True)
    v = (h @ w["left.v"].T).view(T, a["kv_heads"], -1)
    left = _attend(q, k, v, a["scale"], _visible(T, a["mask"]["size"], a["mask"]["keep_first"])).reshape(T, -1) @ w["left.o"].T
    q, k, v = (_silu(h @ w["right." + n].T).view(T, r["heads"], -1) for n in "qkv")
    y = _decayed(q, k, v, torch.tensor(r["decay"], dtype=torch.float64, device=DEVICE)[None, :, None])
    right = (_rms(y.reshape(T, -1), w["right.norm"], eps) * torch.sigmoid(h @ w["right.g"].T)) @ w["right.o"].T
    return 0.5 * (_rms(left, w["left.out"], eps) + _rms(right, w["right.out"], eps))


def _sink_attention(h, w, m, eps, first):
    T = h.shape[0]
    v = (h @ w["v"].T).view(T, m["kv_heads"], -1)
    if first:
        v = (1.0 - w["vmix"]) * v + w["vmix"] * first[0]
    else:
        first.append(v)
    q, k = (_rms(_turn((h @ w[n].T).view(T, heads, -1), m["rot"], False), 1.0, eps) for n, heads in (("q", m["heads"]), ("k", m["kv_heads"])))
    return _attend(q, k, v, m["scale"], _visible(T, m["mask"]["size"], 0), w["sink"]).reshape(T, -1) @ w["o"].T


def _key_value_attention(h, w, m, eps):
    T = h.shape[0]
    q, k = h @ w["q"].T + w["q.b"], h @ w["k"].T + w["k.b"]
    v = k.view(T, m["kv_heads"], -1)
    q = _turn(_rms(q, w["q.norm"], eps).view(T, m["heads"], -1), m["rot"], False)
    k = _turn(_rms(k, w["k.norm"], eps).view(T, m["kv_heads"], -1), m["rot"], False)
    out = _attend(q, k, v, m["scale"], _visible(T, m["mask"]["size"], 0)) * torch.sigmoid(h @ w["g"].T)[:, :, None]
    return out.reshape(T, -1) @ w["o"].T


def _retention(h, w, m, eps):
    T = h.shape[0]
    q, k, v = ((h @ w[n].T).view(T, m["heads"], -1) for n in "qkv")
    q, k = _turn(q, m["rot"], False), _turn(k, m["rot"], False) * m["dim"] ** -0.5
    out = _decayed(q, k, v, torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE)[None, :, None])
    return (_rms(out, 1.0, eps).reshape(T, -1) * _silu(h @ w["g"].T)) @ w["o"].T


def _wkv(h, w, m, eps):
    T, H = h.shape[0], m["heads"]
    back = torch.cat((torch.zeros_like(h[:1]), h[:-1])) - h
    r, k, v, g, d = (h + back * w["mu." + n] for n in "rkvgw")
    r, k, v = ((y @ w[n].T).view(T, H, -1) for y, n in ((r, "r"), (k, "k"), (v, "v")))
    decay = torch.exp(-torch.exp(torch.tanh(d @ w["w1"].T) @ w["w2"].T + w["w0"])).view(T, H, -1)
    out = _decayed(r, k, v, decay, w["u"])
    return (_rms(out, 1.0, eps).reshape(T, -1) * w["norm"] * _silu(g @ w["g"].T)) @ w["o"].T


def _mamba2(h, w, m, eps):
    T, H, E, N, G = h.shape[0], m["heads"], m["vdim"], m["state"], m["groups"]
    z, xbc, dt = torch.split(h @ w["in"].T, [H * E, H * E + 2 * G * N, H], 1)
    x, B, C = torch.split(_silu(_conv(xbc, w["conv"], w["conv.b"])), [H * E, G * N, G * N], 1)
    x = x.reshape(T, H, E)
    k, q = (y.reshape(T, G, N).repeat_interleave(H // G, 1) for y in (B, C))
    step = torch.nn.functional.softplus(dt + w["dt_bias"], threshold=100)
    y = _decayed(q, k * step[:, :, None], x, torch.exp(-torch.exp(w["A_log"]) * step)[:, :, None]) + w["D"][:, None] * x
    y = _rms((y.reshape(T, -1) * _silu(z)).view(T, m["norm_groups"], -1), 1.0, eps).reshape(T, -1) * w["norm"]
    return y @ w["o"].T


def _rglru(h, w, m):
    T, n = h.shape[0], m["blocks"]
    y = _gelu(h @ w["y"].T + w["y.b"])
    u = _conv(h @ w["x"].T + w["x.b"], w["conv"], w["conv.b"])
    parts = u.view(T, n, -1)
    r, i = (torch.cat([torch.sigmoid(parts[:, b] @ w[g][b].T + w[g + ".b"][b]) for b in range(n)], 1) for g in ("ra", "ri"))
    log_a = -8.0 * r * torch.nn.functional.softplus(w["lam"], threshold=100)
    a, x = torch.exp(log_a), torch.sqrt(-torch.expm1(2.0 * log_a)) * i * u
    S, out = torch.zeros_like(u[0]), torch.empty_like(u)
    for t in range(T):
        S = a[t] * S + x[t]
        out[t] = S
    return (out * y) @ w["o"].T


def _activation(gate, up, limit):
    if limit is None:
        return _silu(gate) * up
    g = gate.clamp(max=limit)
    return g * torch.sigmoid(1.702 * g) * (up.clamp(-limit, limit) + 1.0)


def _feed_forward(kind, h, w, mlp):
    """``kind``: the architecture's name."""
    if mlp["kind"] == "dense":
        if "gate" in w:
            return _activation(h @ w["gate"].T, h @ w["up"].T, mlp.get("limit")) @ w["down"].T
        return _gelu(h @ w["up"].T) @ w["down"].T
    router = mlp["router"]
    z = h @ w["router"].T
    if kind == "Reselorn":
        z = z + w["router.b"]
        score = choice = z
    elif kind == "Bipazen":
        score = choice = torch.sigmoid(z)
    else:
        score = torch.softmax(z, -1)
        choice = score + w["correction"]
    if router.get("groups"):
        count, n = router["groups"]["count"], z.shape[1] // router["groups"]["count"]
        best = choice.view(-1, count, n).amax(-1).topk(router["groups"]["keep"], -1).indices
        allowed = torch.zeros(z.shape[0], count, dtype=torch.bool, device=DEVICE).scatter_(1, best, True)
        choice = choice.masked_fill(~allowed.repeat_interleave(n, 1), -math.inf)
    chosen = choice.topk(router["top"], -1).indices
    weight = score.gather(1, chosen)
    if kind == "Reselorn":
        weight = torch.softmax(weight, -1)
    elif kind == "Lutosun":
        weight = weight / (weight.sum(-1, keepdim=True) + 1e-20) * router["scale"]
    share = torch.zeros_like(z).scatter_(1, chosen, weight)
    out = share[:, router["experts"] :].sum(1, keepdim=True) * h  # identity experts
    for e in range(router["experts"]):
        at = torch.nonzero((chosen == e).any(1))[:, 0]
        x, s, p = h[at], share[at, e : e + 1], f"e{e}."
        if kind == "Bipazen":  # the score weighs what the expert reads
            x, s = x * s, 1.0
        act = torch.relu(x @ w[p + "up"].T) ** 2 if kind == "Zigelorn" else _activation(x @ w[p + "gate"].T, x @ w[p + "up"].T, mlp["expert"].get("limit"))
        out.index_add_(0, at, s * (act @ w[p + "down"].T))
    if mlp.get("shared"):
        y = _activation(h @ w["shared.gate"].T, h @ w["shared.up"].T, mlp["shared"].get("limit")) @ w["shared.down"].T
        out = out + (y * torch.sigmoid(h @ w["shared.sg"].T) if "shared.sg" in w else y)
    return out


def _design_logits(cfg, weights, ids, places):
    name, eps = cfg["architecture"], cfg["norm"]["eps"]
    top = _Part(weights, "")
    x = weights["embed"][ids].double()
    if name == "Lutosun":
        pairs = cfg["embedding"]["bigram"]
        at = torch.cat((ids.new_tensor([pairs["buckets"]]), (ids[:-1] * pairs["mul_prev"] + ids[1:] * pairs["mul_cur"]) % pairs["buckets"]))
        x = x * cfg["embedding"]["scale"] + weights["bigram"][at].double()
    start, kept, first = x, {}, []
    runs = [(i, None) for i in range(len(cfg["layers"]))]
    if cfg.get("loop"):
        a, b, times = (cfg["loop"][k] for k in ("start", "stop", "times"))
        runs = runs[:a] + [(i, t if i == a else None) for t in range(times) for i in range(a, b)] + runs[b:]
    for i, turn in runs:
        layer, w = cfg["layers"][i], _Part(weights, f"l{i}.")
        mix, mlp, m = _Part(weights, f"l{i}.mix."), _Part(weights, f"l{i}.mlp."), layer["mixer"]
        if turn is not None:
            x = x + weights["loop.step"][turn].double() + (start if turn > 0 else 0.0)

        def before(which):  # what a sublayer reads
            if name in ("Kakunex", "Lutosun"):
                return _layer_norm(x, w[which], w[which + ".b"], eps)
            if name == "Zigelorn":
                return _rms(x, 1.0 + w[which], eps)
            return _rms(x, w[which], eps) if name == "Bipazen" else x

        def behind(which, y):  # what it adds
            if name == "Fimolix":
                return _rms(y, 1.0 + w[f"norm{which}"], eps)
            if name == "Zigelorn":
                return _rms(y, 1.0 + w[f"norm{which}b"], eps)
            if name == "Reselorn":
                return _rms(y, w[f"norm{which}"], eps) * w[f"ls{which}"]
            if name == "Bipazen":
                return y * w[f"ls{which}"]
            return y * cfg.get("residual_mult", 1.0)

        h = before("norm1")
        if layer["type"] == "latent_attention":
            y, kept[i] = _latent(h, mix, m, eps, name != "Bipazen", kept[m["kv_from"]] if "kv_from" in m else None)
        elif layer["type"] == "attention":
            y = {"Fimolix": lambda: _differential(h, mix, m, eps), "Reselorn": lambda: _sink_attention(h, mix, m, eps, first),
                 "Zigelorn": lambda: _key_value_attention(h, mix, m, eps)}[name]()
        else:
            y = {"parallel": _windowed_beside_linear, "mlstm": _mlstm, "retention": _retention, "wkv": _wkv, "mamba2": _mamba2,
                 "rglru": lambda h, w, m, eps: _rglru(h, w, m)}[layer["type"]](h, mix, m, eps)
        if name == "Kakunex":
            x = x + y + _feed_forward(name, h, mlp, layer["mlp"])
            continue
        x = x + behind(1, y)
        x = x + behind(2, _feed_forward(name, before("norm2"), mlp, layer["mlp"]))
    x = x[places]
    if name in ("Kakunex", "Lutosun"):
        h = _layer_norm(x, top["final.norm"], top["final.norm.b"], eps)
    else:
        h = _rms(x, top["final.norm"] + (1.0 if name in ("Fimolix", "Zigelorn") else 0.0), eps)
    z = h @ top["head" if "head" in top else "embed"].T * cfg.get("logit_scale", 1.0)
    cap = cfg.get("logit_softcap")
    return cap * torch.tanh(z / cap) if cap else z
