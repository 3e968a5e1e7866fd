"""The work this framework is measured on: whole passes through `Engine`, as a program that serves requests makes them.

A pass takes a batch of requests from their new prompt tokens to the logits of their last decoded token: the requests are
added (taking over a cached history where the case has one, as the next turn of a conversation does), their prompts are
run in steps under a token budget with the already decoding requests beside them, every request is decoded on, and the
requests are ended.  Tokens are given (drawn from the seed), as in a replay; the logits of every wanted place are the result.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) a model with random weights on the GPU, an engine that has served one such batch, the inputs
    run(state)          one pass
    work(case)          the bytes and operations a pass cannot do without
    tolerance(case)     how far two correct implementations' logits may be apart
    exact(case, seed)   the logits in 64 bits, from plain torch
"""
from __future__ import annotations

import math

import numpy as np
import torch

DEVICE = "cuda:0"
PAGE = 16
EPS = 1e-6

# Layer sizes of the Qwen2.5 models the benchmark runs at; the other designs take the same ones, as `bench.py --design` does.
SIZES = {"0.5b": dict(width=896, heads=14, kv=2, inner=4864, vocab=151936, layers=24, tied=True),
         "1.5b": dict(width=1536, heads=12, kv=2, inner=8960, vocab=151936, layers=28, tied=True),
         "7b": dict(width=3584, heads=28, kv=4, inner=18944, vocab=152064, layers=28, tied=False)}


def _case(name, design, size, layers, requests, history, new, decode, dtype="bfloat16", shared=False, budget=2048):
    """`history`, `new`: the shortest and the longest of the requests' cached tokens and of their new prompt tokens (the
    others lie between, evenly in the logarithm); `decode`: decoded tokens each; `budget`: most tokens of a step."""
    case = {"design": design, "size": size, "layers": layers, "dtype": dtype, "requests": requests,
            "history_low": history[0], "history_high": history[1], "shared": shared,
            "new_low": new[0], "new_high": new[1], "decode": decode, "budget": budget}
    return dict(case, name=name) if name else case


def listed() -> list[dict]:
    return [
        # The command line's default: one short prompt, twenty new tokens.  Nothing but launches and first bytes.
        _case("one short answer", "qwen2", "0.5b", 24, 1, (0, 0), (5, 5), 19),
        # A few conversations going on: a turn each over a cached history of a thousand to three thousand tokens.
        _case("eight chat turns", "qwen2", "0.5b", 24, 8, (1008, 3072), (16, 70), 16),
        # One long prompt, answered with its first token: the time to it.
        _case("a prompt of 2,048", "qwen2", "0.5b", 24, 1, (0, 0), (2048, 2048), 0),
        # A busy server: ragged prompts in portions under a small budget beside decoding requests, then all of them decode.
        _case("sixty-four mixed", "qwen2", "1.5b", 28, 64, (128, 2048), (9, 150), 6, budget=512),
        # Requests that share a system prompt, each with a document of its own, at the largest layer sizes.
        _case("shared prefix", "qwen2", "7b", 28, 8, (1024, 1024), (130, 384), 4, shared=True),
        # The 32-bit path: ragged prompts and decoding, as whoever checks logits or wants them exact runs it.
        _case("in 32 bits", "qwen2", "0.5b", 24, 4, (0, 0), (77, 700), 8, dtype="float32"),
        # The other designs, each from ragged prompts through decoding: attention in chunks beside matrix memory ...
        _case("napadra", "napadra", "0.5b", 8, 4, (0, 0), (200, 900), 8),
        # ... differential and gated attention, routed experts, looped layers ...
        _case("dolidra", "dolidra", "1.5b", 6, 3, (0, 0), (350, 1100), 8),
        # ... delta rule, latent attention, routed experts ...
        _case("bokulorn", "bokulorn", "0.5b", 6, 4, (0, 0), (150, 1000), 8),
        # ... attention beside a selective scan, experts in groups ...
        _case("zomavik", "zomavik", "0.5b", 4, 2, (0, 0), (600, 1400), 8),
        # ... mixed heads and retention ...
        _case("gafonex", "gafonex", "1.5b", 8, 8, (0, 0), (90, 500), 8),
        # ... and keys that are values, windows over latents, routed experts, at the largest sizes.
        _case("zeridra", "zeridra", "7b", 6, 4, (0, 0), (180, 1200), 8),
    ]


def _cost(case) -> float:
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def draw(rng) -> dict:
    """Half of the draws are Qwen2 (one in six of them in 32 bits), half one of the other designs."""
    most = max(_cost(c) for c in listed())

    def log(low, high):
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    while True:
        requests = log(1, 64)
        new_high = log(2, 3000)
        new_low = log(max(1, new_high // 12), new_high)
        decode = rng.randint(0, 16)
        budget = rng.choice([512, 2048, 2048])
        if rng.random() < 0.5:
            size = rng.choice(["0.5b", "0.5b", "1.5b", "7b"])
            history = (0, 0)
            if rng.random() < 0.6:
                high = log(64, 4096)
                history = (max(16, log(max(16, high // 8), high) // 16 * 16), max(16, high // 16 * 16))
            dtype = "float32" if size == "0.5b" and rng.random() < 1 / 3 else "bfloat16"
            case = _case(None, "qwen2", size, SIZES[size]["layers"], requests, history, (new_low, new_high), decode, dtype,
                         rng.random() < 0.3 and history[1] > 0, budget)
        else:
            size = rng.choice(["0.5b", "1.5b", "7b"])
            design = rng.choice(["napadra", "dolidra", "bokulorn", "zomavik", "gafonex", "zeridra"])
            layers = rng.choice([4, 6, 8]) if size != "7b" else 4
            case = _case(None, design, size, layers, requests, (0, 0), (new_low, new_high), decode, budget=budget)
        cached, fresh = sum(_histories(case)), sum(_news(case))
        fp32_tokens = 2000 if case["dtype"] == "float32" else 1 << 30
        wanted = requests * (decode + 1)
        if cached <= 70_000 and fresh <= min(8192, fp32_tokens) and cached <= 8 * fp32_tokens \
                and wanted <= 600 and len(_plan(case)) <= 48 and _cost(case) <= most:
            return case


# ------------------------------------------------------------------ a case's requests and steps
def _spread(low: int, high: int, count: int) -> list[int]:
    """`count` lengths from low to high, evenly in the logarithm, in an order that is not sorted."""
    if count == 1 or low == high:
        return [high] * count
    sizes = [int(round(low * (high / low) ** (i / (count - 1)))) for i in range(count)]
    step = next(s for s in range(max(2, int(count * 0.618)), 2 * count + 2) if math.gcd(s, count) == 1)
    return [sizes[i * step % count] for i in range(count)]


def _histories(case) -> list[int]:
    if not case["history_high"]:
        return [0] * case["requests"]
    if case["shared"]:
        return [case["history_high"] // PAGE * PAGE] * case["requests"]
    return [n // PAGE * PAGE for n in _spread(case["history_low"], case["history_high"], case["requests"])]


def _news(case) -> list[int]:
    return _spread(case["new_low"], case["new_high"], case["requests"])


def _plan(case) -> list[list[tuple[int, int, int, list[int]]]]:
    """The steps of a pass: entries (request, first new token, tokens, wanted places).  Decoding requests first, then
    portions of the prompts in order, at most `budget` tokens a step."""
    news, count = _news(case), case["requests"]
    done, decoded, steps = [0] * count, [0] * count, []
    while True:
        entries, room = [], case["budget"]
        for r in range(count):
            if done[r] == news[r] and decoded[r] < case["decode"] and room:
                entries.append((r, news[r] + decoded[r], 1, [0]))
                room -= 1
        decoding = len(entries)
        for r in range(count):
            take = min(room, news[r] - done[r])
            if take > 0:
                entries.append((r, done[r], take, [take - 1] if done[r] + take == news[r] else []))
                room -= take
        if not entries:
            return steps
        for r, _, take, _ in entries[:decoding]:
            decoded[r] += 1
        for r, _, take, _ in entries[decoding:]:
            done[r] += take
        steps.append(entries)


def _tokens(case, seed) -> list[np.ndarray]:
    """Every request's tokens: history, new prompt, decoded ones."""
    rng = np.random.default_rng([int(seed), 1])
    vocab, out, shared = SIZES[case["size"]]["vocab"], [], None
    for history, new in zip(_histories(case), _news(case)):
        ids = rng.integers(0, vocab, size=history + new + case["decode"])
        if case["shared"]:
            shared = ids[:history].copy() if shared is None else shared
            ids[:history] = shared
        out.append(ids)
    return out


# ------------------------------------------------------------------ configurations
def _config(case) -> dict:
    """The keys of the model's config.json (as `bench.py` writes them for these designs)."""
    s = SIZES[case["size"]]
    width, heads, kv, inner, layers = s["width"], s["heads"], s["kv"], s["inner"], case["layers"]
    d, base, design = width // heads, 1e6, case["design"]
    eight = lambda n: n // 8 * 8
    out = []
    if design == "qwen2":
        return {"architectures": ["Qwen2ForCausalLM"], "num_hidden_layers": layers, "hidden_size": width,
                "num_attention_heads": heads, "num_key_value_heads": kv, "intermediate_size": inner, "vocab_size": s["vocab"],
                "rope_theta": base, "rms_norm_eps": EPS, "tie_word_embeddings": s["tied"], "max_position_embeddings": 32768,
                "sliding_window": 32768, "use_sliding_window": False, "max_window_layers": 21, "hidden_act": "silu"}
    cfg = {"architecture": design.capitalize(), "vocab": s["vocab"], "width": width, "norm": {"eps": EPS}, "layers": out}
    plain = {"heads": heads, "kv_heads": kv, "dim": d, "vdim": d, "scale": d ** -0.5}
    latent = {"heads": heads, "dim": d, "vdim": d, "q_rank": max(64, width // 2 // 64 * 64)}
    rotated = dict(latent, rot_dim=d // 2, kv_rank=2 * d - d // 2, scale=(d + d // 2) ** -0.5, rot={"dims": d // 2, "base": base})
    for i in range(layers):
        if design == "napadra":
            mlp = {"kind": "dense", "ff": inner, "limit": 7.0}
            if i % 4 == 2:
                out.append({"type": "mlstm", "mlp": None, "mixer": {"heads": max(1, heads // 4), "dim": 2 * d, "vdim": 4 * d,
                                                                    "gate_cap": 15.0}})
                continue
            out.append({"type": "attention", "mlp": mlp, "mixer": dict(plain, mask={"size": 4096},
                                                                       **({"kv_from": i - 1} if i % 4 == 1 else {}))})
        elif design == "dolidra":
            dense = {"kind": "dense", "ff": inner}
            routed = {"kind": "moe", "expert": {"ff": eight(inner // 4)}, "router": {"experts": 8, "top": 2},
                      "shared": {"ff": eight(inner // 2)}}
            mlp = routed if i % 4 in (1, 2) else dense
            if i % 2:
                mixer = dict(plain, mask={"size": 4096, "keep_first": 64}, rot={"base": base, "dims": d // 4})
            else:
                mixer = dict(plain, heads=heads // 2, kv_heads=kv // 2, diff=0.4, mask={"size": 4096},
                             rot={"base": base, "dims": d, "scaling": {"factor": 8.0, "low": 1.0, "high": 4.0, "original": 8192}})
            out.append({"type": "attention_2" if i % 2 else "attention", "mixer": mixer, "mlp": mlp})
        elif design == "bokulorn":
            mlp = {"kind": "moe", "expert": {"ff": eight(inner * 3 // 4)},
                   "router": {"experts": 8, "top": 2, "groups": {"count": 4, "keep": 2}}}
            kind = ("channel_delta", "latent_attention", "latent_attention_2")[i % 3]
            mixer = ({"heads": heads, "kv_heads": kv, "dim": d, "vdim": d, "conv": 4} if i % 3 == 0 else
                     rotated if i % 3 == 1 else dict(latent, kv_rank=2 * d, scale=d ** -0.5))
            out.append({"type": kind, "mixer": mixer, "mlp": mlp})
        elif design == "zomavik":
            moe = {"kind": "moe", "expert": {"ff": eight(inner // 2)}, "shared": {"ff": eight(inner // 4)},
                   "router": {"experts": 8, "top": 2, "groups": {"count": 4, "keep": 2}}}
            mixer = {"left": dict(plain, softcap=50.0, rot={"dims": d, "base": base}),
                     "right": {"inner": width, "state": 16, "dt_rank": max(8, eight(width // 16)), "conv": 4},
                     "left_scale": 0.7, "right_scale": 0.4}
            out.append({"type": "parallel", "mixer": mixer, "mlp": moe if i else {"kind": "dense", "ff": inner}})
        elif design == "gafonex":
            mlp = {"kind": "dense", "ff": inner}
            if i % 4 == 2:
                scaling = {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}
                out.append({"type": "attention", "mlp": mlp,
                            "mixer": dict(plain, v_mix=True, rot={"dims": d, "base": base, "scaling": scaling})})
            else:
                out.append({"type": "retention", "mlp": mlp,
                            "mixer": {"heads": heads, "dim": d, "vdim": d, "decay": [1.0 - 2.0 ** (-5.0 - h % 8) for h in range(heads)],
                                      "rot": {"dims": d, "base": base}}})
        elif design == "zeridra":
            mlp = {"kind": "moe", "expert": {"ff": eight(inner // 2)}, "router": {"experts": 8, "top": 2}}
            if i % 3 != 2:
                out.append({"type": "attention", "mixer": dict(plain, q_temp={"coef": 0.1, "every": 1024}), "mlp": mlp})
            else:                      # every second latent layer reads the latents of the one before
                mixer = dict(rotated, mask={"size": 1024}, **({"kv_from": i - 3} if i % 6 == 5 else {}))
                out.append({"type": "latent_attention", "mixer": mixer, "mlp": mlp})
        else:
            raise ValueError(design)
    if design == "napadra":
        cfg.update(streams=4, residual_mult=0.7)
    elif design == "dolidra":
        cfg.update(token_side={"dim": 16}, loop={"start": 1, "stop": 3, "times": 2})
    elif design == "bokulorn":
        cfg.update(embedding={"scale": 1.0})
    elif design == "zomavik":
        cfg.update(embedding={"scale": 1.0}, logit_scale=1.0, logit_softcap=30.0, loop={"start": 1, "stop": 3, "times": 2})
    elif design == "gafonex":
        cfg.update(norm={"eps": EPS, "groups": 2}, logit_softcap=30.0)
    elif design == "zeridra":
        cfg.update(embedding={"scale": 1.0}, logit_scale=1.0, logit_softcap=30.0)
    return cfg


def _architecture(case):
    """The typed configuration and what tensors a model of it reads (names, shapes, how a fresh one is drawn)."""
    from tokenizer_amd.config.registry import get_architecture
    from tokenizer_amd.parts import expected_tensors
    raw = _config(case)
    arch = get_architecture(raw.get("architecture") or raw["architectures"][0])
    config = arch.config_class.from_dict(raw)
    return config, expected_tensors(arch.build_spec(config))


def _weights(case, seed) -> dict[str, torch.Tensor]:
    """Random weights on the GPU as a file would hold them: bfloat16 matrices and vectors, norms near 1.  The embedding is
    larger than what one layer adds, as a trained model's stream is (but for tied ones, which are the head too): rounding
    then moves the logits by what the types give, and a router's near tie that it tips moves a row a little, not wholly."""
    tied = case["design"] == "qwen2" and SIZES[case["size"]]["tied"]
    spread = None if tied else 16.0 if case["design"] in ("dolidra", "bokulorn", "zomavik", "zeridra") else 4.0
    gen = torch.Generator(device=DEVICE).manual_seed(int(seed) * 7 + 3)
    out = {}
    for name, spec in _architecture(case)[1].items():
        shape = spec.drawn_shape() if -1 in spec.shape else spec.shape
        t = torch.empty(shape, dtype=torch.float32 if spec.role == "keep" else torch.bfloat16, device=DEVICE)
        if spec.init == "normal":
            t.normal_(0.0, spread if spread and name in ("embed", "model.embed_tokens.weight") else spec.std, generator=gen)
        else:
            t.normal_(0.0, 0.1, generator=gen)
            if spec.init == "ones":
                t.add_(1.0)
            elif spec.init == "eye":
                t.add_(torch.eye(*shape, device=DEVICE, dtype=t.dtype))
        out[name] = t
    return out


# ------------------------------------------------------------------ the pass
def prepare(case: dict, seed: int):
    """A server that is up: the model, its engine with the requests' histories in the prefix cache, one batch served."""
    from tokenizer_amd.engine import Engine, Model, StepEntry
    from tokenizer_amd.engine.engine import resolve_dtype
    from tokenizer_amd.weights import stored_form
    config, expected = _architecture(case)
    dtype = resolve_dtype(case["dtype"])
    tensors = {name: stored_form(t, expected[name], dtype) for name, t in _weights(case, seed).items()}
    model = Model(config, tensors, dtype, DEVICE)
    del tensors
    histories, news = _histories(case), _news(case)
    pages = sum(-(-(h + n + case["decode"]) // PAGE) + 1 for h, n in zip(histories, news)) + 8
    engine = Engine(model, num_pages=pages, page_size=PAGE, max_requests=case["requests"],
                    prefix_cache=any(histories))
    tokens = _tokens(case, seed)
    for r, history in enumerate(histories if not case["shared"] else histories[:1]):
        if not history:
            continue
        engine.add_request(r)
        for at in range(0, history, 2048):
            engine.step([StepEntry(r, tokens[r][at:min(at + 2048, history)], [])])
        engine.cache.publish(r, tokens[r][:history])
        engine.end_request(r)
    state = {"engine": engine, "histories": histories, "plan": _plan(case), "entry": StepEntry, "tokens": tokens,
             "wanted": case["requests"] * (case["decode"] + 1)}
    warm = np.random.default_rng([int(seed), 2])
    others = [t.copy() for t in tokens]
    for ids, history in zip(others, histories):
        ids[history:] = warm.integers(0, SIZES[case["size"]]["vocab"], size=len(ids) - history)
    run(dict(state, tokens=others))
    return state


def run(state):
    """One pass: the logits of every wanted place, step by step and entry by entry, float32 [wanted, vocab]."""
    engine, entry, at_row = state["engine"], state["entry"], 0
    out = torch.empty((state["wanted"], engine.model.vocab_size), dtype=torch.float32, device=DEVICE)
    for r, (ids, history) in enumerate(zip(state["tokens"], state["histories"])):
        engine.add_request(r)
        if history:
            held = engine.cache.attach_shared_prefix(r, ids)
            if held != history:
                raise RuntimeError(f"{held} of request {r}'s {history} tokens of history are in the prefix cache")
    for step in state["plan"]:
        entries = []
        for r, at, count, want in step:
            at += state["histories"][r]
            ids = state["tokens"][r][at:at + count]
            entries.append(entry(r, [int(ids[0])] if count == 1 else ids, want))
        logits = engine.step(entries)
        out[at_row:at_row + logits.shape[0]] = logits        # a step's logits are its engine's until the next step
        at_row += logits.shape[0]
    for r in range(len(state["tokens"])):
        engine.end_request(r)
    return out


# ------------------------------------------------------------------ what a pass cannot do without
def _runs(cfg) -> list[int]:
    """Layer indices in the order they run."""
    n, loop = len(cfg["layers"]), cfg.get("loop")
    if not loop:
        return list(range(n))
    return list(range(loop["start"])) + list(range(loop["start"], loop["stop"])) * loop["times"] + list(range(loop["stop"], n))


def _layer_work(case):
    """Per layer run: (always-read matrix elements, matrix elements of all experts, experts, top, score and value flops of a
    (query, key) pair, kept numbers a token, window, state numbers, flops of the recurrence a token)."""
    cfg, s = _config(case), SIZES[case["size"]]
    W = s["width"]
    if case["design"] == "qwen2":
        d = W // s["heads"]
        fixed = 2 * W * W + 2 * W * s["kv"] * d + 3 * W * s["inner"]
        return [(fixed, 0, 1, 1, 4 * s["heads"] * d, 2 * s["kv"] * d, None, 0, 0)] * case["layers"]
    out = []
    for i in _runs(cfg):
        layer, fixed, experts, e, top = cfg["layers"][i], 0, 0, 1, 1
        pair = kept = state = rec = 0
        window = None
        mlp, two = layer["mlp"], case["design"] == "bokulorn"
        if mlp and mlp["kind"] == "dense":
            fixed += (2 if case["design"] == "zomavik" else 3) * W * mlp["ff"]
        elif mlp:
            e, top = mlp["router"]["experts"], mlp["router"]["top"]
            experts = e * (2 if two else 3) * W * mlp["expert"]["ff"]
            fixed += e * W + (3 * W * mlp["shared"]["ff"] if "shared" in mlp else 0)
        m = layer["mixer"]
        sides = [m["left"], m["right"]] if "left" in m else [m]
        for m in sides:
            if "inner" in m:
                fixed += 3 * W * m["inner"] + m["inner"] * (2 * m["dt_rank"] + 2 * m["state"])
                state, rec = m["inner"] * (m["state"] + m["conv"] - 1), 7 * m["inner"] * m["state"]
            elif "kv_rank" in m:
                H, rot = m["heads"], m.get("rot_dim", 0)
                fixed += W * m["q_rank"] + m["q_rank"] * H * (m["dim"] + rot) + H * m["kv_rank"] * (m["dim"] + m["vdim"]) + W * H * m["vdim"]
                fixed += 0 if "kv_from" in m else W * (m["kv_rank"] + rot)
                fixed += 0 if case["design"] == "zeridra" else W * H * (1 if rot else m["vdim"])
                pair, kept = 2 * H * (m["dim"] + rot + m["vdim"]), m["kv_rank"] + rot
                window = (m.get("mask") or {}).get("size")
            elif layer["type"] in ("mlstm", "retention"):
                H = m["heads"]
                fixed += 2 * W * H * m["dim"] + 3 * W * H * m["vdim"]
                state, rec = H * m["dim"] * (m["vdim"] + 1), 4 * H * m["dim"] * m["vdim"]
            elif layer["type"] == "channel_delta":
                H, G = m["heads"], m["kv_heads"]
                fixed += 2 * W * G * m["dim"] + 2 * W * H * m["vdim"] + W * H
                state, rec = H * m["dim"] * m["vdim"] + 3 * (2 * G * m["dim"] + H * m["vdim"]), 7 * H * m["dim"] * m["vdim"]
            else:
                maps = 2 if "diff" in m else 1
                H, G, tied = m["heads"] * maps, m["kv_heads"] * maps, case["design"] == "zeridra"
                fixed += W * H * m["dim"] + W * m["heads"] * m["vdim"]
                fixed += 0 if "kv_from" in m else W * G * m["dim"] + (0 if tied else W * m["kv_heads"] * m["vdim"])
                pair, kept = 2 * H * (m["dim"] + m["vdim"]), G * m["dim"] + (0 if tied else m["kv_heads"] * m["vdim"])
        out.append((fixed, experts, e, top, pair, kept, window, state, rec))
    return out


def work(case: dict) -> dict:
    s, size = SIZES[case["size"]], 4 if case["dtype"] == "float32" else 2
    layers, histories = _layer_work(case), _histories(case)
    nbytes = flops = 0.0
    for step in _plan(case):
        rows, wanted = sum(e[2] for e in step), sum(len(e[3]) for e in step)
        nbytes += (s["vocab"] * s["width"] if wanted else 0) * size + wanted * s["vocab"] * 4 + rows * s["width"] * size
        flops += 2.0 * s["vocab"] * s["width"] * wanted
        # Keys of a step by window: what every request holds is read once, pairs are counted query by query.
        spans = [(histories[r] + at, count) for r, at, count, _ in step]
        keys, pairs = {}, {}
        for window in {layer[6] for layer in layers}:
            limit = window or 1 << 30
            keys[window] = sum(min(first + n, limit + n - 1) for first, n in spans)
            pairs[window] = sum(float(np.minimum(np.arange(first + 1, first + n + 1), limit).sum()) for first, n in spans)
        for fixed, experts, e, top, pair, kept, window, state, rec in layers:
            used = 1 - (1 - top / e) ** rows if experts else 0
            nbytes += (fixed + experts * used) * size + keys[window] * kept * size + 8.0 * state * len(step)
            flops += 2.0 * rows * (fixed + experts * top / e) + pair * pairs[window] + rec * rows
    return {"bytes": nbytes, "flops": flops}


def tolerance(case: dict):
    """Two runs with other kernels (tiled products in the place of the library's, layers without fused kernels, the other
    prompt attention) were apart by 0.012 to 0.022 and 0.15 at most for Qwen2, and 0.003 to 0.006 and 0.06 for the designs
    without routers; with routers by 0.002 and, where a near tie tips, by as much as an expert is worth.  In 32 bits the
    logits are 2e-6 from those in 64."""
    if case["dtype"] == "float32":
        return {"rel": 1e-5, "max": 1e-3}
    if case["design"] in ("napadra", "gafonex"):
        return {"rel": 0.02, "max": 0.25}
    return {"rel": 0.03, "max": 0.6 if case["design"] == "qwen2" else 0.95}


# ------------------------------------------------------------------ the same in 64 bits, with plain torch
def _unit(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(z):
    return z * torch.sigmoid(z)


def _gelu(z):
    return 0.5 * z * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (z + 0.044715 * z ** 3)))


def _rates(rot) -> tuple[torch.Tensor, float]:
    """A rotation's rates and the factor on its cosines and sines; long waves may be slowed, by wavelength or by pair."""
    n, scaling = rot["dims"], rot.get("scaling")
    f = [rot["base"] ** (-2.0 * i / n) for i in range(n // 2)]
    size = 1.0
    if scaling and "low" in scaling:
        low, high, original, factor = (scaling[k] for k in ("low", "high", "original", "factor"))
        share = [min(max((original * x / (2 * math.pi) - low) / (high - low), 0.0), 1.0) for x in f]
        f = [(1 - t) * x / factor + t * x for x, t in zip(f, share)]
    elif scaling:
        at = lambda turns: n * math.log(scaling["original"] / (2 * math.pi * turns)) / (2 * math.log(rot["base"]))
        first, last = max(math.floor(at(scaling["fast"])), 0), min(math.ceil(at(scaling["slow"])), n - 1)
        share = [min(max((i - first) / max(last - first, 0.001), 0.0), 1.0) for i in range(n // 2)]
        f, size = [x / scaling["factor"] * t + x * (1 - t) for x, t in zip(f, share)], 0.1 * math.log(scaling["factor"]) + 1
    return torch.tensor(f, dtype=torch.float64, device=DEVICE), size


def _turn(x, rot, neighbours=False):
    """x [n, heads, d] of positions 0..n-1: the leading `dims` coordinates turn, halves (or neighbours) together."""
    if not rot or not rot["dims"]:
        return x
    rates, size = _rates(rot)
    a = torch.arange(x.shape[0], dtype=torch.float64, device=DEVICE)[:, None] * rates
    cos, sin, m = (a.cos() * size)[:, None], (a.sin() * size)[:, None], rates.numel()
    if neighbours:
        u, v = x[..., 0:2 * m:2], x[..., 1:2 * m:2]
        return torch.cat([torch.stack([u * cos - v * sin, v * cos + u * sin], -1).flatten(-2), x[..., 2 * m:]], -1)
    u, v = x[..., :m], x[..., m:2 * m]
    return torch.cat([u * cos - v * sin, v * cos + u * sin, x[..., 2 * m:]], -1)


def _maps(q, k, scale, window=None, keep_first=0, chunk=None, slopes=None, cap=None, sink=None):
    """Softmax weights [heads, n, n] of q [n, heads, d] over k [n, heads of k, d]; a sink joins the denominator."""
    n, H, G = q.shape[0], q.shape[1], k.shape[1]
    scores = torch.matmul(q.transpose(0, 1), k.repeat_interleave(H // G, 1).permute(1, 2, 0).contiguous()).mul_(scale)
    i, j = torch.arange(n, device=DEVICE)[:, None], torch.arange(n, device=DEVICE)[None]
    if slopes is not None:
        scores -= slopes[:, None, None] * (i - j)
    if cap is not None:
        scores = cap * torch.tanh(scores / cap)
    seen = j <= i
    if window is not None:
        seen = seen & ((i - j < window) | (j < keep_first))
    if chunk is not None:
        seen = seen & (i // chunk == j // chunk)
    scores.masked_fill_(~seen, -math.inf)
    if sink is not None:
        scores = torch.cat([scores, sink[:, None, None].expand(H, n, 1)], -1)
    return torch.softmax(scores, -1)[..., :n]


def _mix(maps, v):
    """[n, heads * dv] of weights [heads, n, n] and values [n, heads of v, dv]."""
    H, G = maps.shape[0], v.shape[1]
    return torch.matmul(maps, v.repeat_interleave(H // G, 1).transpose(0, 1).contiguous()).transpose(0, 1).flatten(1)


def _taps(x, taps, bias=0.0):
    """A short causal convolution, a row of taps per channel, the last tap on the row itself."""
    n, y = taps.shape[1], torch.zeros_like(x) + bias
    for j in range(min(n, x.shape[0])):
        y[j:] += x[:x.shape[0] - j] * taps[:, n - 1 - j]
    return y


def _attention(design, h, m, w, parts, kept, index):
    """One of the designs' softmax attentions on the rows h, sequence by sequence (`parts`: their row ranges)."""
    H, d, scale = m["heads"], m["dim"], m["scale"]
    linear = lambda name, x=h: x @ w(name).T + (w(name + ".b") if w(name + ".b") is not None else 0.0)
    out = []
    if "kv_rank" in m:
        rank, rot, near = m["kv_rank"], m.get("rot_dim", 0), design == "zeridra"
        q = (_unit(h @ w("dq").T) * w("dq.norm")) @ w("uq").T
        source = m.get("kv_from", index)
        if source == index:
            down = h @ w("dkv").T
            kept[index] = (_unit(down[:, :rank]) * w("dkv.norm"), down[:, rank:])
        c, tail = kept[source]
        k, v = (c @ w("uk").T).view(-1, H, d), (c @ w("uv").T).view(-1, H, m["vdim"])
        for a, b in parts:
            one = q[a:b].view(-1, H, d + rot)
            keys = k[a:b]
            if rot:
                one = torch.cat([one[..., :d], _turn(one[..., d:], m["rot"], near)], -1)
                keys = torch.cat([keys, _turn(tail[a:b, None], m["rot"], near).expand(-1, H, -1)], -1)
            out.append(_mix(_maps(one, keys, scale, window=(m.get("mask") or {}).get("size"), sink=w("sink")), v[a:b]))
        o = torch.cat(out)
        if design == "bokulorn":
            gate = torch.sigmoid(h @ w("g").T)
            o = o * gate.repeat_interleave(m["vdim"], 1) if rot else o * gate
        return o @ w("o").T
    maps_of = 2 if "diff" in m else 1
    q = linear("q")
    source = m.get("kv_from", index)
    if source == index:
        k = linear("k")
        kept[index] = [k, k if design == "zeridra" else linear("v")]
    k, v = kept[source]
    v = v.view(-1, m["kv_heads"], m["vdim"])
    if "keep_first" in (m.get("mask") or {}):
        q, k = _unit(q) * w("q.norm"), _unit(k) * w("k.norm")
    q, k = q.view(-1, H * maps_of, d), k.view(-1, m["kv_heads"] * maps_of, d)
    if design == "gafonex":
        q, k, v = _unit(q) * w("q.norm"), _unit(k) * w("k.norm"), _unit(v)
        if "first" in kept:
            v = (1 - w("vmix")) * v + w("vmix") * kept["first"]
        kept.setdefault("first", v)
    for a, b in parts:
        one, keys, mask = _turn(q[a:b], m.get("rot")), _turn(k[a:b], m.get("rot")), m.get("mask") or {}
        if design == "napadra":
            slopes = torch.tensor([2.0 ** (-8.0 * (i + 1) / H) for i in range(H)], dtype=torch.float64, device=DEVICE)
            maps = _maps(one, keys, scale, chunk=mask["size"], slopes=slopes, sink=w("sink"))
        elif design == "zeridra":
            turns = torch.div(torch.arange(1, b - a + 1, device=DEVICE), m["q_temp"]["every"], rounding_mode="floor")
            one = one * (1 + m["q_temp"]["coef"] * torch.log(turns.double() + 1))[:, None, None]
            maps = _maps(one, keys, scale, sink=torch.zeros(H, dtype=torch.float64, device=DEVICE))
        elif maps_of == 2:
            lam = torch.exp((w("lq1") * w("lk1")).sum()) - torch.exp((w("lq2") * w("lk2")).sum()) + m["diff"]
            first = _maps(one[:, 0::2], keys[:, 0::2], scale, window=mask["size"])
            maps = first - lam * _maps(one[:, 1::2], keys[:, 1::2], scale, window=mask["size"])
        else:
            maps = _maps(one, keys, scale, window=mask.get("size"), keep_first=mask.get("keep_first", 0),
                         cap=m.get("softcap"), sink=w("sink"))
        if design == "gafonex":
            maps = torch.matmul(w("talk"), maps.flatten(1)).view_as(maps)
        o = _mix(maps, v[a:b])
        if maps_of == 2:
            o = (_unit(o.view(-1, H, m["vdim"])) * (1 - m["diff"])).flatten(1)
        out.append(o)
    o = torch.cat(out)
    if "keep_first" in (m.get("mask") or {}):
        o = o * torch.sigmoid(h @ w("g").T).repeat_interleave(m["vdim"], 1)
    return o @ w("o").T


def _recurrence(kind, h, m, w, parts):
    """A mixer with a state: matrix memory, retention, delta rule or selective scan, from an empty state per sequence."""
    out, n = [], h.shape[0]
    if kind in ("mlstm", "retention"):
        # The state enters a token's read linearly, so a sequence's reads are one lower triangular product.
        H, d = m["heads"], m["dim"]
        q, k, v = (h @ w("q").T).view(n, H, d), (h @ w("k").T).view(n, H, d), (h @ w("v").T).view(n, H, m["vdim"])
        for a, b in parts:
            t = torch.arange(b - a, device=DEVICE)
            later = (t[:, None] >= t[None]).expand(H, -1, -1)
            if kind == "retention":
                one, keys = _turn(q[a:b], m.get("rot")), _turn(k[a:b], m.get("rot"))
                log = (t[:, None] - t[None]) * torch.log(torch.tensor(m["decay"], dtype=torch.float64, device=DEVICE))[:, None, None]
                weights, least = torch.where(later, torch.exp(log), 0.0), None
            else:
                one, keys, cap = q[a:b], k[a:b], m["gate_cap"]
                take = cap * torch.tanh((h[a:b] @ w("i").T + w("i.b")) / cap)
                keep = torch.nn.functional.logsigmoid(cap * torch.tanh((h[a:b] @ w("f").T + w("f.b")) / cap)).cumsum(0)
                log = torch.where(later, (keep[:, None] - keep[None] + take[None]).permute(2, 0, 1), -math.inf)
                top = torch.maximum(log.amax(-1), keep.T)
                weights, least = torch.exp(log - top[..., None]), torch.exp(-top)
            scores = torch.matmul(one.transpose(0, 1), keys.permute(1, 2, 0).contiguous()) * weights * d ** -0.5
            read = torch.matmul(scores, v[a:b].transpose(0, 1).contiguous())
            if least is not None:
                read = read / (torch.maximum(scores.sum(-1).abs(), least) + 1e-6)[..., None]
            out.append(_unit(read).transpose(0, 1).flatten(1))
        o, gate = torch.cat(out), h @ w("g").T
        o = o * _silu(gate) if kind == "retention" else o * w("norm") * torch.sigmoid(gate)
        return o @ w("o").T
    if kind == "channel_delta":
        H, G, d, dv = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v, beta = h @ w("q").T, h @ w("k").T, h @ w("v").T, torch.sigmoid(h @ w("b").T)
        step = torch.nn.functional.softplus((h @ w("a1").T) @ w("a2").T + w("dt_bias"), threshold=30.0).view(n, H, d)
        decay = torch.exp(-torch.exp(w("A_log"))[None, :, None] * step)
        for a, b in parts:
            one, keys = (_silu(_taps(x[a:b], w(c))).view(-1, G, d) for x, c in ((q, "q.conv"), (k, "k.conv")))
            one, keys = (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6) for x in (one, keys))
            one, keys = (x.repeat_interleave(H // G, 1) for x in (one * d ** -0.5, keys))
            value, state = _silu(_taps(v[a:b], w("v.conv"))).view(-1, H, dv), torch.zeros(H, d, dv, dtype=torch.float64, device=DEVICE)
            for t in range(b - a):
                state = state * decay[a + t][..., None]
                u = beta[a + t][:, None] * (value[t] - (state * keys[t][..., None]).sum(1))
                state = state + keys[t][..., None] * u[:, None]
                out.append((state * one[t][..., None]).sum(1))
        o = (_unit(torch.stack(out)) * w("norm")).flatten(1)
        return (o * torch.sigmoid((h @ w("g1").T) @ w("g2").T)) @ w("o").T
    both, rank, states = h @ w("in").T, m["dt_rank"], m["state"]
    A = -torch.exp(w("A_log"))
    for a, b in parts:
        x = _silu(_taps(both[a:b, :m["inner"]], w("conv"), w("conv.b")))
        low = x @ w("x").T
        step = torch.nn.functional.softplus(low[:, :rank] @ w("dt").T + w("dt.b"), threshold=30.0)
        B, C = low[:, rank:rank + states], low[:, rank + states:]
        state = torch.zeros(m["inner"], states, dtype=torch.float64, device=DEVICE)
        for t in range(b - a):
            state = torch.exp(step[t][:, None] * A) * state + (step[t] * x[t])[:, None] * B[t]
            out.append(state @ C[t] + w("D") * x[t])
    return (torch.stack(out) * _silu(both[:, m["inner"]:])) @ w("o").T


def _experts(design, h, mlp, w):
    """Every row through its chosen experts (and the one all rows use)."""
    r, logits = mlp["router"], h @ w("router").T
    E, top, groups = r["experts"], r["top"], r.get("groups")
    if design == "dolidra":
        best = torch.topk(logits, top, -1)
        chosen, weights = best.indices, torch.softmax(best.values, -1)
    else:
        s = torch.softmax(logits, -1) if design == "zomavik" else torch.sigmoid(logits)
        choice = logits if design == "zeridra" else s + w("correction") if design == "bokulorn" else s
        if groups:
            apart = choice.view(-1, groups["count"], E // groups["count"])
            worth = apart.amax(-1) if design == "zomavik" else torch.topk(apart, min(2, apart.shape[-1]), -1).values.sum(-1)
            kept = torch.zeros_like(worth, dtype=torch.bool).scatter_(1, torch.topk(worth, groups["keep"], -1).indices, True)
            choice = apart.masked_fill(~kept[..., None], -math.inf).view(-1, E)
        chosen = torch.topk(choice, top, -1).indices
        weights = torch.gather(s, 1, chosen)
        if design != "zeridra":
            weights = weights / (weights.sum(-1, keepdim=True) + 1e-20)

    def expert(x, name):
        if design == "bokulorn":
            return (torch.relu(x @ w(name + ".up").T) ** 2) @ w(name + ".down").T
        return (_silu(x @ w(name + ".gate").T) * (x @ w(name + ".up").T)) @ w(name + ".down").T

    out = torch.zeros_like(h)
    for e in range(E):
        row, pick = (chosen == e).nonzero(as_tuple=True)
        if row.numel():
            a = weights[row, pick][:, None]
            out.index_add_(0, row, expert(a * h[row], f"e{e}") if design == "zeridra" else a * expert(h[row], f"e{e}"))
    if "shared" in mlp:
        gate = torch.sigmoid(h @ w("shared.sg").T) if design == "zomavik" else 1.0
        out += gate * expert(h, "shared")
    return out


def _qwen2_names(name):
    """A Qwen2 file's names under the ones used here."""
    table = {"embed": "model.embed_tokens.weight", "final.norm": "model.norm.weight", "head": "lm_head.weight"}
    if name in table:
        return table[name]
    layer, _, rest = name.partition(".")
    inside = {"norm1": "input_layernorm.weight", "norm2": "post_attention_layernorm.weight",
              **{f"mix.{c}": f"self_attn.{c}_proj.weight" for c in "qkvo"}, **{f"mix.{c}.b": f"self_attn.{c}_proj.bias" for c in "qkvo"},
              **{f"mlp.{c}": f"mlp.{c}_proj.weight" for c in ("gate", "up", "down")}}
    return f"model.layers.{layer[1:]}.{inside[rest]}" if rest in inside else name


def exact(case: dict, seed: int):
    """Whole sequences, layer by layer, in float64; the rows of all requests stand one after the other."""
    design, cfg, tensors = case["design"], _config(case), _weights(case, seed)
    histories, news, tokens = _histories(case), _news(case), _tokens(case, seed)
    s = SIZES[case["size"]]
    if design == "qwen2":
        tensors = {name: tensors[_qwen2_names(name)] for name in
                   [f"l{i}.{n}" for i in range(case["layers"]) for n in
                    ("norm1", "norm2", "mix.q", "mix.k", "mix.v", "mix.o", "mix.q.b", "mix.k.b", "mix.v.b", "mlp.gate", "mlp.up", "mlp.down")]
                   + ["embed", "final.norm"] + ([] if s["tied"] else ["head"])}
        d = s["width"] // s["heads"]
        layer = {"type": "attention", "mlp": {"kind": "dense", "ff": s["inner"]},
                 "mixer": {"heads": s["heads"], "kv_heads": s["kv"], "dim": d, "vdim": d, "scale": d ** -0.5, "rot": {"dims": d, "base": 1e6}}}
        cfg = {"layers": [layer] * case["layers"], "norm": {"eps": EPS}}
    ends = np.cumsum([len(t) for t in tokens]).tolist()
    parts = list(zip([0] + ends[:-1], ends))
    ids = torch.from_numpy(np.concatenate(tokens)).to(DEVICE)
    get = lambda name: tensors[name].double() if name in tensors else None
    within = lambda prefix: lambda name: get(f"{prefix}.{name}")
    by_rows = lambda f, h: torch.cat([f(x) for x in h.split(8192)])       # the inner rows of all tokens at once are too many
    groups = cfg["norm"].get("groups", 1)
    grouped = lambda x, weight: _unit(x.view(x.shape[0], groups, -1)).flatten(1) * weight
    x = tensors["embed"][ids].double()

    def mixer(index, h, layer):
        m, w = layer["mixer"], within(f"l{index}.mix")
        if "left" in m:
            return (m["left_scale"] * _attention(design, h, m["left"], within(f"l{index}.mix.left"), parts, kept, index)
                    + m["right_scale"] * _recurrence("scan", h, m["right"], within(f"l{index}.mix.right"), parts))
        if layer["type"] in ("mlstm", "retention", "channel_delta"):
            return _recurrence(layer["type"], h, m, w, parts)
        return _attention(design, h, m, w, parts, kept, index)

    def feed_forward(index, h, layer):
        w, mlp = within(f"l{index}.mlp"), layer["mlp"]
        if mlp["kind"] == "moe":
            return _experts(design, h, mlp, w)
        if design == "zomavik":
            up, down = w("up"), w("down")
            return by_rows(lambda r: (torch.relu(r @ up.T) ** 2) @ down.T, h)
        gate, up, down = w("gate"), w("up"), w("down")
        if design == "napadra":
            L = mlp["limit"]

            def one(r):
                g, u = (r @ gate.T).clamp(max=L), (r @ up.T).clamp(-L, L)
                return (g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ down.T
        else:
            act = {"qwen2": _silu, "dolidra": _gelu, "gafonex": torch.relu}[design]

            def one(r):
                return (act(r @ gate.T) * (r @ up.T)) @ down.T
        return by_rows(one, h)

    kept = {}
    if design == "napadra":
        place = torch.cat([torch.arange(b - a, device=DEVICE) for a, b in parts]).double()
        angle = place[:, None] * 10000.0 ** (-2.0 * torch.arange(s["width"] // 2, device=DEVICE).double() / s["width"])
        x = x + torch.stack([angle.sin(), angle.cos()], -1).flatten(1)
        streams = [x] * cfg["streams"]

        def sublayer(index, which, f):
            hc, S = within(f"l{index}.{which}"), range(cfg["streams"])
            read, write, mix = hc("in"), hc("out"), hc("mix")
            y = f(sum(read[i] * streams[i] for i in S))
            return [sum(mix[i, t] * streams[i] for i in S) + cfg["residual_mult"] * write[t] * y for t in S]

        def shifted(index, u):
            h = _unit(u) * get(f"l{index}.norm1")
            before = torch.cat([torch.cat([torch.zeros_like(h[:1]), h[a:b - 1]]) for a, b in parts])
            return h + (before - h) * get(f"l{index}.shift")

        for i, layer in enumerate(cfg["layers"]):
            streams = sublayer(i, "hc1", lambda u: mixer(i, shifted(i, u), layer) * get(f"l{i}.ls1"))
            if layer["mlp"]:
                streams = sublayer(i, "hc2", lambda u: feed_forward(i, _unit(u) * get(f"l{i}.norm2"), layer) * get(f"l{i}.ls2"))
        x = sum(streams)
    else:
        first, started = x, False
        for i in _runs(cfg):
            layer, norm1, norm2 = cfg["layers"][i], get(f"l{i}.norm1"), get(f"l{i}.norm2")
            if design == "zomavik" and i == cfg["loop"]["start"]:
                x = torch.cat([x, first], -1) @ get("loop.in").T
            if design in ("qwen2", "dolidra"):
                behind = (lambda y, name: _unit(y) * get(f"l{i}.{name}")) if design == "dolidra" else (lambda y, name: y)
                x = x + behind(mixer(i, _unit(x) * norm1, layer), "norm1b")
                x = x + behind(feed_forward(i, _unit(x) * norm2, layer), "norm2b")
                if design == "dolidra":
                    w, dim = within(f"l{i}.side"), cfg["token_side"]["dim"]
                    e = tensors["side.embed"][ids][:, i * dim:(i + 1) * dim].double()
                    x = x + _unit((_gelu(x @ w("gate").T) * e) @ w("proj").T) * w("norm")
            elif design == "gafonex":
                x = x + grouped(mixer(i, x, layer), norm1) * get(f"l{i}.ls1")
                x = x + grouped(feed_forward(i, x, layer), norm2) * get(f"l{i}.ls2")
            else:
                h = _unit(x) * (1.0 + norm1 if design == "bokulorn" else norm1)
                g = _unit(x) * norm2 if design == "zomavik" else h
                y, z = mixer(i, h, layer), feed_forward(i, g, layer)
                x = x + (y + z if design == "bokulorn" else y * get(f"l{i}.ls1") + z * get(f"l{i}.ls2"))
    want = torch.tensor([a + hist + new - 1 + k for (a, _), hist, new in zip(parts, histories, news)
                         for k in range(case["decode"] + 1)], device=DEVICE)
    final = get("final.norm")
    x = grouped(x[want], 1.0 + final if design == "bokulorn" else final)
    del tensors["embed" if "head" in tensors else "final.norm"]
    logits = x @ (get("head") if "head" in tensors else get("embed")).T
    if cfg.get("logit_softcap"):
        logits = cfg["logit_softcap"] * torch.tanh(logits / cfg["logit_softcap"])
    rows = [r * (case["decode"] + 1) + at + count - news[r] for step in _plan(case) for r, at, count, want in step if want]
    return logits[torch.tensor(rows, device=DEVICE)]
