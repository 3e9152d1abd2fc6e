"""What this framework is used for, as measurable cases: one packed linear layer on its own, quantised decoders that chat, decode in a
batch and read prompts, and the dense designs behind the slot scheduler -- prompts, single conversations and large batches.

A case is a dict of plain values; ``prepare`` builds from a seed what a program holds before the call (random weights of real shapes,
caches, an engine), ``run`` is one pass through the public entry points, ``exact`` the same results in float64 by plain torch.
Wherever tokens feed back into a model the caller's own sampler supplies them (a scored or constrained continuation), so every pass over
the same inputs computes the same thing.
"""
from __future__ import annotations

import math

import torch
import torch.nn.functional as F

F64 = torch.float64
DEV = "cuda:0"
CALM = 0.0625                           # residual branches of pre-norm stacks start small: the routed experts' last matrices, times this
SCORED = 64                             # a scored prompt: the logits of its last places

# Layer geometries of the dense designs: the sizes of bench.py's side benchmarks.
DESIGNS = {
    "revitar": {
        "small": dict(width=1024, heads=16, kv_heads=4, dim=64, vdim=64, window=1024, experts=16, top=2, ff=512, n_layers=4),
        "a3b-like": dict(width=2048, heads=32, kv_heads=4, dim=128, vdim=128, window=4096, experts=128, top=8, ff=768, n_layers=4),
        "wide-heads": dict(width=4096, heads=32, kv_heads=8, dim=128, vdim=128, window=2048, experts=8, top=2, ff=2048, n_layers=2),
    },
    "tugolix": {
        "small": dict(width=1024, delta=dict(heads=8, kv_heads=4, dim=64, vdim=128, conv=4), gla=dict(heads=4, dim=128, vdim=256, tau=16.0),
                      latent=dict(heads=8, dim=64, vdim=64, kv_rank=256), ff=4096, moe=dict(experts=32, top=4, ff=512, groups=(8, 4)), pattern="dgls"),
        "a3b-like": dict(width=2048, delta=dict(heads=32, kv_heads=16, dim=128, vdim=128, conv=4), gla=dict(heads=8, dim=128, vdim=256, tau=16.0),
                         latent=dict(heads=16, dim=128, vdim=128, kv_rank=512), ff=8192, moe=dict(experts=128, top=8, ff=768, groups=(8, 4)),
                         pattern="dgls"),
        "recurrent": dict(width=2048, delta=dict(heads=16, kv_heads=16, dim=128, vdim=128, conv=4), gla=dict(heads=8, dim=128, vdim=256, tau=16.0),
                          latent=dict(heads=16, dim=128, vdim=128, kv_rank=512), ff=8192, moe=dict(experts=64, top=4, ff=1024, groups=(4, 2)),
                          pattern="dgdg"),
    },
    "laruzen": {
        "small": dict(width=1024, gla=dict(heads=4, dim=128, vdim=256, tau=16.0), lightning=dict(heads=8, dim=128, vdim=128),
                      left=dict(heads=16, kv_heads=4, dim=64, vdim=64, window=1024), right=dict(width=1024, blocks=8, conv=4), ff=4096,
                      moe=dict(experts=32, top=4, ff=512, shared=1024), pattern="glpg"),
        "a3b-like": dict(width=2048, gla=dict(heads=8, dim=128, vdim=256, tau=16.0), lightning=dict(heads=16, dim=128, vdim=128),
                         left=dict(heads=16, kv_heads=4, dim=128, vdim=128, window=4096), right=dict(width=2560, blocks=10, conv=4), ff=8192,
                         moe=dict(experts=128, top=8, ff=768, shared=1536), pattern="glpg"),
        "recurrent": dict(width=2048, gla=dict(heads=8, dim=128, vdim=256, tau=16.0), lightning=dict(heads=16, dim=128, vdim=128),
                          left=dict(heads=16, kv_heads=2, dim=128, vdim=128, window=2048), right=dict(width=2048, blocks=16, conv=4), ff=8192,
                          moe=dict(experts=64, top=4, ff=1024, shared=1024), pattern="lplp"),
    },
    "gibalorn": {
        "small": dict(width=1024, latent=dict(heads=8, dim=64, rot_dim=32, vdim=64, kv_rank=256, q_rank=384),
                      mamba2=dict(heads=32, vdim=64, state=128, groups=1, conv=4, norm_groups=1), attention=dict(heads=16, kv_heads=4, dim=64, rot_dims=32),
                      moe=dict(experts=32, top=4, ff=512), pattern="mlal"),
        "a3b-like": dict(width=2048, latent=dict(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, q_rank=1024),
                         mamba2=dict(heads=64, vdim=64, state=128, groups=8, conv=4, norm_groups=8), attention=dict(heads=16, kv_heads=4, dim=128, rot_dims=64),
                         moe=dict(experts=128, top=8, ff=768), pattern="mlal"),
        "looped": dict(width=2048, latent=dict(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, q_rank=768),
                       mamba2=dict(heads=64, vdim=64, state=128, groups=1, conv=4, norm_groups=1), attention=dict(heads=16, kv_heads=2, dim=128, rot_dims=128),
                       moe=dict(experts=64, top=2, ff=2048), pattern="mla", loop=(0, 2, 2)),
    },
}


def listed():
    return [
        # one decode call of one packed layer: the smallest thing a program asks for, a few microseconds
        dict(name="linear_token", kind="linear", rows=1, n=4096, k=4096, bits=4, group=128, dtype="bfloat16", bias=False),
        # a handful of rows of unequal requests through an fp16 layer with a bias, 3 bits in groups of 64
        dict(name="linear_ragged", kind="linear", rows=27, n=8192, k=3072, bits=3, group=64, dtype="float16", bias=True),
        # a conversation turn on an 8B decoder of mixed 2 / 3 / 4 bits: a short new message behind a cached prefix, then tokens one by one
        dict(name="llama_chat", kind="chat", model="8b", layers=32, mix="S22", prefix=300, new=17, steps=24),
        # 32 sequences decoded together on the same model
        dict(name="llama_batch", kind="batch", model="8b", layers=32, mix="S22", batch=32, prefix=128, steps=8),
        # a document read by a 3B decoder, all 4 bits; what it leaves in the cache is the result
        dict(name="llama_prompt", kind="prompt", model="3b", layers=28, mix="S40", tokens=3001),
        # a conversation turn on a decoder with 128 quantised experts a layer
        dict(name="moe_chat", kind="chat", model="moe", layers=6, mix="S40", prefix=64, new=450, steps=16),
        # unequal prompts arriving together: gated window attention, softmax router
        dict(name="revitar_prompts", kind="serve", design="revitar", size="a3b-like", prompts="2047,1100,333,1", steps=0),
        # prompts through the recurrent mixers with a decay per channel
        dict(name="tugolix_prompts", kind="serve", design="tugolix", size="a3b-like", prompts="1501,700,65", steps=0),
        # one short conversation on the small geometry: launches and latency
        dict(name="tugolix_chat", kind="serve", design="tugolix", size="small", prompts="19", steps=32),
        # 32 conversations at once
        dict(name="laruzen_batch", kind="serve", design="laruzen", size="a3b-like", prompts=",".join(str(8 + 5 * i) for i in range(32)), steps=16),
        # two long conversations: a document each, then decoding over it
        dict(name="gibalorn_chat", kind="serve", design="gibalorn", size="a3b-like", prompts="2000,777", steps=24),
        # one very long prompt with a looped span
        dict(name="gibalorn_prompt", kind="serve", design="gibalorn", size="looped", prompts="8192", steps=0),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "chat", "batch", "prompt", "serve", "serve", "serve", "serve"])
    if kind == "linear":
        group = rng.choice([32, 64, 128])
        n, k = _log_int(rng, 64, 16384), 128 * _log_int(rng, 2, 112)
        return dict(kind="linear", rows=_log_int(rng, 1, 4096), n=n, k=k, bits=rng.choice([2, 3, 4]), group=group,
                    dtype=rng.choice(["bfloat16", "float16"]), bias=rng.random() < 0.3)
    if kind == "chat":
        model = rng.choice(["8b", "3b", "moe"])
        return dict(kind="chat", model=model, layers=6 if model == "moe" else rng.choice([8, 28]), mix=rng.choice(["S22", "S40"]) if model != "moe" else "S40",
                    prefix=_log_int(rng, 16, 1500), new=_log_int(rng, 1, 400), steps=rng.randint(4, 24))
    if kind == "batch":
        return dict(kind="batch", model=rng.choice(["8b", "3b"]), layers=rng.choice([8, 28]), mix=rng.choice(["S22", "S40"]), batch=_log_int(rng, 2, 32),
                    prefix=_log_int(rng, 16, 240), steps=rng.randint(2, 8))
    if kind == "prompt":
        return dict(kind="prompt", model=rng.choice(["8b", "3b"]), layers=8, mix=rng.choice(["S22", "S40"]), tokens=_log_int(rng, 130, 6000))
    design = rng.choice(sorted(DESIGNS))
    size = rng.choice(sorted(DESIGNS[design]))
    form = rng.choice(["prompts", "chat", "batch"])
    if form == "prompts":
        lens, steps = [_log_int(rng, 1, 2500) for _ in range(rng.randint(1, 3))], 0
    elif form == "chat":
        lens, steps = [_log_int(rng, 4, 2000)], rng.randint(8, 32)
    else:
        lens, steps = [_log_int(rng, 1, 200) for _ in range(rng.randint(2, 32))], rng.randint(4, 16)
    return dict(kind="serve", design=design, size=size, prompts=",".join(str(v) for v in lens), steps=steps)


# ------------------------------------------------------------------------------------------------ inputs
def _quantised_config(case):
    from gbx_lm_amd import synthetic as S
    base = {"8b": S.LLAMA3_8B, "3b": S.LLAMA32_3B, "moe": S.QWEN3_30B_A3B}[case["model"]]
    return dict(base, num_hidden_layers=case["layers"])


def _quantised_model(case, seed):
    from gbx_lm_amd import synthetic as S
    return S.build_model(_quantised_config(case), S.make_strategy(case["mix"], case["layers"], 128), device=DEV, seed=seed)


def _design_config(case):
    from gbx_lm_amd import synthetic as S
    return getattr(S, case["design"] + "_config")(**DESIGNS[case["design"]][case["size"]])


def _ids(shape, vocab, seed):
    return torch.randint(0, vocab, shape, generator=torch.Generator().manual_seed(seed + 7919))


def _lens(case):
    return [int(v) for v in case["prompts"].split(",")]


def _serve_ids(case, vocab, seed):
    """(a prompt per sequence, the continuation [steps, sequences])"""
    lens = _lens(case)
    ids = _ids((sum(lens),), vocab, seed).tolist()
    prompts = [ids[sum(lens[:i]):sum(lens[:i + 1])] for i in range(len(lens))]
    return prompts, _ids((case["steps"], len(lens)), vocab, seed + 1)


def _linear_tensors(case, seed):
    """Packed words, scales, zeros, bias and activations with the distributions of quantised checkpoints."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    n, k, b, g, dt = case["n"], case["k"], case["bits"], case["group"], getattr(torch, case["dtype"])
    words = torch.randint(-2**31, 2**31, (n, k // 32 * b), device=DEV, generator=gen, dtype=torch.int64).to(torch.int32)
    top = float((1 << b) - 1)
    scales = (torch.rand((n, k // g), device=DEV, generator=gen) + 0.5) * (0.04 / top)
    zeros = -scales * top / 2.0 + torch.randn((n, k // g), device=DEV, generator=gen) * 0.1 * scales
    t = {"qweight": words, "scales": scales.to(dt), "zeros": zeros.to(dt)}
    if case["bias"]:
        t["bias"] = (torch.randn((n,), device=DEV, generator=gen) * 0.1).to(dt)
    return t, torch.randn((case["rows"], k), device=DEV, generator=gen).to(dt)


@torch.no_grad()
def prepare(case, seed):
    from gbx_lm_amd.utils import load_weights
    if case["kind"] == "linear":
        from gbx_lm_amd.models.quantized_linear_gba import QuantizedLinear
        tensors, x = _linear_tensors(case, seed)
        layer = QuantizedLinear(case["k"], case["n"], case["bias"], case["group"], case["bits"])
        load_weights(layer, tensors, device=DEV)
        return {"case": case, "layer": layer, "x": x}
    if case["kind"] == "serve":
        from gbx_lm_amd import synthetic as S
        from gbx_lm_amd.batching import BatchScheduler
        from gbx_lm_amd.models.switch_layers import DenseRoutedGLU
        cfg = _design_config(case)
        model = getattr(S, "build_" + case["design"])(cfg, device=DEV, seed=seed)
        for m in model.modules():
            if isinstance(m, DenseRoutedGLU):
                m.down.mul_(CALM)
        prompts, forced = _serve_ids(case, cfg["vocab"], seed)
        places = [list(range(max(len(p) - SCORED, 0), len(p))) for p in prompts]
        return {"case": case, "engine": BatchScheduler(model), "prompts": prompts, "places": places, "forced": forced.to(DEV)}
    from gbx_lm_amd.models.cache import make_prompt_cache
    model = _quantised_model(case, seed)
    vocab = _quantised_config(case)["vocab_size"]
    if case["kind"] == "prompt":
        return {"case": case, "model": model, "tokens": _ids((1, case["tokens"]), vocab, seed).to(DEV)}
    cache = make_prompt_cache(model)
    rows = case["batch"] if case["kind"] == "batch" else 1
    prefix = _ids((rows, case["prefix"]), vocab, seed).to(DEV)
    model.prefill(prefix, cache) if hasattr(model, "prefill") else model(prefix, cache=cache)
    forced = _ids((case["steps"] + 1, rows), vocab, seed + 1).to(DEV)
    state = {"case": case, "model": model, "cache": cache, "forced": forced}
    if case["kind"] == "batch":
        from gbx_lm_amd.decode import DecodeRunner
        state["runner"] = DecodeRunner(model, cache)
    else:
        state["new"] = _ids((case["new"],), vocab, seed + 2).to(DEV)
    return state


@torch.no_grad()
def run(state):
    case = state["case"]
    if case["kind"] == "linear":
        return state["layer"](state["x"])
    if case["kind"] == "serve":
        engine, logprobs = state["engine"], []
        if case["steps"] == 0:                                     # prompts to be scored: logits of the places the caller asks for
            logits = engine.step(list(enumerate(state["prompts"])), state["places"])
            for i in range(len(state["prompts"])):
                engine.release(i)
            return logits

        def continuation(lp):
            logprobs.append(lp)
            return state["forced"][len(logprobs) - 1]

        engine.generate(state["prompts"], max_tokens=case["steps"], sampler=continuation)
        return torch.stack(logprobs)
    from gbx_lm_amd.models.cache import make_prompt_cache
    model = state["model"]
    if case["kind"] == "prompt":
        cache = make_prompt_cache(model)
        logits = model.last_logits(state["tokens"], cache)
        return [logits] + [t for c in cache for t in c.state]
    for c in state["cache"]:                                       # back to the shared prefix: the turn before this one is forgotten
        c.trim(c.offset - case["prefix"])
    if case["kind"] == "batch":
        return [state["runner"].step(state["forced"][i]).clone() for i in range(case["steps"])]
    from gbx_lm_amd.utils import generate_step
    given = iter(range(case["steps"] + 1))
    return [lp for _, lp, _ in generate_step(state["new"], model, max_tokens=case["steps"], prompt_cache=state["cache"],
                                             sampler=lambda lp: state["forced"][next(given)])]


# ------------------------------------------------------------------------------------------------ what a pass cannot do without
def _serve_layers(case):
    """Per layer run: (dense weights, bytes of one expert's weights, experts, top, state bytes per sequence, attended bytes per cached token,
    attention flops per visible pair, recurrence flops per token, window)."""
    g, W = DESIGNS[case["design"]][case["size"]], DESIGNS[case["design"]][case["size"]]["width"]
    if case["design"] == "revitar":
        h, kv, d, dv = g["heads"], g["kv_heads"], g["dim"], g["vdim"]
        return [(W * (h * d + kv * (d + dv) + h * dv) + W * g["experts"] * 2, 3 * W * g["ff"], g["experts"], g["top"], 0, 2 * kv * (d + dv),
                 2 * h * (d + dv), 0, g["window"])] * g["n_layers"]
    out, pattern = [], g["pattern"]
    if g.get("loop"):
        a, b, n = g["loop"]
        pattern = pattern[:a] + pattern[a:b] * n + pattern[b:]
    m = g["moe"]
    for i, c in enumerate(pattern):
        state = kv = pair = rec = 0
        window = 1 << 30
        if c == "d":
            q = g["delta"]
            dense = W * (2 * q["kv_heads"] * q["dim"] + 2 * q["heads"] * q["vdim"])
            state, rec = 4 * q["heads"] * q["dim"] * q["vdim"], 7 * q["heads"] * q["dim"] * q["vdim"]
        elif c == "g" or (c == "l" and case["design"] == "laruzen"):
            q = g["gla"] if c == "g" else g["lightning"]
            dense = W * (2 * q["heads"] * q["dim"] + 3 * q["heads"] * q["vdim"])
            state, rec = 4 * q["heads"] * q["dim"] * q["vdim"], 5 * q["heads"] * q["dim"] * q["vdim"]
        elif c == "m":
            q = g["mamba2"]
            dense = W * (3 * q["heads"] * q["vdim"] + 2 * q["groups"] * q["state"])
            state, rec = 4 * q["heads"] * q["vdim"] * q["state"], 5 * q["heads"] * q["vdim"] * q["state"]
        elif c == "p":
            q, r = g["left"], g["right"]
            dense = W * (2 * q["heads"] * q["dim"] + 2 * q["kv_heads"] * q["dim"] + q["heads"] * q["dim"] + 3 * r["width"]) + 2 * r["width"] ** 2 // r["blocks"]
            kv, pair, window = 4 * q["kv_heads"] * q["dim"], 4 * q["heads"] * q["dim"], q["window"]
        elif c == "a":
            q = g["attention"]
            dense = W * (2 * q["heads"] * q["dim"] + q["kv_heads"] * q["dim"])
            kv, pair = 4 * q["kv_heads"] * q["dim"], 4 * q["heads"] * q["dim"]
        else:
            q = g["latent"]
            rot, rank = q.get("rot_dim", 0), q["kv_rank"]
            dense = W * (rank + rot + q["heads"] * q["vdim"]) + rank * q["heads"] * (q["dim"] + q["vdim"])
            dense += W * q["q_rank"] + q["q_rank"] * q["heads"] * (q["dim"] + rot) if "q_rank" in q else W * q["heads"] * q["dim"]
            kv, pair = 2 * (rank + rot), 2 * q["heads"] * (q["dim"] + rot + q["vdim"])
        routed = case["design"] == "gibalorn" or i > 0
        dense += W * m["experts"] * 2 + 3 * W * m.get("shared", 0) if routed else 3 * W * g["ff"]
        out.append((dense, (2 if case["design"] == "gibalorn" else 3) * W * m["ff"], m["experts"] if routed else 0, m["top"] if routed else 0,
                    state, kv, pair, rec, window))
    return out


def _pairs(first, count, window):
    """Visible (query, key) pairs of ``count`` queries at positions ``first`` on."""
    return sum(min(p + 1, window) for p in range(first, first + count))


def work(case):
    kind = case["kind"]
    if kind == "linear":
        r, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * k * case["bits"] / 8 + 4.0 * n * k / case["group"] + 2.0 * r * (n + k), "flops": 2.0 * r * n * k}
    if kind == "serve":                                            # the weights a step touches are read in every step: no chip memory holds them
        g, lens, vocab = DESIGNS[case["design"]][case["size"]], _lens(case), 32000
        total_b = total_f = 0.0
        steps = [[(0, n) for n in lens]] + [[(n + s, 1) for n in lens] for s in range(max(case["steps"] - 1, 0))]
        for step in steps:
            rows = sum(c for _, c in step)
            for dense, expert, experts, top, state, kv, pair, rec, window in _serve_layers(case):
                hit = experts * (1.0 - (1.0 - top / experts) ** rows) if experts else 0.0
                total_b += 2.0 * dense + 2.0 * expert * hit + len(step) * 2 * state + sum(kv * min(p + c, window) for p, c in step)
                total_f += 2.0 * rows * (dense + top * expert) + rows * rec + sum(pair * _pairs(p, c, window) for p, c in step)
            heads = len(step) if case["steps"] else sum(min(c, SCORED) for _, c in step)
            total_b += 2.0 * g["width"] * vocab + 4.0 * heads * vocab
            total_f += 2.0 * heads * g["width"] * vocab
        return {"bytes": total_b, "flops": total_f}
    cfg, L = _quantised_config(case), case["layers"]
    D, hd = cfg["hidden_size"], cfg.get("head_dim") or cfg["hidden_size"] // cfg["num_attention_heads"]
    H, G = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    attn, head = D * hd * (2 * H + 2 * G), D * cfg["vocab_size"]
    experts, top = cfg.get("num_experts", 0), cfg.get("num_experts_per_tok", 0)
    mlp = 3 * D * (cfg["moe_intermediate_size"] if experts else cfg["intermediate_size"])

    def bits(i):
        b = 4 if case["mix"] == "S40" else (4 if i in (0, L - 1) else 3 if i in (1, 2, L - 2) else 2)
        return b, (b - 1 if experts else b)

    def step(rows_at):
        rows = sum(c for _, c in rows_at)
        hit = experts * (1.0 - (1.0 - top / experts) ** rows) if experts else 1.0
        b = sum(attn * (ba / 8 + 4 / 128) + hit * mlp * (bm / 8 + 4 / 128) for ba, bm in map(bits, range(L))) + 2.0 * head
        b += L * 4 * G * hd * sum(p + c for p, c in rows_at)
        f = 2.0 * rows * L * (attn + max(top, 1) * mlp) + 2.0 * len(rows_at) * head + L * 4 * H * hd * sum(_pairs(p, c, 1 << 30) for p, c in rows_at)
        return b, f

    if kind == "prompt":
        plan = [[(0, case["tokens"])]]
    elif kind == "batch":
        plan = [[(case["prefix"] + s, 1)] * case["batch"] for s in range(case["steps"])]
    else:
        plan = [[(case["prefix"], case["new"])]] + [[(case["prefix"] + case["new"] + s, 1)] for s in range(case["steps"])]
    done = [step(p) for p in plan]
    return {"bytes": sum(b for b, _ in done), "flops": sum(f for _, f in done)}


def tolerance(case):
    """Four times the largest distance from ``exact`` that was seen over the listed cases and a hundred drawn ones.  A scored prompt is
    compared as logits and a generated continuation as log-probabilities, whose norm is mostly their common mean; two roundings of one
    router input may choose different experts, which moves that token's row by a share of an expert."""
    if case["kind"] == "linear":
        return {"rel": 0.011 if case["dtype"] == "bfloat16" else 0.0015}
    if case["kind"] == "serve":
        return {"rel": 0.016 if case["steps"] else 0.17}
    return {"rel": {"chat": 0.02, "batch": 0.15, "prompt": 0.09}[case["kind"]]}


# ------------------------------------------------------------------------------------------------ float64
def _unpack(words, k, bits):
    """uint fields of a little-endian bit stream per row: [n, k * bits / 32] int32 -> float64 [n, k]."""
    w = words.view(torch.int32).to(torch.int64) & 0xFFFFFFFF
    w = F.pad(w, (0, 1))
    at = torch.arange(k, device=w.device) * bits
    lo, hi = w[:, at // 32], w[:, at // 32 + 1]
    return (((lo | (hi << 32)) >> (at % 32)) & ((1 << bits) - 1)).to(F64)


def _dequantised(qweight, scales, zeros, bits, group):
    k = qweight.shape[1] * 32 // bits
    return _unpack(qweight, k, bits) * scales.to(F64).repeat_interleave(group, 1) + zeros.to(F64).repeat_interleave(group, 1)


def _unit(x, eps, w=None):
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return x if w is None else x * w.to(F64)


def _mm(x, w):
    return x @ w.to(F64).t()


def _turn(x, freq, pos, mult=1.0, interleaved=False):
    """x [T, heads, d]: its first 2 len(freq) channels turned by pos * freq."""
    n = freq.numel()
    a = pos[:, None].to(F64) * freq[None, :]
    c, s = (torch.cos(a) * mult)[:, None], (torch.sin(a) * mult)[:, None]
    y = x.clone()
    i, j = (slice(0, 2 * n, 2), slice(1, 2 * n, 2)) if interleaved else (slice(0, n), slice(n, 2 * n))
    u, v = x[..., i], x[..., j]
    y[..., i], y[..., j] = u * c - v * s, v * c + u * s
    return y


def _attend(q, k, v, scale, window=None, sink=None):
    """Causal attention of one sequence, q [T, H, d], k / v [T, G, .]; ``sink`` [H]: a term exp(sink) in every denominator."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty((T, H, v.shape[2]), dtype=F64, device=q.device)
    j = torch.arange(T, device=q.device)
    for h in range(H):
        for t0 in range(0, T, 2048):
            i = j[t0:t0 + 2048, None]
            s = (q[t0:t0 + 2048, h] @ k[:, h // (H // G)].t()) * scale
            s.masked_fill_((j > i) | (i - j >= window) if window else j > i, float("-inf"))
            den = torch.logsumexp(s, -1, keepdim=True)
            if sink is not None:
                den = torch.logaddexp(den, sink[h].to(F64).expand_as(den))
            out[t0:t0 + 2048, h] = torch.exp(s - den) @ v[:, h // (H // G)]
    return out


def _experts(h, idx, w, expert):
    """sum over a token's choices of w * expert(e, its row); ``expert(e, rows, weights)`` returns already weighted rows."""
    out = torch.zeros_like(h)
    for e in idx.unique().tolist():
        t, s = torch.nonzero(idx == e, as_tuple=True)
        out.index_add_(0, t, expert(e, h[t], w[t, s][:, None]))
    return out


def _scan(q, k, v, decay, beta=None):
    """S <- diag(decay) S + k u^T, out S^T q, token after token; u = v, or beta (v - S^T k) with the decayed S.  [T, H, .]"""
    S = torch.zeros((k.shape[1], k.shape[2], v.shape[2]), dtype=F64, device=q.device)
    out = torch.empty_like(v)
    for t in range(q.shape[0]):
        S = S * decay[t][..., None]
        u = v[t] if beta is None else beta[t][:, None] * (v[t] - torch.bmm(k[t][:, None], S)[:, 0])
        S = S + k[t][:, :, None] * u[:, None]
        out[t] = torch.bmm(q[t][:, None], S)[:, 0]
    return out


def _conv(x, taps, bias=None):
    n = taps.shape[1]
    return F.conv1d(F.pad(x.t()[None], (n - 1, 0)), taps.to(F64)[:, None], None if bias is None else bias.to(F64), groups=x.shape[1])[0].t()


def _silu(z):
    return z * torch.sigmoid(z)


def _split(x, *sizes):
    return torch.split(x, list(sizes), dim=-1)


def _revitar(cfg, w, ids, keep):
    eps, m = cfg["norm"]["eps"], cfg["residual_mult"]
    x = w["model.embed_tokens.weight"][ids].to(F64) * cfg["embedding"]["scale"]
    T = x.shape[0]
    i, j = torch.arange(T, device=x.device)[:, None], torch.arange(T, device=x.device)[None]
    for n, layer in enumerate(cfg["layers"]):
        p, a, r = f"model.layers.{n}.", layer["mixer"], layer["mlp"]["router"]
        H, G, d, dv = a["heads"], a["kv_heads"], a["dim"], a["vdim"]
        q, k, v = _split(_mm(x, w[p + "mixer.qkv.weight"]), H * d, G * d, G * dv)
        q, k, v = _unit(q, eps, w[p + "mixer.q_norm"]).view(T, H, d), _unit(k, eps, w[p + "mixer.k_norm"]).view(T, G, d), v.view(T, G, dv)
        mul, rate, bias = (w[p + "mixer." + s].to(F64) for s in ("dist_mul", "dist_rate", "gate_bias"))
        o = torch.empty((T, H, dv), dtype=F64, device=x.device)
        for h in range(H):
            s = a["softcap"] * torch.tanh(q[:, h] @ k[:, h // (H // G)].t() * a["scale"] / a["softcap"])
            g = torch.sigmoid(s - mul[h] * torch.log1p(rate[h] * (i - j).clamp(min=0)) + bias[h])
            o[:, h] = g.masked_fill((j > i) | (i - j >= a["mask"]["size"]), 0.0) @ v[:, h // (H // G)]
        x = x + m * _unit(_mm(o.reshape(T, -1), w[p + "mixer.o.weight"]), eps, w[p + "norm1.weight"])
        wt, idx = torch.softmax(_mm(x, w[p + "mlp.router"]), -1).topk(r["top"], -1)

        def expert(e, rows, wt):
            g, u = _mm(rows, w[p + "mlp.gate_up"][e]).chunk(2, -1)
            return wt * _mm(_silu(g) * u, w[p + "mlp.down"][e])

        x = x + m * _unit(_experts(x, idx, wt, expert), eps, w[p + "norm2.weight"])
    return _mm(_unit(x[keep], eps, w["model.norm.weight"]), w["lm_head.weight"])


def _tugolix(cfg, w, ids, keep):
    eps, streams = cfg["norm"]["eps"], cfg["streams"]
    X = w["embed"][ids].to(F64)[:, None].repeat(1, streams, 1)
    T, latent = X.shape[0], {}

    def norm(x, p):
        return F.layer_norm(x, x.shape[-1:], w[p].to(F64), w[p + ".b"].to(F64), eps)

    def mixer(h, i, p, m, kind):
        H, d, dv = m["heads"], m["dim"], m["vdim"]
        if kind == "gla":
            q, k, v = (_mm(h, w[p + s]).view(T, H, -1) for s in "qkv")
            z = _mm(_mm(h, w[p + "a1"]), w[p + "a2"]) + w[p + "a2.b"].to(F64)
            o = _scan(q * d ** -0.5, k, v, (torch.sigmoid(z) ** (1.0 / m["tau"])).view(T, H, d))
            return _mm(_unit(o, eps, w[p + "norm"]).reshape(T, -1) * _silu(_mm(h, w[p + "g"])), w[p + "o"])
        if kind == "channel_delta":
            q, k, v = (_silu(_conv(_mm(h, w[p + s]), w[p + s + ".conv"])) for s in "qkv")
            rep = H // m["kv_heads"]
            q, k = (t.reshape(T, -1, d) for t in (q, k))
            q, k = (t * torch.rsqrt(t.square().sum(-1, keepdim=True) + 1e-6) for t in (q, k))
            a = _mm(_mm(h, w[p + "a1"]), w[p + "a2"]) + w[p + "dt_bias"].to(F64)
            decay = torch.exp(-torch.exp(w[p + "A_log"].to(F64))[:, None] * F.softplus(a, threshold=40).view(T, H, d))
            o = _scan((q * d ** -0.5).repeat_interleave(rep, 1), k.repeat_interleave(rep, 1), v.reshape(T, H, dv), decay, torch.sigmoid(_mm(h, w[p + "b"])))
            gate = torch.sigmoid(_mm(_mm(h, w[p + "g1"]), w[p + "g2"]))
            return _mm(_unit(o, eps, w[p + "norm"]).reshape(T, -1) * gate, w[p + "o"])
        if "kv_from" not in m:
            latent[i] = _unit(_mm(h, w[p + "dkv"]), eps, w[p + "dkv.norm"])
        c = latent[m.get("kv_from", i)]
        q, k, v = _mm(h, w[p + "q"]).view(T, H, d), _mm(c, w[p + "uk"]).view(T, H, d), _mm(c, w[p + "uv"]).view(T, H, dv)
        return _mm(_attend(q, k, v, m["scale"]).reshape(T, -1), w[p + "o"])

    def ff(h, p, spec):
        if spec["kind"] == "dense":
            g, u = (_mm(h, w[p + s]) + w[p + s + ".b"].to(F64) for s in ("gate", "up"))
            return _mm(_silu(g) * u, w[p + "down"]) + w[p + "down.b"].to(F64)
        r, limit = spec["router"], spec["expert"]["limit"]
        s = torch.sigmoid(_mm(h, w[p + "router"]))
        per = (s + w[p + "correction"].to(F64)).view(T, r["groups"]["count"], -1)
        best = per.topk(2, -1).values.sum(-1).topk(r["groups"]["keep"], -1).indices
        shown = torch.zeros(per.shape[:2], dtype=torch.bool, device=h.device).scatter_(1, best, True)
        idx = per.masked_fill(~shown[..., None], float("-inf")).view(T, -1).topk(r["top"], -1).indices
        wt = s.gather(1, idx)

        def expert(e, rows, wt):
            g, u = _mm(rows, w[f"{p}e{e}.gate"]).clamp(max=limit), _mm(rows, w[f"{p}e{e}.up"]).clamp(-limit, limit)
            return wt * _mm(g * torch.sigmoid(1.702 * g) * (u + 1.0), w[f"{p}e{e}.down"])

        return _experts(h, idx, wt / (wt.sum(-1, keepdim=True) + 1e-20) * r["scale"], expert)

    for i, layer in enumerate(cfg["layers"]):
        for q, fn in ((1, lambda h: mixer(h, i, f"l{i}.mix.", layer["mixer"], layer["type"])), (2, lambda h: ff(h, f"l{i}.mlp.", layer["mlp"]))):
            a, b, M = (w[f"l{i}.hc{q}.{s}"].to(F64) for s in ("in", "out", "mix"))
            y = fn(norm((a[:, None] * X).sum(1), f"l{i}.norm{q}"))
            X = (M.t() @ X) + b[:, None] * y[:, None]
    return _mm(norm(X.sum(1)[keep], "final.norm"), w["head"]) * cfg["logit_scale"]


def _laruzen(cfg, w, ids, keep):
    eps, pair = cfg["norm"]["eps"], cfg["embedding"]["bigram"]
    x = w["embed"][ids].to(F64)
    T = x.shape[0]
    pos = torch.arange(T, device=x.device)
    rows = torch.full_like(ids, pair["buckets"])
    rows[1:] = (ids[:-1] * pair["mul_prev"] + ids[1:] * pair["mul_cur"]) % pair["buckets"]
    x = x + w["bigram"][rows].to(F64)

    def norm(v, g):
        return _unit(v, eps) * (1.0 + w[g].to(F64))

    def glu(h, p, act):
        return _mm(act(_mm(h, w[p + "gate"])) * _mm(h, w[p + "up"]), w[p + "down"])

    def window_attention(h, p, m):
        H, G, d, dv, rot = m["heads"], m["kv_heads"], m["dim"], m["vdim"], m["rot"]
        q, k, v = ((_mm(h, w[p + s]) + w[p + s + ".b"].to(F64)).view(T, n, -1) for s, n in (("q", H), ("k", G), ("v", G)))
        sc, dims, base = rot["scaling"], rot["dims"], rot["base"]
        f = base ** (-2.0 * torch.arange(dims // 2, dtype=F64, device=x.device) / dims)
        lo, hi = (dims * math.log(sc["original"] / (2.0 * math.pi * sc[s])) / (2.0 * math.log(base)) for s in ("fast", "slow"))
        lo, hi = max(math.floor(lo), 0), min(math.ceil(hi), dims - 1)
        ramp = ((torch.arange(dims // 2, dtype=F64, device=x.device) - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
        f, mult = f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
        q, k = (_turn(_unit(t, eps, w[p + s]), f, pos, mult) for t, s in ((q, "q.norm"), (k, "k.norm")))
        o = _attend(q, k, _unit(v, eps), m["scale"], m["mask"]["size"], w[p + "sink"])
        return _mm(o.reshape(T, -1) * torch.sigmoid(_mm(h, w[p + "g"])), w[p + "o"]) + w[p + "o.b"].to(F64)

    def recurrent_unit(h, p, m):
        nb = m["blocks"]
        y = F.gelu(_mm(h, w[p + "y"]) + w[p + "y.b"].to(F64), approximate="tanh")
        u = _conv(_mm(h, w[p + "x"]) + w[p + "x.b"].to(F64), w[p + "conv"], w[p + "conv.b"])
        ub = u.view(T, nb, -1).transpose(0, 1).contiguous()
        r, i = (torch.sigmoid(torch.bmm(ub, w[p + s].to(F64).transpose(1, 2).contiguous()).transpose(0, 1) + w[p + s + ".b"].to(F64)).reshape(T, -1)
                for s in ("ra", "ri"))
        a = torch.exp(-8.0 * r * F.softplus(w[p + "lam"].to(F64), threshold=40))
        b = torch.sqrt(1.0 - a * a) * i * u
        S, out = torch.zeros_like(u[0]), torch.empty_like(u)
        for t in range(T):
            S = a[t] * S + b[t]
            out[t] = S
        return _mm(out * y, w[p + "o"])

    for n, layer in enumerate(cfg["layers"]):
        p, m, kind = f"l{n}.mix.", layer["mixer"], layer["type"]
        h = norm(x, f"l{n}.norm1")
        h = h + (F.pad(h, (0, 0, 1, 0))[:-1] - h) * w[f"l{n}.shift"].to(F64)
        if kind == "parallel":
            left, right = window_attention(h, p + "left.", m["left"]), recurrent_unit(h, p + "right.", m["right"])
            y = 0.5 * (_unit(left, eps, w[p + "left.out"]) + _unit(right, eps, w[p + "right.out"]))
        else:
            H, d = m["heads"], m["dim"]
            q, k, v = (_mm(h, w[p + s]).view(T, H, -1) for s in "qkv")
            gate = _mm(h, w[p + "g"])
            if kind == "gla":
                z = _mm(_mm(h, w[p + "a1"]), w[p + "a2"]) + w[p + "a2.b"].to(F64)
                o = _scan(q * d ** -0.5, k, v, (torch.sigmoid(z) ** (1.0 / m["tau"])).view(T, H, d))
                o = _unit(o, eps, w[p + "norm"]).reshape(T, -1) * _silu(gate)
            else:
                decay = torch.tensor(m["decay"], dtype=F64, device=x.device)[None, :, None].expand(T, H, d)
                o = _unit(_scan(_silu(q), _silu(k), _silu(v), decay).reshape(T, -1), eps, w[p + "norm"]) * torch.sigmoid(gate)
            y = _mm(o, w[p + "o"])
        x = x + norm(y, f"l{n}.norm1b")
        h, p, ff = norm(x, f"l{n}.norm2"), f"l{n}.mlp.", layer["mlp"]
        if ff["kind"] == "dense":
            z = glu(h, p, lambda t: F.gelu(t, approximate="tanh"))
        else:
            logits, idx = _mm(h, w[p + "router"]).topk(ff["router"]["top"], -1)
            z = _experts(h, idx, torch.softmax(logits, -1), lambda e, rows, wt: wt * glu(rows, f"{p}e{e}.", _silu)) + glu(h, p + "shared.", _silu)
        x = x + norm(z, f"l{n}.norm2b")
    return _mm(norm(x[keep], "final.norm"), w["head"])


def _gibalorn(cfg, w, ids, keep):
    eps, e0 = cfg["norm"]["eps"], w["embed"][ids].to(F64)
    x, T = e0, e0.shape[0]
    pos = torch.arange(T, device=x.device)

    def freq(rot):
        return rot["base"] ** (-2.0 * torch.arange(rot["dims"] // 2, dtype=F64, device=x.device) / rot["dims"])

    def latent(h, p, m):
        H, d, r, dv, rank = m["heads"], m["dim"], m["rot_dim"], m["vdim"], m["kv_rank"]
        q = _mm(_unit(_mm(h, w[p + "dq"]), eps, w[p + "dq.norm"]), w[p + "uq"]).view(T, H, d + r)
        c, kr = _split(_mm(h, w[p + "dkv"]), rank, r)
        c, f = _unit(c, eps, w[p + "dkv.norm"]), freq(m["rot"])
        q = torch.cat([q[..., :d], _turn(q[..., d:], f, pos, interleaved=True)], -1)
        k = torch.cat([_mm(c, w[p + "uk"]).view(T, H, d), _turn(kr[:, None], f, pos, interleaved=True).expand(T, H, r)], -1)
        o = _attend(q, k, _mm(c, w[p + "uv"]).view(T, H, dv), m["scale"])
        return _mm(o.reshape(T, -1) * torch.sigmoid(_mm(h, w[p + "g"])), w[p + "o"])

    def shared(h, p, m):
        H, G, d, f = m["heads"], m["kv_heads"], m["dim"], freq(m["rot"])
        q, k = _mm(h, w[p + "q"]).view(T, H, d), _mm(h, w[p + "k"]).view(T, G, d)
        o = _attend(_turn(q, f, pos), _turn(k, f, pos), k, m["scale"], sink=torch.zeros(H, dtype=F64, device=x.device))
        return _mm(o.reshape(T, -1), w[p + "o"])

    def mamba2(h, p, m):
        H, dv, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
        inner = H * dv
        z, xbc, dt = _split(_mm(h, w[p + "in"]), inner, inner + 2 * G * N, H)
        u, B, C = _split(_silu(_conv(xbc, w[p + "conv"], w[p + "conv.b"])), inner, G * N, G * N)
        u, dt = u.reshape(T, H, dv), F.softplus(dt + w[p + "dt_bias"].to(F64), threshold=40)
        B, C = (t.reshape(T, G, N).repeat_interleave(H // G, 1) for t in (B, C))
        decay = torch.exp(-torch.exp(w[p + "A_log"].to(F64)) * dt)[..., None]
        o = _scan(C, B, dt[..., None] * u, decay) + w[p + "D"].to(F64)[:, None] * u
        y = (o.reshape(T, -1) * _silu(z)).view(T, m["norm_groups"], -1)
        return _mm(_unit(y, eps).reshape(T, -1) * w[p + "norm"].to(F64), w[p + "o"])

    n, loop = len(cfg["layers"]), cfg.get("loop")
    runs = [(i, False) for i in range(n)]
    if loop:
        a, b = loop["start"], loop["stop"]
        runs = runs[:a] + [(i, t > 0 and i == a) for t in range(loop["times"]) for i in range(a, b)] + runs[b:]
    mixers = {"latent_attention": latent, "attention": shared, "mamba2": mamba2}
    for i, again in runs:
        layer, p = cfg["layers"][i], f"l{i}.mlp."
        x = x + e0 if again else x
        x = x + mixers[layer["type"]](_unit(x, eps, w[f"l{i}.norm1"]), f"l{i}.mix.", layer["mixer"])
        h = _unit(x, eps, w[f"l{i}.norm2"])
        wt, idx = torch.sigmoid(_mm(h, w[p + "router"])).topk(layer["mlp"]["router"]["top"], -1)
        x = x + _experts(h, idx, wt, lambda e, rows, wt: _mm(_mm(wt * rows, w[f"{p}e{e}.up"]).clamp(min=0.0) ** 2, w[f"{p}e{e}.down"]))
    return _mm(_unit(x[keep], eps, w["final.norm"]), w["head"])


def _quantised_forward(cfg, w, bits, ids):
    """Token ids [B, T] -> (last hidden rows [B, T, D], (keys, values) per layer); ``bits``: of a packed matrix by its name."""
    eps, (B, T), D = cfg["rms_norm_eps"], ids.shape, cfg["hidden_size"]
    H, G = cfg["num_attention_heads"], cfg["num_key_value_heads"]
    d = cfg.get("head_dim") or D // H
    pos = torch.arange(T, device=ids.device)
    period = cfg["rope_theta"] ** (torch.arange(0, d, 2, dtype=F64, device=ids.device) / d)
    sc = cfg.get("rope_scaling")
    if sc:
        turns = sc["original_max_position_embeddings"] / (2.0 * math.pi * period)
        smooth = ((turns - sc["low_freq_factor"]) / (sc["high_freq_factor"] - sc["low_freq_factor"])).clamp(0.0, 1.0)
        period = period / ((1.0 - smooth) / sc["factor"] + smooth)
    freq = 1.0 / period

    def matrix(name, e=None):
        t = [w[f"{name}.{s}"] if e is None else w[f"{name}.{s}"][e] for s in ("qweight", "scales", "zeros")]
        return _dequantised(*t, *bits[name])

    x, caches = w["model.embed_tokens.weight"][ids].to(F64), []
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        h = _unit(x, eps, w[p + "input_layernorm.weight"])
        q, k, v = ((h @ matrix(f"{p}self_attn.{s}_proj").t()).view(B, T, n, d) for s, n in (("q", H), ("k", G), ("v", G)))
        if p + "self_attn.q_norm.weight" in w:
            q, k = _unit(q, eps, w[p + "self_attn.q_norm.weight"]), _unit(k, eps, w[p + "self_attn.k_norm.weight"])
        q, k = (torch.stack([_turn(row, freq, pos) for row in t]) for t in (q, k))
        caches.append((k.transpose(1, 2), v.transpose(1, 2)))
        o = torch.stack([_attend(q[b], k[b], v[b], d ** -0.5) for b in range(B)])
        x = x + o.reshape(B, T, H * d) @ matrix(p + "self_attn.o_proj").t()
        h = _unit(x, eps, w[p + "post_attention_layernorm.weight"])
        if cfg.get("num_experts"):
            rows, s = h.reshape(-1, D), p + "mlp.switch_mlp."
            wt, idx = torch.softmax(rows @ matrix(p + "mlp.gate").t(), -1).topk(cfg["num_experts_per_tok"], -1)
            y = _experts(rows, idx, wt / wt.sum(-1, keepdim=True), lambda e, r, wt: wt * (
                (_silu(r @ matrix(s + "gate_proj", e).t()) * (r @ matrix(s + "up_proj", e).t())) @ matrix(s + "down_proj", e).t()))
            x = x + y.view(B, T, D)
        else:
            x = x + (_silu(h @ matrix(p + "mlp.gate_proj").t()) * (h @ matrix(p + "mlp.up_proj").t())) @ matrix(p + "mlp.down_proj").t()
    return _unit(x, eps, w["model.norm.weight"]), caches


@torch.no_grad()
def exact(case, seed):
    if case["kind"] == "linear":
        t, x = _linear_tensors(case, seed)
        y = x.to(F64) @ _dequantised(t["qweight"], t["scales"], t["zeros"], case["bits"], case["group"]).t()
        return y + t["bias"].to(F64) if case["bias"] else y
    if case["kind"] == "serve":
        from gbx_lm_amd import synthetic as S
        cfg = _design_config(case)
        w = (S.build_revitar(cfg, device=DEV, seed=seed).state_dict() if case["design"] == "revitar" else
             getattr(S, case["design"] + "_checkpoint")(cfg, DEV, seed))
        for name, t in w.items():
            if name.endswith("mlp.down") and t.dim() == 3 or ".mlp.e" in name and name.endswith(".down"):
                t.mul_(CALM)
        prompts, forced = _serve_ids(case, cfg["vocab"], seed)
        forward = {"revitar": _revitar, "tugolix": _tugolix, "laruzen": _laruzen, "gibalorn": _gibalorn}[case["design"]]
        if case["steps"] == 0:
            return torch.cat([forward(cfg, w, torch.tensor(p, device=DEV), slice(max(len(p) - SCORED, 0), None)) for p in prompts])
        rows = []
        for b, prompt in enumerate(prompts):
            ids = torch.tensor(prompt + forced[:-1, b].tolist(), device=DEV)
            rows.append(torch.log_softmax(forward(cfg, w, ids, slice(len(prompt) - 1, None)), -1))
        return torch.stack(rows, 1)
    model, cfg = _quantised_model(case, seed), _quantised_config(case)
    w = dict(model.state_dict())
    bits = {n: (m.bits, m.group_size) for n, m in model.named_modules() if hasattr(m, "group_size")}
    head = w["model.embed_tokens.weight"] if cfg["tie_word_embeddings"] else w["lm_head.weight"]
    vocab = cfg["vocab_size"]
    if case["kind"] == "prompt":
        hidden, caches = _quantised_forward(cfg, w, bits, _ids((1, case["tokens"]), vocab, seed).to(DEV))
        return [_mm(hidden[:, -1], head)] + [t for kv in caches for t in kv]
    rows = case["batch"] if case["kind"] == "batch" else 1
    ids = [_ids((rows, case["prefix"]), vocab, seed)]
    forced = _ids((case["steps"] + 1, rows), vocab, seed + 1)
    if case["kind"] == "batch":
        first, ids = case["prefix"], ids + [forced[:case["steps"]].t()]
    else:
        first, ids = case["prefix"] + case["new"] - 1, ids + [_ids((case["new"],), vocab, seed + 2)[None], forced[:case["steps"] - 1].t()]
    hidden, _ = _quantised_forward(cfg, w, bits, torch.cat(ids, 1).to(DEV))
    logits = [_mm(hidden[:, first + s], head) for s in range(case["steps"])]
    return logits if case["kind"] == "batch" else [torch.log_softmax(t, -1)[0] for t in logits]
