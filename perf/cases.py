"""Performance cases of the framework: what its users have it do, by kind of call.

Kinds (sizes from bench.py, the tests and the benchmark_qwen3 defaults):

  stream         single-query streaming attention over T tokens (stream_attn)
  step           one decode step of one layer's attention block: q/k RMSNorm,
                 RoPE, K/V append, attention, commit (KVCache.append_decode)
  paged          batched GQA decode over shuffled 64-token pages (KVCache.decode)
  prefill        causal prefill attention (prefill_causal)
  append         q/k RMSNorm, RoPE and K/V append of a prompt (KVCache.append)
  mlp            the fp32 layer's MLP: RMSNorm, gate, up, SwiGLU, down, residual
                 (rms_norm, linear, swiglu, axpby)
  model_decode   one greedy step of the 28-layer decoder (Qwen3.decode_step)
  model_prefill  a prompt through the 28-layer decoder (Qwen3.prefill)

A case is a dict of plain values; `draw` gives more of the same ranges.
Outputs and workspaces are allocated once per state, as a serving loop does.
"""
from __future__ import annotations

import importlib.util
import math
import random
import sys
from pathlib import Path

import numpy as np
import torch

ROOT = Path(__file__).resolve().parents[1]
PAGE = 64
EPS = 1e-6
THETA = 1e6
# Decode cases run sessions of this many steps before the cache is rewound.
SESSION = 100


def _load_package():
    name = "streaming_attention_amd"
    if name not in sys.modules:
        pkg = ROOT / "streaming-attention_amd"
        spec = importlib.util.spec_from_file_location(name, pkg / "__init__.py", submodule_search_locations=[str(pkg)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


sa = _load_package()
DTYPE = {"f32": torch.float32, "bf16": torch.bfloat16}
KV_DTYPE = {"f32": sa.SA_DTYPE_F32, "bf16": sa.SA_DTYPE_BF16}
MODEL = sa.QWEN3_0_6B


# ---------------------------------------------------------------- cases

def listed():
    return [
        # One short context: the smallest call, all latency (the test harness's query shape).
        {"name": "stream-t1024", "kind": "stream", "T": 1024, "d": 128},
        # The headline: one query over a long context, fp32.
        {"name": "stream-t262144", "kind": "stream", "T": 262144, "d": 128},
        # Interactive generation, one layer: 128-token prompt, then 100 steps, fp32 cache.
        {"name": "step-b1-f32", "kind": "step", "B": 1, "cached": 128, "Hq": 16, "Hkv": 8, "D": 128, "kv": "f32"},
        # Batched serving, one layer: 64 sequences of very different lengths, bf16 cache.
        {"name": "paged-b64-bf16", "kind": "paged", "B": 64, "lo": 512, "hi": 32768, "Hq": 16, "Hkv": 8, "D": 128,
         "kv": "bf16"},
        # A long prompt's attention, bf16.
        {"name": "prefill-bf16-l8192", "kind": "prefill", "dtype": "bf16", "B": 1, "L": 8192, "Hq": 16, "Hkv": 8,
         "D": 128},
        # An ordinary prompt's attention at the reference's precision.
        {"name": "prefill-f32-l1024", "kind": "prefill", "dtype": "f32", "B": 1, "L": 1024, "Hq": 16, "Hkv": 8,
         "D": 128},
        # A few prompts of a length that is no multiple of any tile.
        {"name": "prefill-bf16-b3-l777", "kind": "prefill", "dtype": "bf16", "B": 3, "L": 777, "Hq": 16, "Hkv": 8,
         "D": 128},
        # A prompt's keys and values on their way into a bf16 cache.
        {"name": "append-l1024-bf16", "kind": "append", "B": 1, "S": 1024, "Hq": 16, "Hkv": 8, "D": 128, "kv": "bf16"},
        # The fp32 layer's MLP over the reference benchmark's default prompt.
        {"name": "mlp-f32-m128", "kind": "mlp", "M": 128, "H": 1024, "I": 3072},
        # One user's greedy decoding through the whole model, fp32 cache.
        {"name": "model-decode-b1-f32", "kind": "model_decode", "B": 1, "lo": 512, "hi": 512, "kv": "f32"},
        # Batched greedy decoding through the whole model, long mixed contexts, bf16 cache.
        {"name": "model-decode-b64-bf16", "kind": "model_decode", "B": 64, "lo": 512, "hi": 16384, "kv": "bf16"},
        # A prompt through the whole model, fp32 cache.
        {"name": "model-prefill-l512-f32", "kind": "model_prefill", "B": 1, "L": 512, "kv": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _heads(rng):
    """(query heads, KV heads): the Qwen3-0.6B shape most often, wider groups beside it."""
    return rng.choice([(16, 8), (16, 8), (16, 8), (32, 8), (16, 4)])


def draw(rng):
    kind = rng.choice(["stream", "step", "paged", "prefill", "append", "mlp", "model_decode", "model_prefill"])
    if kind == "stream":
        return {"kind": kind, "T": _log_int(rng, 128, 262144), "d": rng.choice([64, 128, 128])}
    if kind == "mlp":
        H, I = rng.choice([(1024, 3072), (1024, 3072), (2048, 6144)])
        return {"kind": kind, "M": _log_int(rng, 1, 1024), "H": H, "I": I}
    if kind == "model_decode":
        B, hi = _log_int(rng, 1, 64), _log_int(rng, 64, 8192)
        return {"kind": kind, "B": B, "lo": max(16, hi // 16), "hi": hi, "kv": rng.choice(["f32", "bf16"])}
    if kind == "model_prefill":
        L = _log_int(rng, 16, 2048)
        return {"kind": kind, "B": rng.randint(1, max(1, min(8, 2048 // L))), "L": L, "kv": rng.choice(["f32", "bf16"])}
    Hq, Hkv = _heads(rng)
    D = rng.choice([128, 128, 64])
    if kind == "step":
        return {"kind": kind, "B": _log_int(rng, 1, 16), "cached": _log_int(rng, 16, 4096), "Hq": Hq, "Hkv": Hkv,
                "D": D, "kv": rng.choice(["f32", "bf16"])}
    if kind == "paged":
        B, hi = _log_int(rng, 1, 64), _log_int(rng, 256, 32768)
        return {"kind": kind, "B": B, "lo": max(16, hi // 64), "hi": hi, "Hq": Hq, "Hkv": Hkv, "D": D,
                "kv": rng.choice(["f32", "bf16", "bf16"])}
    if kind == "prefill":
        L = _log_int(rng, 64, 8192)
        B = rng.randint(1, max(1, min(4, 8192 // L)))
        return {"kind": kind, "dtype": rng.choice(["f32", "bf16"]), "B": B, "L": L, "Hq": 16, "Hkv": min(Hkv, 8),
                "D": D}
    S = _log_int(rng, 16, 4096)
    return {"kind": "append", "B": rng.randint(1, max(1, min(8, 4096 // S))), "S": S, "Hq": Hq, "Hkv": Hkv, "D": D,
            "kv": rng.choice(["f32", "bf16"])}


def lengths(case):
    """Cached tokens of each sequence of a batch: fixed by the case."""
    r = random.Random(1000003 * case["B"] + 1009 * case["lo"] + case["hi"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["B"])]


# ---------------------------------------------------------------- inputs

def _gen(seed, tag, device="cuda"):
    return torch.Generator(device=device).manual_seed((seed * 1000003 + tag * 7919 + 17) % (1 << 62))


def _normal(seed, tag, shape, std=1.0, dtype=torch.float32, mean=0.0):
    return torch.empty(shape, dtype=dtype, device="cuda").normal_(mean, std, generator=_gen(seed, tag))


def _stream_inputs(case, seed):
    """0.5 N(0,1) with 1 % of the K rows as outliers (x8)."""
    T, d = case["T"], case["d"]
    Q = _normal(seed, 1, (d,), 0.5)
    K = _normal(seed, 2, (T, d), 0.5)
    V = _normal(seed, 3, (T, d), 0.5)
    out = torch.rand(T, device="cuda", generator=_gen(seed, 4)) < 0.01
    K[out] *= 8.0
    return Q, K, V


def _page_lists(seed, counts):
    """Shuffled pages, counts[i] of them for sequence i."""
    perm = torch.randperm(sum(counts), generator=_gen(seed, 5, "cpu")).tolist()
    lists, at = [], 0
    for n in counts:
        lists.append(perm[at:at + n])
        at += n
    return lists


def _pages_for(tokens):
    return -(-tokens // PAGE)


def _make_cache(case, seed, layers, Hkv, D, room):
    """A cache whose sequence i can hold room[i] tokens on shuffled pages."""
    counts = [_pages_for(n) for n in room]
    cache = sa.KVCache(layers, Hkv, D, len(room), max(counts), sum(counts), KV_DTYPE[case["kv"]])
    for i, pages in enumerate(_page_lists(seed, counts)):
        cache.set_pages(i, pages)
    return cache


def _pool(seed, layer, which, pages, Hkv, D, dtype):
    """Cached keys (which 0) or values (1) of one layer: normed, rotated keys and values are N(0,1)."""
    return _normal(seed, 100 + 2 * layer + which, (pages * Hkv * PAGE * D,), dtype=DTYPE[dtype])


def _pool_views(cache, layer):
    """(K, V) page pools of one layer; each view keeps the cache, whose memory it shows, alive."""
    views = sa.kv_pool_views(cache, layer)
    for view in views:
        view.owner = cache
    return views


def _fill_cache(cache, case, seed, layers, lens=None):
    for layer in range(layers):
        for which, view in enumerate(_pool_views(cache, layer)):
            if lens is None:
                view.zero_()
            else:
                view.normal_(0.0, 1.0, generator=_gen(seed, 100 + 2 * layer + which))
    for i, n in enumerate(lens or []):
        cache.set_len(i, n)


def _norm_weights(seed, tag, n):
    return _normal(seed, tag, (n,), 0.02, mean=1.0)


def _model_tensors():
    """(which, layer, shape, std, mean) of every weight of the model; layer -1: global."""
    d = MODEL
    H, I, V = d["hidden"], d["intermediate"], d["vocab"]
    nq, nk, D = d["n_q_heads"] * d["head_dim"], d["n_kv_heads"] * d["head_dim"], d["head_dim"]
    yield sa.QW_EMBED, -1, (V, H), 0.02, 0.0
    yield sa.QW_FINAL_NORM, -1, (H,), 0.02, 1.0
    yield sa.QW_LM_HEAD, -1, (V, H), 0.02, 0.0
    for layer in range(d["num_layers"]):
        yield sa.QW_IN_NORM, layer, (H,), 0.02, 1.0
        yield sa.QW_QKV, layer, (nq + 2 * nk, H), 0.02, 0.0
        yield sa.QW_Q_NORM, layer, (D,), 0.02, 1.0
        yield sa.QW_K_NORM, layer, (D,), 0.02, 1.0
        yield sa.QW_O, layer, (H, nq), 0.02, 0.0
        yield sa.QW_POST_NORM, layer, (H,), 0.02, 1.0
        yield sa.QW_GATE_UP, layer, (2 * I, H), 0.02, 0.0
        yield sa.QW_DOWN, layer, (H, I), 0.02, 0.0


NORMS = (sa.QW_FINAL_NORM, sa.QW_IN_NORM, sa.QW_Q_NORM, sa.QW_K_NORM, sa.QW_POST_NORM)


def _weight_tag(which, layer):
    return 10000 + 16 * (layer + 1) + which


def _make_model(seed, max_batch, max_pos):
    model = sa.Qwen3(max_batch, max_pos)
    for which, layer, _, std, mean in _model_tensors():
        model.tensor(which, max(layer, 0)).normal_(mean, std, generator=_gen(seed, _weight_tag(which, layer)))
    return model


def prepare(case, seed):
    kind = case["kind"]
    if kind == "stream":
        Q, K, V = _stream_inputs(case, seed)
        need = sa.lib().sa_stream_attn_ws_bytes(case["T"], case["d"])
        return {"case": case, "Q": Q, "K": K, "V": V, "scale": 1.0 / math.sqrt(case["d"]),
                "out": torch.empty_like(Q), "ws": torch.zeros(max(need, 16), dtype=torch.uint8, device="cuda")}
    if kind == "prefill":
        B, L, Hq, Hkv, D, dt = (case[n] for n in ("B", "L", "Hq", "Hkv", "D", "dtype"))
        need = sa.prefill_ws_bytes(KV_DTYPE[dt], B, Hq, Hkv, L, D)
        return {"case": case, "q": _normal(seed, 1, (B, Hq, L, D), dtype=DTYPE[dt]),
                "k": _normal(seed, 2, (B, Hkv, L, D), dtype=DTYPE[dt]),
                "v": _normal(seed, 3, (B, Hkv, L, D), dtype=DTYPE[dt]), "scale": 1.0 / math.sqrt(D),
                "out": torch.empty(B, Hq, L, D, device="cuda"),
                "ws": torch.zeros(need, dtype=torch.uint8, device="cuda") if need else None}
    if kind == "mlp":
        M, H, I = case["M"], case["H"], case["I"]
        new = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
        return {"case": case, "x": _normal(seed, 1, (M, H)), "w": _norm_weights(seed, 2, H),
                "gate": _normal(seed, 3, (I, H), 0.02), "up": _normal(seed, 4, (I, H), 0.02),
                "down": _normal(seed, 5, (H, I), 0.02), "h": new(M, H), "g": new(M, I), "u": new(M, I),
                "a": new(M, I), "d": new(M, H), "y": new(M, H)}
    if kind == "model_decode":
        B, lens = case["B"], lengths(case)
        cache = _make_cache(case, seed, MODEL["num_layers"], MODEL["n_kv_heads"], MODEL["head_dim"],
                            [n + SESSION for n in lens])
        _fill_cache(cache, case, seed, MODEL["num_layers"], lens)
        return {"case": case, "model": _make_model(seed, B, max(lens) + SESSION), "cache": cache, "lens": lens,
                "step": 0, "tokens": _tokens(seed, (SESSION, B)),
                "next": torch.empty(B, dtype=torch.int32, device="cuda"),
                "logits": torch.empty(B, MODEL["vocab"], device="cuda")}
    if kind == "model_prefill":
        B, L = case["B"], case["L"]
        cache = _make_cache(case, seed, MODEL["num_layers"], MODEL["n_kv_heads"], MODEL["head_dim"], [L] * B)
        _fill_cache(cache, case, seed, MODEL["num_layers"])
        pools = [_pool_views(cache, layer) for layer in range(MODEL["num_layers"])]
        return {"case": case, "model": _make_model(seed, B, L), "cache": cache, "tokens": _tokens(seed, (B, L)),
                "next": torch.empty(B, dtype=torch.int32, device="cuda"),
                "logits": torch.empty(B, MODEL["vocab"], device="cuda"),
                "k": [p[0] for p in pools], "v": [p[1] for p in pools]}
    # one layer over a paged cache
    B, Hq, Hkv, D = (case[n] for n in ("B", "Hq", "Hkv", "D"))
    s = {"case": case, "scale": 1.0 / math.sqrt(D), "step": 0}
    if kind == "paged":
        lens = lengths(case)
        cache = _make_cache(case, seed, 1, Hkv, D, lens)
        _fill_cache(cache, case, seed, 1, lens)
        s.update(q=_normal(seed, 1, (B, Hq, D)))
    else:
        S = case["S"] if kind == "append" else SESSION
        lens = None if kind == "append" else [case["cached"]] * B
        room = [(0 if lens is None else lens[0]) + S] * B
        cache = _make_cache(case, seed, 1, Hkv, D, room)
        _fill_cache(cache, case, seed, 1, lens)
        rows = (B, S) if kind == "append" else (S, B)
        s.update(q=_normal(seed, 1, (*rows, Hq, D)), k=_normal(seed, 2, (*rows, Hkv, D)),
                 v=_normal(seed, 3, (*rows, Hkv, D)), q_norm=_norm_weights(seed, 4, D),
                 k_norm=_norm_weights(seed, 6, D), rope=sa.rope_tables(room[0], D, THETA))
        s["k_pool"], s["v_pool"] = _pool_views(cache, 0)
    s.update(cache=cache, lens=lens)
    if kind == "append":
        s["q_out"] = torch.empty_like(s["q"])
    else:
        s["out"] = torch.empty(B, Hq, D, device="cuda")
        s["ws"] = torch.zeros(max(cache.decode_ws_bytes(B, Hq), 16), dtype=torch.uint8, device="cuda")
    return s


def _tokens(seed, shape):
    return torch.randint(0, MODEL["vocab"], shape, dtype=torch.int32, device="cuda", generator=_gen(seed, 7))


# ---------------------------------------------------------------- one pass

def _next_step(s):
    """The index of this decode step in its session; a finished session starts over from the cached prompt."""
    if s["step"] == SESSION:
        for i, n in enumerate(s["lens"]):
            s["cache"].set_len(i, n)
        s["step"] = 0
    s["step"] += 1
    return s["step"] - 1


def run(s):
    kind = s["case"]["kind"]
    if kind == "stream":
        return sa.stream_attn(s["Q"], s["K"], s["V"], 64, s["scale"], out=s["out"], ws=s["ws"])
    if kind == "prefill":
        return sa.prefill_causal(s["q"], s["k"], s["v"], s["scale"], out=s["out"], ws=s["ws"])
    if kind == "mlp":
        sa.rms_norm(s["x"], s["w"], EPS, out=s["h"])
        sa.linear(s["h"], s["gate"], out=s["g"])
        sa.linear(s["h"], s["up"], out=s["u"])
        sa.swiglu(s["g"], s["u"], out=s["a"])
        sa.linear(s["a"], s["down"], out=s["d"])
        sa.axpby(s["x"], 1.0, s["d"], 1.0, out=s["y"])
        return {"mlp": s["d"], "y": s["y"]}
    if kind == "paged":
        return s["cache"].decode(0, s["q"], s["scale"], out=s["out"], ws=s["ws"])
    if kind == "append":
        s["cache"].append(0, s["q"], s["k"], s["v"], s["q_norm"], s["k_norm"], EPS, s["rope"], q_out=s["q_out"])
        return {"q": s["q_out"], "k": s["k_pool"], "v": s["v_pool"]}
    if kind == "step":
        i = _next_step(s)
        s["cache"].append_decode(0, s["q"][i], s["k"][i], s["v"][i], s["scale"], s["q_norm"], s["k_norm"], EPS,
                                 s["rope"], out=s["out"], ws=s["ws"], commit=True)
        return {"out": s["out"], "k": s["k_pool"], "v": s["v_pool"]}
    if kind == "model_decode":
        i = _next_step(s)
        s["model"].decode_step(s["cache"], s["tokens"][i], s["next"], s["logits"])
        return {"logits": s["logits"], "next": s["next"]}
    for i in range(s["case"]["B"]):
        s["cache"].set_len(i, 0)
    s["model"].prefill(s["cache"], s["tokens"], s["next"], s["logits"])
    return {"logits": s["logits"], "next": s["next"], "k": s["k"], "v": s["v"]}


# ---------------------------------------------------------------- work and tolerance

def _model_params():
    """(weights of the layers, weights of the lm_head)."""
    per = sum(int(np.prod(shape)) for which, layer, shape, _, _ in _model_tensors() if layer >= 0)
    return per, MODEL["vocab"] * MODEL["hidden"]


def work(case):
    kind = case["kind"]
    if kind == "stream":
        T, d = case["T"], case["d"]
        return {"bytes": 8 * T * d + 8 * d, "flops": 4 * T * d}
    if kind == "mlp":
        M, H, I = case["M"], case["H"], case["I"]
        return {"bytes": 4 * (3 * H * I + 3 * M * H + H), "flops": 6 * M * H * I}
    if kind == "model_decode":
        B, tokens = case["B"], sum(lengths(case)) + case["B"]
        layers, head = _model_params()
        n, Hq, Hkv, D = (MODEL[k] for k in ("num_layers", "n_q_heads", "n_kv_heads", "head_dim"))
        elem = 2 if case["kv"] == "bf16" else 4
        return {"bytes": 2 * (layers + head) + n * tokens * 2 * Hkv * D * elem + B * (2 * MODEL["hidden"] + 4 * MODEL["vocab"]),
                "flops": 2 * B * (layers + head) + n * 4 * Hq * D * tokens}
    if kind == "model_prefill":
        B, L = case["B"], case["L"]
        layers, head = _model_params()
        n, Hq, Hkv, D = (MODEL[k] for k in ("num_layers", "n_q_heads", "n_kv_heads", "head_dim"))
        elem = 2 if case["kv"] == "bf16" else 4
        return {"bytes": 2 * (layers + head) + B * (L * (n * 2 * Hkv * D * elem + 2 * MODEL["hidden"]) + 4 * MODEL["vocab"]),
                "flops": 2 * B * L * layers + 2 * B * head + n * 2 * B * Hq * D * L * (L + 1)}
    B, Hq, Hkv, D = (case[n] for n in ("B", "Hq", "Hkv", "D"))
    if kind == "prefill":
        L, elem = case["L"], 2 if case["dtype"] == "bf16" else 4
        return {"bytes": B * L * D * ((Hq + 2 * Hkv) * elem + 4 * Hq), "flops": 2 * B * Hq * D * L * (L + 1)}
    elem = 2 if case["kv"] == "bf16" else 4
    if kind == "append":
        rows = B * case["S"]
        return {"bytes": rows * D * (8 * Hq + 2 * Hkv * (4 + elem)), "flops": rows * D * 8 * (Hq + Hkv)}
    tokens = B * (case["cached"] + 1) if kind == "step" else sum(lengths(case))
    new = B * D * 2 * Hkv * (4 + elem) if kind == "step" else 0
    return {"bytes": tokens * 2 * Hkv * D * elem + 8 * B * Hq * D + new, "flops": 4 * Hq * D * tokens}


def tolerance(case):
    """About four times the error against 64 bits that each path shows."""
    kind = case["kind"]
    if kind == "stream":
        return {"rel": 2e-6}
    if kind == "prefill":
        # bf16 probabilities are 2e-3 off 64 bits; fp32 sums 4e-7.
        return {"rel": 8e-3, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 2e-6}
    if kind == "mlp":
        return {"rel": 5e-6}
    if kind == "model_decode":
        return {"rel": 1e-5 if case["kv"] == "f32" else 2e-5}
    if kind == "model_prefill":
        # bf16 storage: an element near a rounding boundary may go either way (2^-8 of it).
        return {"rel": 1e-5} if case["kv"] == "f32" else {"rel": 4e-4, "max": 1e-2}
    if kind in ("append", "step") and case["kv"] == "bf16":
        return {"rel": 1e-4, "max": 1e-2}
    return {"rel": 1.5e-6}


# ---------------------------------------------------------------- 64 bits

def _tables64(max_pos, D):
    """RoPE tables as the framework defines them: fp32 frequencies and angles, then cos and sin."""
    half = np.arange(D // 2, dtype=np.float32) / np.float32(D)
    inv = np.float32(1.0) / np.power(np.float64(THETA), half.astype(np.float64)).astype(np.float32)
    ang = np.arange(max_pos, dtype=np.float32)[:, None] * inv[None, :].astype(np.float32)
    ang = torch.from_numpy(ang.astype(np.float64)).cuda()
    return torch.cos(ang), torch.sin(ang)


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS) * w


def _rope64(x, pos, tables):
    """x [rows, heads, D] at positions pos [rows]; rotate-half."""
    c, s = tables[0][pos][:, None, :], tables[1][pos][:, None, :]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _stored(x, kv):
    """Values as the cache keeps them."""
    return x.to(torch.float32).to(DTYPE[kv]).double()


def _attend64(q, k, v, scale):
    """q [Hq, D] over k, v [Hkv, T, D]."""
    Hq, D = q.shape
    Hkv = k.shape[0]
    s = torch.matmul(q.reshape(Hkv, Hq // Hkv, D), k.transpose(1, 2).contiguous()) * scale
    return torch.matmul(torch.softmax(s, -1), v).reshape(Hq, D)


def _causal64(q, k, v, scale):
    """One head: q, k, v [L, D], causal, in row blocks."""
    L = q.shape[0]
    out = torch.empty_like(q)
    kt = k.t().contiguous()
    for a in range(0, L, 2048):
        b = min(L, a + 2048)
        s = (q[a:b] @ kt[:, :b].contiguous()) * scale
        s.masked_fill_(torch.arange(b, device="cuda")[None, :] > torch.arange(a, b, device="cuda")[:, None], -math.inf)
        out[a:b] = torch.softmax(s, -1) @ v[:b]
    return out


def _gather64(pool, pages, n, Hkv, D):
    """Tokens 0 .. n-1 of a page list: [Hkv, n, D]."""
    rows = pool.view(-1, Hkv, PAGE, D)[torch.tensor(pages, device="cuda")]
    return rows.permute(1, 0, 2, 3).reshape(Hkv, -1, D)[:, :n].double()


def _place(pool, pages, start, rows):
    """rows [n, Hkv, D] at tokens start .. of a page list."""
    n, Hkv, D = rows.shape
    t = torch.arange(start, start + n, device="cuda")
    page = torch.tensor(pages, device="cuda")[t // PAGE]
    pool.view(-1, Hkv, PAGE, D)[page, :, t % PAGE] = rows


def _model_forward64(case, seed, x, layer_attention):
    """x [rows, hidden] through the layers; layer_attention(layer, q, k, v) -> [rows, Hq D]."""
    d = MODEL
    Hq, Hkv, D, I = d["n_q_heads"], d["n_kv_heads"], d["head_dim"], d["intermediate"]
    shapes = {(w, layer): (shape, std, mean) for w, layer, shape, std, mean in _model_tensors()}

    def weight(which, layer):
        shape, std, mean = shapes[which, layer]
        dt = torch.float32 if which in NORMS else torch.bfloat16
        return _normal(seed, _weight_tag(which, layer), (int(np.prod(shape)),), std, dt, mean).double().reshape(shape)

    def project(a, which, layer):
        return a @ weight(which, layer).t().contiguous()

    for layer in range(d["num_layers"]):
        h = _rms64(x, weight(sa.QW_IN_NORM, layer))
        qkv = project(h, sa.QW_QKV, layer).reshape(-1, Hq + 2 * Hkv, D)
        q = _rms64(qkv[:, :Hq], weight(sa.QW_Q_NORM, layer))
        k = _rms64(qkv[:, Hq:Hq + Hkv], weight(sa.QW_K_NORM, layer))
        x = x + project(layer_attention(layer, q, k, qkv[:, Hq + Hkv:]), sa.QW_O, layer)
        gu = project(_rms64(x, weight(sa.QW_POST_NORM, layer)), sa.QW_GATE_UP, layer)
        x = x + project(torch.nn.functional.silu(gu[:, :I]) * gu[:, I:], sa.QW_DOWN, layer)
    x = _rms64(x, weight(sa.QW_FINAL_NORM, -1))

    def logits(rows):
        return project(rows, sa.QW_LM_HEAD, -1)

    return x, logits


def _embed64(seed, tokens):
    w = _normal(seed, _weight_tag(sa.QW_EMBED, -1), (MODEL["vocab"] * MODEL["hidden"],), 0.02, torch.bfloat16)
    return w.view(MODEL["vocab"], MODEL["hidden"])[tokens.long()].double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "stream":
        Q, K, V = (t.double() for t in _stream_inputs(case, seed))
        return torch.softmax((K @ Q) / math.sqrt(case["d"]), 0) @ V
    if kind == "mlp":
        M, H, I = case["M"], case["H"], case["I"]
        x = _normal(seed, 1, (M, H)).double()
        h = _rms64(x, _norm_weights(seed, 2, H).double())
        gate, up = _normal(seed, 3, (I, H), 0.02).double(), _normal(seed, 4, (I, H), 0.02).double()
        down = _normal(seed, 5, (H, I), 0.02).double()
        d = (torch.nn.functional.silu(h @ gate.t()) * (h @ up.t())) @ down.t()
        return {"mlp": d, "y": x + d}
    if kind == "model_decode":
        return _exact_model_decode(case, seed)
    if kind == "model_prefill":
        return _exact_model_prefill(case, seed)
    B, Hq, Hkv, D = (case[n] for n in ("B", "Hq", "Hkv", "D"))
    scale = 1.0 / math.sqrt(D)
    if kind == "prefill":
        dt, L = DTYPE[case["dtype"]], case["L"]
        q, k, v = (_normal(seed, t, (B, h, L, D), dtype=dt) for t, h in ((1, Hq), (2, Hkv), (3, Hkv)))
        out = torch.empty(B, Hq, L, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            for h in range(Hq):
                kv = h // (Hq // Hkv)
                out[b, h] = _causal64(q[b, h].double(), k[b, kv].double(), v[b, kv].double(), scale)
        return out
    if kind == "paged":
        lens = lengths(case)
        lists = _page_lists(seed, [_pages_for(n) for n in lens])
        pages = sum(len(p) for p in lists)
        kp, vp = (_pool(seed, 0, w, pages, Hkv, D, case["kv"]) for w in (0, 1))
        q = _normal(seed, 1, (B, Hq, D)).double()
        return torch.stack([_attend64(q[i], _gather64(kp, p, n, Hkv, D), _gather64(vp, p, n, Hkv, D), scale)
                            for i, (p, n) in enumerate(zip(lists, lens))])
    start = case["cached"] if kind == "step" else 0
    S = SESSION if kind == "step" else case["S"]
    rows = (S, B) if kind == "step" else (B, S)
    lists = _page_lists(seed, [_pages_for(start + S)] * B)
    pages = sum(len(p) for p in lists)
    tables = _tables64(start + S, D)
    q, k, v = (_normal(seed, t, (*rows, h, D)).double() for t, h in ((1, Hq), (2, Hkv), (3, Hkv)))
    if kind == "step":  # the session's first step
        q, k, v = (t[0].reshape(B, 1, -1, D) for t in (q, k, v))
        kp, vp = (_pool(seed, 0, w, pages, Hkv, D, case["kv"]).double() for w in (0, 1))
    else:
        kp, vp = (torch.zeros(pages * Hkv * PAGE * D, dtype=torch.float64, device="cuda") for _ in (0, 1))
    pos = torch.arange(start, start + q.shape[1], device="cuda")
    qw, kw = _norm_weights(seed, 4, D).double(), _norm_weights(seed, 6, D).double()
    q = torch.stack([_rope64(_rms64(x, qw), pos, tables) for x in q])
    for i in range(B):
        _place(kp, lists[i], start, _stored(_rope64(_rms64(k[i], kw), pos, tables), case["kv"]))
        _place(vp, lists[i], start, _stored(v[i], case["kv"]))
    if kind == "append":
        return {"q": q, "k": kp, "v": vp}
    n = start + 1
    out = torch.stack([_attend64(q[i, 0], _gather64(kp, p, n, Hkv, D), _gather64(vp, p, n, Hkv, D), scale)
                       for i, p in enumerate(lists)])
    return {"out": out, "k": kp, "v": vp}


def _exact_model_decode(case, seed):
    B, lens = case["B"], lengths(case)
    Hq, Hkv, D = MODEL["n_q_heads"], MODEL["n_kv_heads"], MODEL["head_dim"]
    lists = _page_lists(seed, [_pages_for(n + SESSION) for n in lens])
    pages = sum(len(p) for p in lists)
    tables = _tables64(max(lens) + SESSION, D)
    pos = torch.tensor(lens, device="cuda")

    def attention(layer, q, k, v):
        kp, vp = (_pool(seed, layer, w, pages, Hkv, D, case["kv"]) for w in (0, 1))
        q, k = _rope64(q, pos, tables), _stored(_rope64(k, pos, tables), case["kv"])
        v = _stored(v, case["kv"])
        rows = []
        for i, (p, n) in enumerate(zip(lists, lens)):
            K = torch.cat([_gather64(kp, p, n, Hkv, D), k[i][:, None]], 1)
            V = torch.cat([_gather64(vp, p, n, Hkv, D), v[i][:, None]], 1)
            rows.append(_attend64(q[i], K, V, 1.0 / math.sqrt(D)).reshape(-1))
        return torch.stack(rows)

    x, logits = _model_forward64(case, seed, _embed64(seed, _tokens(seed, (SESSION, B))[0]), attention)
    return {"logits": logits(x), "next": None}


def _exact_model_prefill(case, seed):
    B, L = case["B"], case["L"]
    Hq, Hkv, D = MODEL["n_q_heads"], MODEL["n_kv_heads"], MODEL["head_dim"]
    lists = _page_lists(seed, [_pages_for(L)] * B)
    pages = sum(len(p) for p in lists)
    tables = _tables64(L, D)
    pos = torch.arange(L, device="cuda").repeat(B)
    ks, vs = [], []

    def attention(layer, q, k, v):
        q, k = _rope64(q, pos, tables), _rope64(k, pos, tables)
        kp, vp = (torch.zeros(pages * Hkv * PAGE * D, dtype=torch.float64, device="cuda") for _ in (0, 1))
        out = torch.empty(B * L, Hq, D, dtype=torch.float64, device="cuda")
        for b in range(B):
            r = slice(b * L, (b + 1) * L)
            _place(kp, lists[b], 0, _stored(k[r], case["kv"]))
            _place(vp, lists[b], 0, _stored(v[r], case["kv"]))
            for h in range(Hq):
                kv = h // (Hq // Hkv)
                out[r, h] = _causal64(q[r, h].contiguous(), k[r, kv].contiguous(), v[r, kv].contiguous(),
                                      1.0 / math.sqrt(D))
        ks.append(kp)
        vs.append(vp)
        return out.reshape(B * L, Hq * D)

    x, logits = _model_forward64(case, seed, _embed64(seed, _tokens(seed, (B, L)).reshape(-1)), attention)
    return {"logits": logits(x.reshape(B, L, -1)[:, -1]), "next": None, "k": ks, "v": vs}
