"""GPU parity of the whole-model prefill (sa_qwen3_prefill): a prompt run as
one causal forward, then single-token decode steps, against the reference's
qwen3_forward_with_cache on the same weights (prompt as one forward, then
single tokens; compiled from the reference's sources into oracle/_ref).

fp32 KV cache: logits max-abs <= 1e-4 and relative L2 <= 1e-5 at the last
prompt position and after every later token, argmax identical.  Prompts of
one to several hundred tokens cover several 64-row GEMM tiles and query
tiles of the prefill kernel; the cache contents after prefill equal what
token-by-token decode steps append.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from test_gpu_model import SHAPE_KEYS, host_weights, rel_l2

pytestmark = pytest.mark.gpu

CFG = dict(num_layers=2, hidden=128, intermediate=192, vocab=256, n_q_heads=4, n_kv_heads=2, head_dim=64,
           rms_eps=1e-6, rope_theta=1e6)


def empty_cache(sa, cfg, B, cap, kv_dtype):
    per = (cap + 63) // 64
    cache = sa.KVCache(cfg["num_layers"], cfg["n_kv_heads"], cfg["head_dim"], B, per, B * per, kv_dtype)
    for s in range(B):
        cache.set_pages(s, list(range(s * per, (s + 1) * per)))
        cache.set_len(s, 0)
    return cache


def run(sa, cfg, model, tokens, prompt, kv_dtype):
    """Prefill tokens[:, :prompt], then decode the rest one at a time; logits
    at the last prompt position and after each later token."""
    B, N = tokens.shape
    cache = empty_cache(sa, cfg, B, N + 1, kv_dtype)
    logits = torch.empty(B, cfg["vocab"], dtype=torch.float32, device="cuda")
    dev = torch.from_numpy(np.ascontiguousarray(tokens)).to("cuda")
    nxt = model.prefill(cache, dev[:, :prompt], logits=logits)
    out, toks = [logits.cpu().numpy()], [nxt.cpu().numpy()]
    assert [cache.length(s) for s in range(B)] == [prompt] * B
    for t in range(prompt, N):
        nxt = model.decode_step(cache, dev[:, t].contiguous(), logits=logits)
        out.append(logits.cpu().numpy())
        toks.append(nxt.cpu().numpy())
    return np.stack(out), np.stack(toks), cache


# head_dim 128: the prompt's attention runs on the three-term kernel, and
# prompts of 8 or more 32-query tiles take its paired key ranges (the model
# passes the workspace).
CFG128 = dict(CFG, hidden=256, head_dim=128)


@pytest.mark.parametrize("B,prompt,steps,cfg", [(1, 1, 3, CFG), (2, 7, 4, CFG), (3, 130, 3, CFG), (1, 300, 2, CFG),
                                                (2, 300, 2, CFG128), (1, 77, 2, CFG128)])
def test_prefill_then_decode_matches_reference(sa, ref, B, prompt, steps, cfg):
    max_pos = prompt + steps + 1
    model = sa.Qwen3(B, max_pos, **{k: cfg[k] for k in SHAPE_KEYS})
    model.init_random(11 + prompt, 0.1)
    w = host_weights(sa, model, cfg)
    if cfg is CFG128 and prompt >= 256:
        assert sa.prefill_ws_bytes(sa.SA_DTYPE_F32, B, cfg["n_q_heads"], cfg["n_kv_heads"], prompt, 128) > 0
    tokens = ((np.arange(B * (prompt + steps)).reshape(B, -1) * 41 + 5 * prompt) % cfg["vocab"]).astype(np.int32)
    want = ref.qwen3_forward(w, dict(cfg, max_pos=max_pos), tokens, prompt)
    got, toks, cache = run(sa, cfg, model, tokens, prompt, sa.SA_DTYPE_F32)
    cache.close()
    model.close()
    assert np.abs(got - want).max() <= 1e-4
    for t in range(got.shape[0]):
        assert rel_l2(got[t], want[t]) <= 1e-5, t
    assert (toks == want.argmax(-1)).all()


def test_prefill_cache_equals_decode_appends(sa):
    """The K/V a prefill appends (normed, rotated K; V as projected) equal what
    the same tokens appended one decode step at a time leave in the cache."""
    B, P = 2, 70
    model = sa.Qwen3(B, P + 1, **{k: CFG[k] for k in SHAPE_KEYS})
    model.init_random(3, 0.1)
    tokens = torch.from_numpy(((np.arange(B * P).reshape(B, P) * 13 + 1) % CFG["vocab"]).astype(np.int32)).cuda()
    a = empty_cache(sa, CFG, B, P, sa.SA_DTYPE_F32)
    model.prefill(a, tokens)
    b = empty_cache(sa, CFG, B, P, sa.SA_DTYPE_F32)
    for t in range(P):
        model.decode_step(b, tokens[:, t].contiguous())
    torch.cuda.synchronize()
    for layer in range(CFG["num_layers"]):
        for s in range(B):
            ka, va = a.gather(layer, s, P)
            kb, vb = b.gather(layer, s, P)
            assert (ka - kb).abs().max().item() <= 1e-4
            assert (va - vb).abs().max().item() <= 1e-4
    a.close()
    b.close()
    model.close()


def test_prefill_rejects_bad_calls(sa):
    model = sa.Qwen3(2, 16, **{k: CFG[k] for k in SHAPE_KEYS})
    model.init_random(1, 0.1)
    cache = empty_cache(sa, CFG, 2, 16, sa.SA_DTYPE_F32)
    toks = torch.zeros(2, 17, dtype=torch.int32, device="cuda")
    with pytest.raises(sa.SaError):          # longer than the RoPE table
        model.prefill(cache, toks)
    model.prefill(cache, toks[:, :4].contiguous())
    with pytest.raises(sa.SaError, match="empty"):
        model.prefill(cache, toks[:, :4].contiguous())
    bare = sa.KVCache(CFG["num_layers"], CFG["n_kv_heads"], CFG["head_dim"], 2, 1, 2, sa.SA_DTYPE_F32)
    with pytest.raises(sa.SaError, match="full") as e:   # no pages reserved
        model.prefill(bare, toks[:, :4].contiguous())
    assert e.value.status == sa.SA_EFULL and bare.length(0) == 0
    bare.close()
    cache.close()
    model.close()


# One layer of the Qwen3-0.6B shape: prompts whose rows take every tile of the
# projections (32, 64 and 128 rows, split or not), with ragged last tiles; and
# sizes that are multiples of 64 but not of a tile's 128 columns or of its
# k parts.
WIDE = dict(CFG, num_layers=1, hidden=1024, intermediate=3072, vocab=1024, n_q_heads=16, n_kv_heads=8, head_dim=128)
ODD = dict(CFG, num_layers=1, hidden=320, intermediate=608, vocab=192, n_q_heads=5, n_kv_heads=1, head_dim=64)


@pytest.mark.parametrize("B,P,cfg", [(1, 17, WIDE), (3, 43, WIDE), (1, 300, WIDE), (7, 64, WIDE), (32, 20, WIDE),
                                     (61, 16, WIDE), (64, 32, WIDE), (1, 33, ODD), (2, 131, ODD)])
def test_prefill_rows_match_float64(sa, B, P, cfg):
    """Keys, values and the last position's logits of a one-layer model in
    float64.  Bound: fp32 sums over k <= 3072 products are 5e-7 off in the
    2-norm (measured 1e-7 .. 4e-7 per projection); the logits pass six of
    them and two norms."""
    import torch.nn.functional as F
    H, I, Hq, Hkv, D = (cfg[k] for k in ("hidden", "intermediate", "n_q_heads", "n_kv_heads", "head_dim"))
    model = sa.Qwen3(B, P, **{k: cfg[k] for k in SHAPE_KEYS})
    model.init_random(5, 0.05)
    w = lambda which, layer=0: model.tensor(which, layer).double()  # noqa: E731
    tokens = ((torch.arange(B * P, device="cuda") * 37 + 11) % cfg["vocab"]).view(B, P).int()
    cache = empty_cache(sa, cfg, B, P, sa.SA_DTYPE_F32)
    logits = torch.empty(B, cfg["vocab"], device="cuda")
    nxt = model.prefill(cache, tokens, logits=logits)

    def norm(x, g):
        return x / torch.sqrt((x * x).mean(-1, keepdim=True) + cfg["rms_eps"]) * g
    x = w(sa.QW_EMBED).view(-1, H)[tokens.long()]
    qkv = norm(x, w(sa.QW_IN_NORM)) @ w(sa.QW_QKV).view(-1, H).T
    q, k, v = (t.reshape(B, P, -1, D).transpose(1, 2) for t in qkv.split([Hq * D, Hkv * D, Hkv * D], -1))
    cos, sin = (t.double() for t in sa.rope_tables(P, D, cfg["rope_theta"]))

    def rope(t):
        a, b = t[..., :D // 2], t[..., D // 2:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)
    q, k = rope(norm(q, w(sa.QW_Q_NORM))), rope(norm(k, w(sa.QW_K_NORM)))
    kk, vv = (t.repeat_interleave(Hq // Hkv, 1).contiguous() for t in (k, v))
    s = (q @ kk.transpose(-1, -2).contiguous()) / D ** 0.5
    s = s.masked_fill(torch.ones(P, P, dtype=torch.bool, device="cuda").triu(1), float("-inf"))
    attn = (s.softmax(-1) @ vv).transpose(1, 2).reshape(B, P, Hq * D)
    x = x + attn @ w(sa.QW_O).view(H, -1).T
    gate, up = (norm(x, w(sa.QW_POST_NORM)) @ w(sa.QW_GATE_UP).view(2 * I, H).T).split(I, -1)
    x = x + (F.silu(gate) * up) @ w(sa.QW_DOWN).view(H, I).T
    want = norm(x[:, -1], w(sa.QW_FINAL_NORM)) @ w(sa.QW_LM_HEAD).view(-1, H).T

    rel = lambda a, b: ((a.double() - b).norm() / b.norm()).item()  # noqa: E731
    assert rel(logits, want) <= 5e-6
    got = [cache.gather(0, i, P) for i in range(B)]
    assert rel(torch.stack([g[0] for g in got]).view_as(k), k) <= 2e-6
    assert rel(torch.stack([g[1] for g in got]).view_as(v), v) <= 2e-6
    assert (nxt.long() == logits.argmax(-1)).all()
    cache.close()
    model.close()
