"""Performance cases of the framework: what its users have it do, through its public entry points.

A case is a dict of plain values; ``kind`` names the path:

* ``model``: a whole float32 forward (``forward_batch``, float32 being the models' default type) of
  ``tokens`` positions per sequence over a full cache that holds ``ctx``, then the rollback a decode
  round ends with. Returns the logits.
* ``layer``: everything of a bf16 Llama decoder layer but its attention, as ``Decoder._core`` calls it:
  norm, qkv projection with RoPE, o projection with the residual norm, SwiGLU MLP, residual norm.
* ``attn``: one layer's K/V append and causal attention over the paged full cache; prefill
  (``ctx`` 0 or short, many rows), verify (a few rows) or decode (one row).
* ``draft``: one draft step's attention over the compressed mirror, with the attention mass an arm
  that evicts needs.
* ``resync``: the mirror follows the full cache: ``rows`` = 0 builds it (or rebuilds it under a new arm),
  ``rows`` > 0 replaces the last rows, as every decode round does.
* ``quantize``: the group quantizer on float32 rows.
* ``round``: the sampling side of a decode round: gamma draft samples and the accept decision.

The attention shapes are those of the models the framework names: Llama-3-8B, SmolLM2-135M, distilgpt2.
"""

import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "draft-kv_amd"))

from draftkv import ops  # noqa: E402
from draftkv.compress import CompressedKVCache, quantize  # noqa: E402
from draftkv.config import CompressionConfig  # noqa: E402
from draftkv.gpt2 import DISTILGPT2, GPT2  # noqa: E402
from draftkv.llama import LLAMA3_8B, SMOLLM2_135M, LlamaLike  # noqa: E402
from draftkv.paged import PagedKVCache  # noqa: E402

DEV = "cuda"
F32, BF16, F64 = torch.float32, torch.bfloat16, torch.float64
# query heads, KV heads, head width
HEADS = {"llama3_8b": (32, 8, 128), "smollm2": (9, 3, 64), "distilgpt2": (12, 12, 64)}
LLAMAS = {"llama3_8b": LLAMA3_8B, "smollm2": SMOLLM2_135M}


def listed():
    return [
        # one decode step of a small model at batch 1: the smallest forward, launches and latency count
        dict(name="decode_smollm2_f32", kind="model", model="smollm2", batch=1, tokens=1, ctx=1024),
        # a prompt through the real model of the reference's own evaluation, its whole context
        dict(name="prefill_distilgpt2_f32", kind="model", model="distilgpt2", batch=1, tokens=1000, ctx=0),
        # verify block of the served model at batch 32 with gamma 4
        dict(name="layer_verify_llama8b", kind="layer", model="llama3_8b", rows=160),
        # prefill of a 4096-token prompt
        dict(name="layer_prefill_llama8b", kind="layer", model="llama3_8b", rows=4096),
        # the same prompt's attention
        dict(name="attn_prefill_llama8b", kind="attn", model="llama3_8b", bf16=True, batch=1, tokens=4096, ctx=0),
        # the benchmark's verify pass: batch 32, ctx 32k, gamma 4
        dict(name="attn_verify_llama8b", kind="attn", model="llama3_8b", bf16=True, batch=32, tokens=5, ctx=32763),
        # verify block of the float32 default path, an odd context
        dict(name="attn_verify_smollm2_f32", kind="attn", model="smollm2", bf16=False, batch=8, tokens=5, ctx=4001),
        # the engine's default arm (4 bits, keep 0.5, 64-channel groups, float32 pairs) at batch 1
        dict(name="draft_default_smollm2", kind="draft", model="smollm2", bf16=False, batch=1, ctx=8192, bits=4,
             keep=0.5, group=64, half=False),
        # the benchmark's drafter: int4 in groups of 32 with fp16 pairs, a quarter of the rows
        dict(name="draft_int4_llama8b", kind="draft", model="llama3_8b", bf16=True, batch=32, ctx=32768, bits=4,
             keep=0.25, group=32, half=True),
        # a controller's switch to an 8-bit arm over a 16k context
        dict(name="rebuild_int8_llama8b", kind="resync", model="llama3_8b", bf16=True, batch=4, ctx=16384, layers=2,
             rows=0, bits=8, keep=1.0, group=64, half=False),
        # the round trip of one layer's keys (8 heads, 8k tokens) through the 4-bit grid
        dict(name="quantize_int4", kind="quantize", rows=65536, width=128, bits=4, group=64, half=False),
        # sampled round at batch 32 with gamma 4 over the served vocabulary
        dict(name="round_llama8b", kind="round", batch=32, gamma=4, vocab=128256, temperature=0.8),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["model", "model", "layer", "layer", "attn", "attn", "attn", "draft", "draft", "resync",
                       "quantize", "round"])
    if kind == "model":
        c = dict(kind=kind, model=rng.choice(["smollm2", "distilgpt2"]))
        most = 1000 if c["model"] == "distilgpt2" else 4000
        if rng.random() < 0.4:   # prefill
            return dict(c, batch=rng.choice([1, 1, 2]), tokens=_log(rng, 16, 350), ctx=0)
        return dict(c, batch=_log(rng, 1, 16), tokens=rng.choice([1, 1, 2, 3, 5, 9]), ctx=_log(rng, 64, most))
    if kind == "layer":
        return dict(kind=kind, model=rng.choice(["llama3_8b", "llama3_8b", "smollm2"]), rows=_log(rng, 1, 4000))
    if kind == "attn":
        model, bf16 = rng.choice([("llama3_8b", True), ("llama3_8b", True), ("smollm2", True), ("smollm2", False),
                                  ("distilgpt2", False)])
        c = dict(kind=kind, model=model, bf16=bf16)
        if rng.random() < 0.4:
            most = 4000 if bf16 else 900
            return dict(c, batch=1, tokens=_log(rng, 32, most), ctx=rng.choice([0, 0, rng.randrange(1, 500)]))
        batch = _log(rng, 1, 32)
        return dict(c, batch=batch, tokens=rng.randrange(1, 10),
                    ctx=_log(rng, 256, min(32000 if bf16 else 8000, 1000000 // batch)))
    if kind in ("draft", "resync"):
        model, bf16 = rng.choice([("llama3_8b", True), ("llama3_8b", True), ("smollm2", False), ("distilgpt2", False)])
        bits, keep = rng.choice([2, 3, 4, 8, 16]), rng.choice([0.25, 0.5, 1.0])
        group, half = rng.choice([(64, False), (64, False), (32, True)])
        c = dict(kind=kind, model=model, bf16=bf16, bits=bits, keep=keep, group=group, half=half)
        batch = _log(rng, 1, 32)
        most = 32000 if bf16 else 8000
        if kind == "draft":
            return dict(c, batch=batch, ctx=_log(rng, 256, min(most, 500000 // batch)))
        ctx = _log(rng, 256, min(most, 120000 // batch))
        return dict(c, batch=batch, ctx=ctx, layers=rng.choice([1, 2]), rows=rng.choice([0, 1, 3, 5]))
    if kind == "quantize":
        return dict(kind=kind, rows=_log(rng, 500, 60000), width=rng.choice([64, 80, 128, 128, 576]),
                    bits=rng.choice([2, 3, 4, 8]), group=rng.choice([32, 64, 64]), half=rng.random() < 0.3)
    return dict(kind=kind, batch=_log(rng, 1, 32), gamma=rng.randrange(1, 9), vocab=rng.choice([128, 49152, 50257, 128256]),
                temperature=rng.choice([0.0, 0.7, 0.8, 1.0]))


# ---------------------------------------------------------------- inputs
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, std=1.0, dtype=F32):
    return torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, std, generator=g)


def _kv(g, b, n, heads, d, dtype):
    """K and V rows [b, n, heads, d]: normal, K with the uneven channel gains that trained models show."""
    gain = torch.exp(0.4 * _normal(g, heads, d)).to(dtype)
    return _normal(g, b, n, heads, d, dtype=dtype).mul_(gain), _normal(g, b, n, heads, d, dtype=dtype)


def _dtype(case):
    return BF16 if case["bf16"] else F32


def _model_weights(case, g):
    if case["model"] == "distilgpt2":
        c = DISTILGPT2
        d, ff = c["n_embd"], 4 * c["n_embd"]
        w = {"wte.weight": _normal(g, c["vocab_size"], d, std=0.02), "wpe.weight": _normal(g, c["n_positions"], d, std=0.02),
             "ln_f.weight": 1 + _normal(g, d, std=0.1), "ln_f.bias": _normal(g, d, std=0.02)}
        for i in range(c["n_layer"]):
            for n, k, m in (("attn.c_attn", d, 3 * d), ("attn.c_proj", d, d), ("mlp.c_fc", d, ff), ("mlp.c_proj", ff, d)):
                w[f"h.{i}.{n}.weight"] = _normal(g, k, m, std=0.02)
                w[f"h.{i}.{n}.bias"] = _normal(g, m, std=0.02)
            for n in ("ln_1", "ln_2"):
                w[f"h.{i}.{n}.weight"], w[f"h.{i}.{n}.bias"] = 1 + _normal(g, d, std=0.1), _normal(g, d, std=0.02)
        return c, w
    c = LLAMAS[case["model"]]
    d, ff = c["hidden_size"], c["intermediate_size"]
    hq, hkv, dh = c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"]
    w = {"model.embed_tokens.weight": _normal(g, c["vocab_size"], d, std=0.02), "model.norm.weight": 1 + _normal(g, d, std=0.1)}
    for i in range(c["num_hidden_layers"]):
        p = f"model.layers.{i}."
        for n, o, k in (("self_attn.q_proj", hq * dh, d), ("self_attn.k_proj", hkv * dh, d), ("self_attn.v_proj", hkv * dh, d),
                        ("self_attn.o_proj", d, hq * dh), ("mlp.gate_proj", ff, d), ("mlp.up_proj", ff, d),
                        ("mlp.down_proj", d, ff)):
            w[p + n + ".weight"] = _normal(g, o, k, std=0.02)
        for n in ("input_layernorm", "post_attention_layernorm"):
            w[p + n + ".weight"] = 1 + _normal(g, d, std=0.1)
    return c, w


def _model_inputs(case, seed):
    g = _gen(seed)
    cfg, w = _model_weights(case, g)
    hq, hkv, d = HEADS[case["model"]]
    n_layers = cfg.get("n_layer") or cfg["num_hidden_layers"]
    b, ctx = case["batch"], case["ctx"]
    kv = [_kv(g, b, ctx, hkv, d, F32) for _ in range(n_layers)] if ctx else []
    tok = torch.randint(0, cfg["vocab_size"], (b, case["tokens"]), generator=g, device=DEV, dtype=torch.int32)
    return cfg, w, kv, tok


def _layer_inputs(case, seed):
    g = _gen(seed)
    c = LLAMAS[case["model"]]
    d, ff, M = c["hidden_size"], c["intermediate_size"], case["rows"]
    hq, hkv, dh = HEADS[case["model"]]
    w = {n: _normal(g, o, k, std=0.02, dtype=BF16) for n, o, k in
         (("qkv", (hq + 2 * hkv) * dh, d), ("o", d, hq * dh), ("gate", ff, d), ("up", ff, d), ("down", d, ff))}
    n1, n2, n3 = ((1 + _normal(g, d, std=0.1)).to(BF16) for _ in range(3))
    h = _normal(g, M, d)
    a = _normal(g, M, hq * dh, std=0.3)
    pos = torch.arange(M, device=DEV, dtype=torch.int32)
    inv = 1.0 / (c["rope_theta"] ** (torch.arange(0, dh, 2, device=DEV, dtype=F64) / dh))
    ang = torch.arange(M, device=DEV, dtype=F64)[:, None] * inv
    return c, w, (n1, n2, n3), h, a, pos, torch.stack([ang.cos(), ang.sin()])


def _attn_inputs(case, seed):
    g = _gen(seed)
    hq, hkv, d = HEADS[case["model"]]
    b, T = case["batch"], case["tokens"]
    k, v = _kv(g, b, case["ctx"] + T, hkv, d, _dtype(case))
    return _normal(g, b, T, hq, d), k, v


def _draft_inputs(case, seed):
    g = _gen(seed)
    hq, hkv, d = HEADS[case["model"]]
    k, v = _kv(g, case["batch"], case["ctx"], hkv, d, _dtype(case))
    return _normal(g, case["batch"], hq, d), k, v


def _round_inputs(case, seed):
    g = _gen(seed)
    b, gamma, V = case["batch"], case["gamma"], case["vocab"]
    target = _normal(g, b, gamma + 1, V, std=2.5)
    draft = target[:, :gamma].transpose(0, 1) + _normal(g, gamma, b, V, std=0.3)   # the drafter is close to the target
    u = torch.rand((gamma, b), generator=g, device=DEV, dtype=F64)
    uv = torch.rand((b, gamma + 1), generator=g, device=DEV, dtype=F64)
    return target, draft.contiguous(), u, uv


def _full_cache(kv_layers, dtype, room=0):
    """A paged full cache holding the given K/V rows, with blocks reserved for ``room`` more."""
    k0 = kv_layers[0][0]
    b, n, hkv, d = k0.shape
    blocks = -(-(n + room) // 16)
    full = PagedKVCache(len(kv_layers), hkv, d, 16, blocks * len(kv_layers), dtype, batch=b, max_tokens=blocks * 16)
    full.reserve([n + room] * b)
    zero = torch.zeros(b, dtype=torch.int32, device=DEV)
    for L, (k, v) in enumerate(kv_layers):
        full.append_layer(L, k, v, zero)
    full.commit([n] * b)
    return full


def _arm(case):
    return CompressionConfig(case["bits"], case["keep"], group=case["group"], scale_fp16=case["half"])


def prepare(case, seed):
    kind = case["kind"]
    if kind == "model":
        cfg, w, kv, tok = _model_inputs(case, seed)
        model = GPT2(w, cfg) if case["model"] == "distilgpt2" else LlamaLike(w, cfg)
        b, ctx = case["batch"], case["ctx"]
        cache = model.new_cache(batch=b, max_tokens=ctx + case["tokens"] + 16)
        if ctx:
            cache.reserve([ctx] * b)
            zero = torch.zeros(b, dtype=torch.int32, device=DEV)
            for L, (k, v) in enumerate(kv):
                cache.append_layer(L, k, v, zero)
            cache.commit([ctx] * b)
        return dict(kind=kind, model=model, cache=cache, tok=tok, start=[ctx] * b)
    if kind == "layer":
        c, w, norms, h, a, pos, cs = _layer_inputs(case, seed)
        ff, d = w["gate"].shape
        gate_up = torch.stack([w["gate"], w["up"]], 1).reshape(2 * ff, d).contiguous()   # rows (gate_i, up_i)
        tile = lambda t: ops.TiledW(t) if ops.tile_ok(t) else t   # noqa: E731  as the models hold their weights
        return dict(kind=kind, heads=HEADS[case["model"]], eps=c["rms_norm_eps"], wqkv=tile(w["qkv"]), wo=tile(w["o"]),
                    w1=tile(gate_up), w2=tile(w["down"]), norms=norms, h=h, a=a, pos=pos, cs=cs.to(F32).contiguous(),
                    rows=case["rows"])
    if kind == "attn":
        q, k, v = _attn_inputs(case, seed)
        n, T, b = case["ctx"], case["tokens"], case["batch"]
        full = _full_cache([(k, v)], _dtype(case))
        start = torch.full((b,), n, dtype=torch.int32, device=DEV)
        return dict(kind=kind, full=full, q=q, k=k[:, n:].contiguous(), v=v[:, n:].contiguous(), start=start, max_len=n + T)
    if kind == "draft":
        q, k, v = _draft_inputs(case, seed)
        full = _full_cache([(k, v)], _dtype(case))
        mirror = CompressedKVCache(1, _arm(case), batch=case["batch"], cap=case["ctx"] + 64)
        mirror.sync_from(full, 0)
        return dict(kind=kind, mirror=mirror, q=q)
    if kind == "resync":
        _, hkv, d = HEADS[case["model"]]
        g = _gen(seed)
        full = _full_cache([_kv(g, case["batch"], case["ctx"], hkv, d, _dtype(case)) for _ in range(case["layers"])],
                           _dtype(case))
        mirror = CompressedKVCache(case["layers"], _arm(case), batch=case["batch"], n_kv_heads=hkv, d_head=d,
                                   cap=case["ctx"] + 64)
        mirror.pages.zero_()   # slots that hold no row are compared too
        mirror.sync_from(full, 0)
        return dict(kind=kind, mirror=mirror, full=full, start=max(0, case["ctx"] - case["rows"]) if case["rows"] else 0)
    if kind == "quantize":
        g = _gen(seed)
        x = _normal(g, case["rows"], case["width"]).mul_(torch.exp(0.4 * _normal(g, case["width"])))
        return dict(kind=kind, x=x, bits=case["bits"], group=case["group"], half=case["half"])
    target, draft, u, uv = _round_inputs(case, seed)
    return dict(kind=kind, target=target, draft=draft, u=u, uv=uv, T=case["temperature"])


# ---------------------------------------------------------------- one pass
def run(s):
    kind = s["kind"]
    if kind == "model":
        logits = s["model"].forward_batch(s["tok"], s["cache"], s["start"])
        s["cache"].truncate(s["start"])
        return logits
    if kind == "layer":
        hq, hkv, d = s["heads"]
        n1, n2, n3 = s["norms"]
        x = ops.rmsnorm(s["h"], n1, s["eps"], BF16)
        q, k, v = ops.qkv_split(ops.gemm_bf16(x, s["wqkv"], defer=True), None, hq, hkv, d, s["pos"], s["cs"], s["rows"])
        h = s["h"].clone()
        x = ops.add_norm(h, ops.gemm_bf16(s["a"], s["wo"], defer=True), None, n2, None, s["eps"], False, BF16)
        x = ops.gemm_bf16(x, s["w1"], swiglu=True)
        x = ops.add_norm(h, ops.gemm_bf16(x, s["w2"], defer=True), None, n3, None, s["eps"], False, BF16)
        return q, k, v, h, x
    if kind == "attn":
        s["full"].append_layer(0, s["k"], s["v"], s["start"])
        return s["full"].attend(0, s["q"], s["start"], s["max_len"])
    if kind == "draft":
        out = s["mirror"].attend(0, s["q"])
        return out, s["mirror"].score
    if kind == "resync":
        m = s["mirror"]
        m.sync_from(s["full"], s["start"])
        return m.pages, m.pos, m.score, m.n_rows
    if kind == "quantize":
        return quantize(s["x"], s["bits"], s["group"], s["half"])
    gamma, b, _ = s["draft"].shape
    stats = ops.row_stats(b, DEV, (gamma,)) if s["T"] > 0 else None
    tok = torch.empty((b, gamma), dtype=torch.int32, device=DEV)
    for i in range(gamma):
        tok[:, i] = ops.sample(s["draft"][i], s["T"], s["u"][i], stats_out=None if stats is None else stats[i])
    acc, nxt, used = ops.accept(s["target"], s["draft"], tok, s["T"], s["uv"], stats)
    # a row's normaliser is its first three words (max, sum, 1 / sum); the fourth is for the greedy rule
    return (tok, acc, nxt, used) if stats is None else (tok, acc, nxt, used, stats[..., :3])


# ---------------------------------------------------------------- what a pass cannot do without
def _kept(case):
    """Rows a mirror keeps of ctx, after a build with all scores 0."""
    return min(case["ctx"], max(int(round(case["keep"] * case["ctx"])), 4 + 32))


def _mirror_row_bytes(case, d):
    if case["bits"] == 16:
        return 4.0 * d   # the copy is float32
    return d * (4 if case["bits"] <= 4 else 8) / 8.0 + (4 if case["half"] else 8) * -(-d // case["group"])


def work(case):
    kind = case["kind"]
    if kind == "quantize":
        n = case["rows"] * case["width"]
        return dict(bytes=8.0 * n, flops=4.0 * n)
    if kind == "round":
        b, g, V = case["batch"], case["gamma"], case["vocab"]
        return dict(bytes=4.0 * b * (2 * g + 1) * V, flops=4.0 * b * (2 * g + 1) * V)
    hq, hkv, d = HEADS[case["model"]]
    if kind == "layer":
        c, M = LLAMAS[case["model"]], case["rows"]
        dm, ff = c["hidden_size"], c["intermediate_size"]
        n = dm * (hq + 2 * hkv) * d + hq * d * dm + 3 * dm * ff
        io = M * (4 * dm + 4 * hq * d + 4 * (hq + 2 * hkv) * d + 4 * dm + 2 * dm)
        return dict(bytes=2.0 * n + io, flops=2.0 * n * M)
    b = case["batch"]
    if kind == "resync":
        rows = case["rows"] or _kept(case)
        e = 2 if case["bf16"] else 4
        return dict(bytes=2.0 * case["layers"] * b * hkv * rows * (d * e + _mirror_row_bytes(case, d)),
                    flops=8.0 * case["layers"] * b * hkv * rows * d)
    if kind == "draft":
        kept = _kept(case)
        mass = 16.0 * b * kept if case["keep"] < 1 else 0.0
        return dict(bytes=2.0 * b * hkv * kept * _mirror_row_bytes(case, d) + 8.0 * b * hq * d + mass,
                    flops=4.0 * b * hq * kept * d)
    T, ctx = case["tokens"], case["ctx"]
    e = 2.0 if kind == "attn" and case["bf16"] else 4.0
    keys = T * ctx + T * (T + 1) / 2   # (query, key) pairs of a sequence
    kv_bytes = 2.0 * b * (ctx + T) * hkv * d * e
    att = 4.0 * b * hq * d * keys
    if kind == "attn":
        return dict(bytes=kv_bytes + 8.0 * b * T * hq * d + 2.0 * b * T * hkv * d * e, flops=att)
    if case["model"] == "distilgpt2":
        n_layers, V, dm = DISTILGPT2["n_layer"], DISTILGPT2["vocab_size"], DISTILGPT2["n_embd"]
        n = n_layers * 12 * dm * dm + V * dm
    else:
        c = LLAMAS[case["model"]]
        n_layers, V, dm = c["num_hidden_layers"], c["vocab_size"], c["hidden_size"]
        n = n_layers * (dm * (hq + 2 * hkv) * d + hq * d * dm + 3 * dm * c["intermediate_size"]) + V * dm
    R = b * T
    return dict(bytes=4.0 * n + n_layers * kv_bytes + 4.0 * R * V, flops=2.0 * n * R + n_layers * att)


def tolerance(case):
    kind = case["kind"]
    if kind in ("quantize", "resync"):
        return "exact"      # codes, pairs and positions are defined to the bit
    if kind == "round":
        return {"rel": 1e-10, "max": 1e-8, "differ": 0.0}      # float64 sums; decisions are the same
    if kind == "layer":
        return {"rel": 1e-2, "max": 1e-1}      # products stored in bf16
    if kind == "model":
        return {"rel": 3e-5, "max": 1e-3}      # float32 sums through every layer: up to 8e-6 from 64 bits
    if kind == "attn":   # bf16 keys and values, q and p split in two bf16 halves: 4e-6; float32: 1e-6
        return {"rel": 2e-5, "max": 1e-3} if case["bf16"] else {"rel": 5e-6, "max": 2e-4}
    # p times the row's scale goes in as two fp16 halves, the low one subnormal for most rows: 1e-4 to 2e-4
    return {"rel": 5e-4, "max": 1e-2}


# ---------------------------------------------------------------- 64-bit results
def _attend64(q, k, v, first):
    """q [T, Hq, D] at positions first.. over k, v [n, Hkv, D] (float64): output and probabilities [Hq, T, n]."""
    T, hq, d = q.shape
    n, hkv, _ = k.shape
    mask = torch.arange(n, device=DEV)[None, :] > first + torch.arange(T, device=DEV)[:, None]
    out = torch.empty_like(q)
    for h in range(hq):
        kh, vh = (t[:, h // (hq // hkv)].contiguous() for t in (k, v))
        p = torch.softmax((q[:, h].contiguous() @ kh.t() / math.sqrt(d)).masked_fill(mask, -math.inf), -1)
        out[:, h] = p @ vh
    return out


def _rope64(x, cos, sin):
    h = x.shape[-1] // 2
    a, b = x[..., :h], x[..., h:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _rms64(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


def _exact_model(case, seed):
    cfg, w, kv, tok = _model_inputs(case, seed)
    w = {n: t.double() for n, t in w.items()}
    hq, hkv, d = HEADS[case["model"]]
    b, T, ctx = case["batch"], case["tokens"], case["ctx"]
    gpt = case["model"] == "distilgpt2"
    pos = torch.arange(ctx, ctx + T, device=DEV)
    n_layers = cfg["n_layer"] if gpt else cfg["num_hidden_layers"]

    def ln(x, n):
        mu = x.mean(-1, keepdim=True)
        var = ((x - mu) ** 2).mean(-1, keepdim=True)
        return (x - mu) / torch.sqrt(var + cfg.get("layer_norm_epsilon", 1e-5)) * w[n + ".weight"] + w[n + ".bias"]

    def attention(i, q, k, v):
        out = []
        for s in range(b):
            ks, vs = k[s], v[s]
            if ctx:
                ks, vs = torch.cat([kv[i][0][s].double(), ks]), torch.cat([kv[i][1][s].double(), vs])
            out.append(_attend64(q[s], ks, vs, ctx))
        return torch.stack(out).reshape(b * T, hq * d)

    if gpt:
        h = (w["wte.weight"][tok.long()] + w["wpe.weight"][pos]).reshape(b * T, -1)
        for i in range(n_layers):
            p = f"h.{i}."
            x = ln(h, p + "ln_1") @ w[p + "attn.c_attn.weight"] + w[p + "attn.c_attn.bias"]
            q, k, v = (t.reshape(b, T, hq, d) for t in x.split(hq * d, -1))
            h = h + attention(i, q, k, v) @ w[p + "attn.c_proj.weight"] + w[p + "attn.c_proj.bias"]
            x = ln(h, p + "ln_2") @ w[p + "mlp.c_fc.weight"] + w[p + "mlp.c_fc.bias"]
            x = 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))
            h = h + x @ w[p + "mlp.c_proj.weight"] + w[p + "mlp.c_proj.bias"]
        return (ln(h, "ln_f") @ w["wte.weight"].t()).reshape(b, T, -1)
    eps = cfg["rms_norm_eps"]
    inv = 1.0 / (cfg["rope_theta"] ** (torch.arange(0, d, 2, device=DEV, dtype=F64) / d))
    ang = pos.double()[:, None] * inv
    cos, sin = ang.cos()[:, None], ang.sin()[:, None]
    h = w["model.embed_tokens.weight"][tok.long()].reshape(b * T, -1)
    for i in range(n_layers):
        p = f"model.layers.{i}."
        x = _rms64(h, w[p + "input_layernorm.weight"], eps)
        q, k, v = ((x @ w[p + f"self_attn.{n}_proj.weight"].t()).reshape(b, T, -1, d) for n in "qkv")
        h = h + attention(i, _rope64(q, cos, sin), _rope64(k, cos, sin), v) @ w[p + "self_attn.o_proj.weight"].t()
        x = _rms64(h, w[p + "post_attention_layernorm.weight"], eps)
        x = torch.nn.functional.silu(x @ w[p + "mlp.gate_proj.weight"].t()) * (x @ w[p + "mlp.up_proj.weight"].t())
        h = h + x @ w[p + "mlp.down_proj.weight"].t()
    return (_rms64(h, w["model.norm.weight"], eps) @ w["model.embed_tokens.weight"].t()).reshape(b, T, -1)


def _exact_layer(case, seed):
    c, w, norms, h, a, pos, cs = _layer_inputs(case, seed)
    hq, hkv, d = HEADS[case["model"]]
    n1, n2, n3 = (n.double() for n in norms)
    h, a, M, eps = h.double(), a.double(), case["rows"], c["rms_norm_eps"]
    mul = lambda x, n: x @ w[n].double().t()   # noqa: E731
    q, k, v = (t.reshape(M, -1, d) for t in mul(_rms64(h, n1, eps), "qkv").split([hq * d, hkv * d, hkv * d], -1))
    cos, sin = cs[0][:, None], cs[1][:, None]
    h = h + mul(a, "o")
    x = _rms64(h, n2, eps)
    h = h + mul(torch.nn.functional.silu(mul(x, "gate")) * mul(x, "up"), "down")
    return _rope64(q, cos, sin), _rope64(k, cos, sin), v, h, _rms64(h, n3, eps)


def _grid32(x, case):
    """x [.., d] through the arm's grid: the format's own float32 steps."""
    if case["bits"] == 16:
        return x.float()
    d, g, top = x.shape[-1], case["group"], float(2 ** case["bits"] - 1)
    x = torch.nn.functional.pad(x.float(), (0, -d % g)).unflatten(-1, (-1, g))
    lo, hi = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    scale = torch.div(hi - lo, torch.full_like(hi, top)).clamp_min(1e-8)   # by a tensor: a true division
    if case["half"]:
        lo, scale = lo.half().float(), scale.half().float()
        scale = torch.where(scale == 0, torch.full_like(scale, 2.0 ** -24), scale)
    code = torch.round((x - lo) / scale).clamp(0, top)
    return (code * scale + lo).flatten(-2)[..., :d]


def _exact_draft(case, seed):
    q, k, v = _draft_inputs(case, seed)
    hq, hkv, d = HEADS[case["model"]]
    n, kept = case["ctx"], _kept(case)
    rows = torch.cat([torch.arange(4, device=DEV), torch.arange(n - kept + 4, n, device=DEV)]) if kept < n \
        else torch.arange(n, device=DEV)
    cap = -(-(n + 64) // 32) * 32
    out = torch.empty(case["batch"], hq, d, device=DEV, dtype=F64)
    mass = torch.zeros(case["batch"], 1, cap, device=DEV, dtype=F64)
    for s in range(case["batch"]):
        ks, vs = (_grid32(t[s, rows], case).double() for t in (k, v))
        for h in range(hq):
            kh, vh = (t[:, h // (hq // hkv)].contiguous() for t in (ks, vs))
            p = torch.softmax(kh @ q[s, h].double() / math.sqrt(d), 0)
            out[s, h] = p @ vh
            if case["keep"] < 1:
                mass[s, 0, :kept] += p
    return out, mass


def exact(case, seed):
    kind = case["kind"]
    if kind == "model":
        return _exact_model(case, seed)
    if kind == "layer":
        return _exact_layer(case, seed)
    if kind == "attn":
        q, k, v = _attn_inputs(case, seed)
        return torch.stack([_attend64(q[s].double(), k[s].double(), v[s].double(), case["ctx"])
                            for s in range(case["batch"])])
    if kind == "draft":
        return _exact_draft(case, seed)
    if kind == "round" and case["temperature"] > 0:
        _, draft, _, _ = _round_inputs(case, seed)
        x = draft.double() / torch.tensor(case["temperature"], dtype=F32).item()   # the call takes it in float32
        m = x.amax(-1)
        total = torch.exp(x - m[..., None]).sum(-1)
        return None, None, None, None, torch.stack([m, total, 1 / total], -1)
    return None   # bits, bytes and tokens: compared as they are
