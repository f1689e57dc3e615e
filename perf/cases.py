"""What is timed, and what counts as the same answer: the calls that a program serving a
Qwen3-Next / Qwen3.6 mixture-of-experts model makes of this package, at the shapes that the
benchmark and the tests of this repository use.

Kinds of case (``case["kind"]``):

  moe        the decode step of a stack of MoE layers, one call per layer (MoELayerGPU.decode):
             every request of a batch contributes one token
  moe_norm   the same for one token with the residual add and the post-attention norm folded in
             (MoELayerGPU.decode_norm), the hidden state passing from layer to layer
  prefill    one MoE layer over a prompt chunk (MoELayerGPU.prefill)
  delta      one token through a stack of gated DeltaNet blocks (DeltaNetGPU.forward_token):
             input norm and projections, the recurrent step, out_proj
  attention  one token through a stack of gated attention blocks (AttentionGPU.forward_token)
             over a KV cache that holds `position` earlier tokens
  tail       the end of a token: final norm and lm_head, then sampling
  token      one token of a model: DeltaNet and attention blocks, each followed by its MoE
             step, then norm, lm_head and sampling

Weights are 4- or 8-bit codes with a scale and a bias per 64 inputs, as mlx's affine format
stores them; every layer of a stack has weights of its own, so that a pass reads memory as a
model does and not one layer out of the caches.
"""

from __future__ import annotations

import math

import torch

from swiftlet_amd._lib import SWQ_BF16, SWQ_DELTA_INTERLEAVED, SWQ_DELTA_SPLIT, SWQ_F16
from swiftlet_amd.attention import AttentionGPU
from swiftlet_amd.deltanet import DeltaNetGPU
from swiftlet_amd.engine import GPULinear, HipEngine
from swiftlet_amd.moe import MoELayerGPU

DEV = "cuda"
HIDDEN = 2048
EPS = 1e-6
VOCAB = 248320
GROUP = 64

# experts, picks per token, routed and shared intermediate size, code width of the expert
# matrices, type of scales and biases; the router's codes have 8 bits
MODELS = {
    "qwen3.6-35b-a3b-q4": (256, 8, 512, 512, 4, "f16"),
    "qwen3.6-35b-a3b-q8": (256, 8, 512, 512, 8, "f16"),
    "qwen3-next-80b-a3b-q4": (512, 10, 512, 512, 4, "bf16"),
}
# linear_attn: key heads, value heads, key and value head size, conv taps
DELTA = (16, 32, 128, 128, 4)
# self_attn: query heads, kv heads, head size, rotated dims, theta
ATTN = (16, 2, 256, 64, 1e7)


def listed():
    return [
        # one conversation: the MoE half of the layers of a token, hidden state handed on
        {"name": "moe-norm-35b-q4-b1", "kind": "moe_norm", "model": "qwen3.6-35b-a3b-q4", "layers": 8},
        # one conversation with the larger model
        {"name": "moe-80b-q4-b1", "kind": "moe", "model": "qwen3-next-80b-a3b-q4", "layers": 8, "batch": 1, "x": "bf16", "out": "bf16"},
        # four conversations with 8-bit experts
        {"name": "moe-35b-q8-b4", "kind": "moe", "model": "qwen3.6-35b-a3b-q8", "layers": 4, "batch": 4, "x": "bf16", "out": "bf16"},
        # the widest decode batch
        {"name": "moe-35b-q4-b16", "kind": "moe", "model": "qwen3.6-35b-a3b-q4", "layers": 2, "batch": 16, "x": "bf16", "out": "f32"},
        # a short turn of a chat, its length as it comes, f32 activations
        {"name": "prefill-35b-q8-t77", "kind": "prefill", "model": "qwen3.6-35b-a3b-q8", "tokens": 77, "x": "f32", "out": "f32"},
        # a prompt chunk of the size the benchmark uses
        {"name": "prefill-35b-q4-t512", "kind": "prefill", "model": "qwen3.6-35b-a3b-q4", "tokens": 512, "x": "bf16", "out": "bf16"},
        # a long prompt in one call
        {"name": "prefill-35b-q4-t4096", "kind": "prefill", "model": "qwen3.6-35b-a3b-q4", "tokens": 4096, "x": "bf16", "out": "bf16"},
        # the linear-attention blocks of a token
        {"name": "delta-split", "kind": "delta", "layout": "split", "layers": 6, "position": 1000},
        # the full-attention blocks of a token: a conversation of some length, and a long document
        {"name": "attention-4k", "kind": "attention", "layers": 4, "position": 4095},
        {"name": "attention-33k", "kind": "attention", "layers": 2, "position": 33000},
        # logits and the next token, with the sampling options that the model's card gives
        {"name": "lm-head-sample", "kind": "tail", "temperature": 0.7, "top_k": 20, "top_p": 0.8, "presence": 1.5, "seen": 200},
        # a whole token of a four-layer model, greedy
        {"name": "token-4-layers", "kind": "token", "model": "qwen3.6-35b-a3b-q4", "position": 1500},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["moe", "moe", "moe_norm", "prefill", "prefill", "delta", "attention", "attention", "tail", "token"])
    model = rng.choice(sorted(MODELS))
    if kind == "moe":
        batch = rng.choice([1, 1, 2, 3, 4, 5, 6, 7, 8, 11, 13, 16])
        return {"kind": kind, "model": model, "layers": rng.randint(1, 8 if batch < 4 else 2), "batch": batch,
                "x": rng.choice(["bf16", "bf16", "f32"]), "out": rng.choice(["bf16", "f32"])}
    if kind == "moe_norm":
        return {"kind": kind, "model": model, "layers": rng.randint(1, 8)}
    if kind == "prefill":
        return {"kind": kind, "model": model, "tokens": _log(rng, 1, 4096 if model.endswith("35b-a3b-q4") else 2048),
                "x": "f32" if rng.random() < 0.25 else "bf16", "out": rng.choice(["bf16", "f32"])}
    if kind == "delta":
        return {"kind": kind, "layout": rng.choice(["split", "interleaved"]), "layers": rng.randint(1, 6), "position": _log(rng, 1, 100000)}
    if kind == "attention":
        return {"kind": kind, "layers": rng.randint(1, 2), "position": _log(rng, 1, 33000)}
    if kind == "tail":
        return {"kind": kind, "temperature": rng.choice([0.0, 0.6, 1.0]), "top_k": rng.randint(1, 40), "top_p": rng.choice([0.8, 0.95, 1.0]),
                "presence": rng.choice([0.0, 1.5]), "seen": _log(rng, 1, 2000)}
    return {"kind": kind, "model": model, "position": _log(rng, 1, 8000)}


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _quantized(g, rows, cols, bits, stype, experts=None):
    """Uniform codes; scales so that a weight's spread is about 1/sqrt(2048) times two; biases
    near the middle of the code range, so that weights lie on both sides of zero."""
    lead = (experts or 1) * rows
    words = torch.randint(-2 ** 31, 2 ** 31, (lead, cols * bits // 32), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    s = torch.rand((lead, cols // GROUP), generator=g, device=DEV)
    s = (0.005 + 0.015 * s) * (15.0 / (2 ** bits - 1))
    mid = (2 ** bits - 1) / 2
    b = -s * (mid + 0.1 * mid * (torch.rand(s.shape, generator=g, device=DEV) - 0.5))
    dt = {"f16": torch.float16, "bf16": torch.bfloat16}[stype]
    s, b = s.to(dt), b.to(dt)
    flat = [t.reshape(-1).view(torch.uint8) for t in (words, s, b)]
    return GPULinear(*flat, rows, cols, GROUP, bits, {"f16": SWQ_F16, "bf16": SWQ_BF16}[stype],
                     expert_stride_w=rows * cols * bits // 8 if experts else 0,
                     expert_stride_sb=rows * (cols // GROUP) * 2 if experts else 0, num_experts=experts or 1)


def _moe_layer(g, model):
    E, K, I, Is, bits, st = MODELS[model]
    return MoELayerGPU(
        router=_quantized(g, E, HIDDEN, 8, st),
        gate=_quantized(g, I, HIDDEN, bits, st, E), up=_quantized(g, I, HIDDEN, bits, st, E), down=_quantized(g, HIDDEN, I, bits, st, E),
        shared_gate=_quantized(g, Is, HIDDEN, bits, st), shared_up=_quantized(g, Is, HIDDEN, bits, st),
        shared_down=_quantized(g, HIDDEN, Is, bits, st), shared_expert_gate=_quantized(g, 1, HIDDEN, 8, st), top_k=K)


def _norm_weight(g, n, dtype=torch.bfloat16):
    return (1.0 + 0.1 * torch.randn(n, generator=g, device=DEV)).to(dtype)


def _dtype(name):
    return {"bf16": torch.bfloat16, "f32": torch.float32}[name]


def _clear_rows(g, router, top_k, n, dtype, shared):
    """n rows of activations whose k-th and (k+1)-th router logits are not within rounding of
    each other, so that every correct implementation picks the same experts.  ``shared``: the
    size of a component that all rows have in common, as the tokens of one prompt do; it makes
    some experts busier than others."""
    m = n + 16 + n // 4
    x = torch.randn((m, HIDDEN), generator=g, device=DEV)
    if shared:
        x = x + shared * torch.randn((1, HIDDEN), generator=g, device=DEV)
    x = x.to(dtype)
    logits = x.double() @ _weight(router).t()
    top = logits.topk(top_k + 1, dim=1).values
    good = (top[:, top_k - 1] - top[:, top_k] > 1e-3).nonzero().reshape(-1)
    return x[good[:n]].contiguous()


def _delta_block(g, layout):
    nk, nv, dk, dv, taps = DELTA
    key, val = nk * dk, nv * dv
    rows = (2 * key + val, val, nv, nv) if layout == "split" else (2 * key + 2 * val, 2 * nv)
    r = lambda *s: torch.randn(s, generator=g, device=DEV)  # noqa: E731
    return DeltaNetGPU(nk, nv, dk, dv, taps, SWQ_DELTA_SPLIT if layout == "split" else SWQ_DELTA_INTERLEAVED, EPS,
                       r((2 * key + val) * taps) * 0.3, r(nv) * 0.5, r(nv) * 0.5, 1.0 + 0.1 * r(dv),
                       projections=[_quantized(g, n, HIDDEN, 4, "f16") for n in rows], out_proj=_quantized(g, HIDDEN, val, 4, "f16"))


def _delta_state(g, block):
    """The state of a conversation under way."""
    st = block.new_state()
    ring, rec = block.state_views(st)
    ring.normal_(generator=g)
    rec.normal_(0.0, 0.1, generator=g)
    return st


def _attention_block(g, position):
    H, KVH, hd, rot, theta = ATTN
    return AttentionGPU(H, KVH, hd, rot, theta, EPS, position + 1, 1.0 + 0.1 * torch.randn(hd, generator=g, device=DEV),
                        1.0 + 0.1 * torch.randn(hd, generator=g, device=DEV),
                        projections=[_quantized(g, n, HIDDEN, 4, "f16") for n in (H * 2 * hd, KVH * hd, KVH * hd)],
                        o_proj=_quantized(g, HIDDEN, H * hd, 4, "f16"))


def _attention_cache(g, block, position):
    cache = block.new_cache()
    k, v = block.cache_views(cache)
    k[:position].normal_(0.0, 0.5, generator=g)
    v[:position].normal_(generator=g)
    return cache


def _tail_parts(g):
    return {"engine": HipEngine(), "w_final": _norm_weight(g, HIDDEN), "head": _quantized(g, VOCAB, HIDDEN, 4, "f16"),
            "logits": torch.empty(VOCAB, dtype=torch.float32, device=DEV)}


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind in ("moe", "moe_norm"):
        K = MODELS[case["model"]][1]
        layers = [_moe_layer(g, case["model"]) for _ in range(case["layers"])]
        n = len(layers)
        B = case.get("batch", 1)
        s["layers"], s["ws"] = layers, [l.new_workspace(B) for l in layers]
        s["ids"] = [torch.empty((B, K), dtype=torch.int32, device=DEV) for _ in range(n)]
        s["wts"] = [torch.empty((B, K), dtype=torch.float32, device=DEV) for _ in range(n)]
        if kind == "moe":
            s["x"] = [_clear_rows(g, l.router, K, B, _dtype(case["x"]), 0.0) for l in layers]
            s["out"] = [torch.empty((B, HIDDEN), dtype=_dtype(case["out"]), device=DEV) for _ in range(n)]
        else:
            s["h"] = torch.randn(HIDDEN, generator=g, device=DEV)
            s["r"] = [torch.randn(HIDDEN, generator=g, device=DEV) for _ in range(n)]  # the attention halves' outputs
            s["w"] = [_norm_weight(g, HIDDEN) for _ in range(n)]
            s["out"] = [torch.empty(HIDDEN, dtype=torch.float32, device=DEV) for _ in range(n)]
    elif kind == "prefill":
        T, K = case["tokens"], MODELS[case["model"]][1]
        layer = _moe_layer(g, case["model"])
        s["layer"], s["ws"] = layer, layer.new_prefill_workspace(T)
        s["x"] = _clear_rows(g, layer.router, K, T, _dtype(case["x"]), 0.6)
        s["out"] = torch.empty((T, HIDDEN), dtype=_dtype(case["out"]), device=DEV)
        s["ids"] = torch.empty((T, K), dtype=torch.int32, device=DEV)
        s["wts"] = torch.empty((T, K), dtype=torch.float32, device=DEV)
    elif kind == "delta":
        n = case["layers"]
        s["engine"], s["position"] = HipEngine(), case["position"]
        s["blocks"] = [_delta_block(g, case["layout"]) for _ in range(n)]
        s["states"] = [_delta_state(g, b) for b in s["blocks"]]
        s["x"] = [torch.randn(HIDDEN, generator=g, device=DEV) for _ in range(n)]
        s["w"] = [_norm_weight(g, HIDDEN) for _ in range(n)]
    elif kind == "attention":
        n = case["layers"]
        s["engine"] = HipEngine()
        s["blocks"] = [_attention_block(g, case["position"]) for _ in range(n)]
        s["caches"] = [_attention_cache(g, b, case["position"]) for b in s["blocks"]]
        s["ws"] = s["blocks"][0].new_workspace()
        s["x"] = [torch.randn(HIDDEN, generator=g, device=DEV) for _ in range(n)]
        s["w"] = [_norm_weight(g, HIDDEN) for _ in range(n)]
    else:
        s.update(_tail_parts(g))
        s["sample_ws"] = s["engine"].new_sample_workspace(VOCAB)
        s["h"] = torch.randn(HIDDEN, generator=g, device=DEV)
        if kind == "tail":
            ids = torch.randperm(VOCAB, generator=g, device=DEV)[:case["seen"]].tolist()
            s["seen"] = {t: 1 + i % 3 for i, t in enumerate(ids)}
            s["u"] = float(torch.rand(1, generator=g, device=DEV))
        else:
            pos = case["position"]
            s["position"] = pos
            blocks = [_delta_block(g, "split") for _ in range(3)] + [_attention_block(g, pos)]
            s["blocks"] = blocks
            s["states"] = [_delta_state(g, b) for b in blocks[:3]] + [_attention_cache(g, blocks[3], pos)]
            s["attn_ws"] = blocks[3].new_workspace()
            s["moe"] = [_moe_layer(g, case["model"]) for _ in blocks]
            s["moe_ws"] = [l.new_workspace(1) for l in s["moe"]]
            s["w_in"] = [_norm_weight(g, HIDDEN) for _ in blocks]
            s["w_post"] = [_norm_weight(g, HIDDEN) for _ in blocks]
            s["hidden"] = [torch.empty(HIDDEN, dtype=torch.float32, device=DEV) for _ in blocks]
    return s


# ---------------------------------------------------------------------------
# one pass


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "moe":
        for l, x, out, ws, ids, wts in zip(s["layers"], s["x"], s["out"], s["ws"], s["ids"], s["wts"]):
            l.decode(x, out=out, ws=ws, topk_ids=ids, topk_weights=wts)
        return {"out": s["out"], "ids": s["ids"], "weights": s["wts"]}
    if kind == "moe_norm":
        h = s["h"]
        for l, r, w, out, ws, ids, wts in zip(s["layers"], s["r"], s["w"], s["out"], s["ws"], s["ids"], s["wts"]):
            l.decode_norm(h, w, EPS, residual=r, out=out, ws=ws, topk_ids=ids, topk_weights=wts)
            h = out
        return {"out": s["out"], "ids": s["ids"], "weights": s["wts"]}
    if kind == "prefill":
        s["layer"].prefill(s["x"], out=s["out"], ws=s["ws"], topk_ids=s["ids"], topk_weights=s["wts"])
        return {"out": s["out"], "ids": s["ids"], "weights": s["wts"]}
    if kind == "delta":
        pos = s["position"]
        s["position"] = pos + 1
        out = [b.forward_token(s["engine"], x, st, pos, norm_weight=w, eps=EPS)
               for b, x, st, w in zip(s["blocks"], s["x"], s["states"], s["w"])]
        return {"out": out, "state": [list(b.state_views(st)) for b, st in zip(s["blocks"], s["states"])]}
    if kind == "attention":
        pos = case["position"]  # the same one each time: the token's row of the cache is written anew
        out = [b.forward_token(s["engine"], x, c, s["ws"], pos, norm_weight=w, eps=EPS)
               for b, x, c, w in zip(s["blocks"], s["x"], s["caches"], s["w"])]
        return {"out": out, "new_rows": [[t[pos] for t in b.cache_views(c)] for b, c in zip(s["blocks"], s["caches"])]}
    eng, h = s["engine"], s["h"]
    if kind == "token":
        pos, delta_pos = case["position"], s["position"]
        s["position"] = delta_pos + 1
        for b, st, w_in, w_post, moe, ws, out in zip(s["blocks"], s["states"], s["w_in"], s["w_post"], s["moe"], s["moe_ws"], s["hidden"]):
            if isinstance(b, DeltaNetGPU):
                r = b.forward_token(eng, h, st, delta_pos, norm_weight=w_in, eps=EPS)
            else:
                r = b.forward_token(eng, h, st, s["attn_ws"], pos, norm_weight=w_in, eps=EPS)
            moe.decode_norm(h, w_post, EPS, residual=r, out=out, ws=ws)
            h = out
    eng.encode_gemv_multi([s["head"]], h, [s["logits"]], norm_weight=s["w_final"], eps=EPS)
    if kind == "token":
        tok = eng.sample(s["logits"], 0.0, 1, 1.0, ws=s["sample_ws"])
        return {"logits": s["logits"], "hidden": s["hidden"], "token": tok}
    tok = eng.sample(s["logits"], case["temperature"], case["top_k"], case["top_p"], presence=case["presence"], frequency=0.5 * (case["presence"] > 0),
                     seen=s["seen"], banned=(VOCAB - 1,), u=s["u"], ws=s["sample_ws"])
    return {"logits": s["logits"], "token": tok}


# ---------------------------------------------------------------------------
# the least that a pass has to read, write and compute


def _matrix(rows, cols, bits):
    return rows * cols * bits / 8 + rows * (cols / GROUP) * 4


def _moe_work(model, tokens, x_bytes, out_bytes):
    E, K, I, Is, bits, _ = MODELS[model]
    distinct = E * (1 - (1 - K / E) ** tokens)
    size = distinct * (2 * _matrix(I, HIDDEN, bits) + _matrix(HIDDEN, I, bits)) + 2 * _matrix(Is, HIDDEN, bits) + _matrix(HIDDEN, Is, bits)
    size += _matrix(E + 1, HIDDEN, 8) + tokens * (HIDDEN * (x_bytes + out_bytes) + 8 * K)
    return size, 2.0 * tokens * HIDDEN * (3 * (K * I + Is) + E + 1)


def _delta_work():
    nk, nv, dk, dv, taps = DELTA
    conv, val = 2 * nk * dk + nv * dv, nv * dv
    size = _matrix(conv + val + 2 * nv, HIDDEN, 4) + _matrix(HIDDEN, val, 4)
    size += 4 * (2 * nv * dv * dk + conv * 2 * taps + 2 * HIDDEN)
    return size, 2.0 * HIDDEN * (conv + 2 * val + 2 * nv) + 7.0 * nv * dv * dk


def _attention_work(position):
    H, KVH, hd, _, _ = ATTN
    n = position + 1
    size = _matrix(H * 2 * hd + 2 * KVH * hd, HIDDEN, 4) + _matrix(HIDDEN, H * hd, 4) + 4 * (2 * n * KVH * hd + 2 * HIDDEN)
    return size, 2.0 * HIDDEN * (3 * H * hd + 2 * KVH * hd) + 4.0 * n * H * hd


def _tail_work():
    return _matrix(VOCAB, HIDDEN, 4) + 4 * VOCAB + 6 * HIDDEN, 2.0 * VOCAB * HIDDEN


def work(case):
    kind, size, flops = case["kind"], 0.0, 0.0
    width = {"bf16": 2, "f32": 4}
    n = case.get("layers", 1)
    if kind == "moe":
        parts = [_moe_work(case["model"], case["batch"], width[case["x"]], width[case["out"]])] * n
    elif kind == "moe_norm":
        parts = [_moe_work(case["model"], 1, 8, 6)] * n
    elif kind == "prefill":
        parts = [_moe_work(case["model"], case["tokens"], width[case["x"]], width[case["out"]])]
    elif kind == "delta":
        parts = [_delta_work()] * n
    elif kind == "attention":
        parts = [_attention_work(case["position"])] * n
    elif kind == "tail":
        parts = [_tail_work()]
    else:
        parts = [_moe_work(case["model"], 1, 8, 6)] * 4 + [_delta_work()] * 3 + [_attention_work(case["position"]), _tail_work()]
    return {"bytes": sum(p[0] for p in parts), "flops": sum(p[1] for p in parts)}


# ---------------------------------------------------------------------------
# agreement


def tolerance(case):
    """About four times what the start shows against 64 bits.  16-bit outputs are within half a
    unit of their last place (2^-9 at most); elsewhere it is the sums of 32-bit products, and
    in the expert layers the hidden activations' 16 significant bits."""
    kind = case["kind"]
    if case.get("out") == "bf16":
        return {"rel": 4e-3, "max": 1.6e-2}
    if kind in ("moe", "prefill"):
        return {"rel": 2e-5, "max": 2e-4}
    if kind in ("moe_norm", "token"):
        return {"rel": 4e-5, "max": 4e-4}
    return {"rel": 1e-5, "max": 1e-4}


def _weight(lin, expert=0):
    """The matrix (of one expert) in 64 bits: scale * code + bias."""
    per = 32 // lin.bits
    rows, cols = lin.out_dim, lin.in_dim
    words = lin.w.view(torch.int32).reshape(-1, rows, cols // per)[expert]
    shift = torch.arange(per, device=words.device, dtype=torch.int32) * lin.bits
    codes = ((words.unsqueeze(-1) >> shift) & (2 ** lin.bits - 1)).reshape(rows, cols // GROUP, GROUP).double()
    dt = torch.float16 if lin.scales_type == SWQ_F16 else torch.bfloat16
    sc = lin.scales.view(dt).reshape(-1, rows, cols // GROUP, 1)[expert].double()
    bi = lin.biases.view(dt).reshape(-1, rows, cols // GROUP, 1)[expert].double()
    return (codes * sc + bi).reshape(rows, cols)


def _silu(v):
    return v * torch.sigmoid(v)


def _moe_exact(l, x):
    """x [T, H] in 64 bits -> (out, ids, weights)."""
    logits = x @ _weight(l.router).t()
    top, ids = logits.topk(l.top_k, dim=1)
    wts = torch.softmax(top, dim=1)
    out = torch.zeros_like(x)
    for e in ids.unique().tolist():
        t, k = (ids == e).nonzero(as_tuple=True)
        xe = x[t]
        h = _silu(xe @ _weight(l.gate, e).t()) * (xe @ _weight(l.up, e).t())
        out.index_add_(0, t, (h @ _weight(l.down, e).t()) * wts[t, k].unsqueeze(1))
    h = _silu(x @ _weight(l.shared_gate).t()) * (x @ _weight(l.shared_up).t())
    out += (h @ _weight(l.shared_down).t()) * torch.sigmoid(x @ _weight(l.shared_expert_gate).t())
    return out, ids, wts


def _rms(x, w=None, eps=EPS):
    y = x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w.double()


def _delta_exact(b, x, state, position, w):
    """One block in 64 bits: (output, conv ring, recurrent state) after the token."""
    nk, nv, dk, dv, taps = DELTA
    rep, key, val = nv // nk, nk * dk, nv * dv
    conv_dim = 2 * key + val
    xn = _rms(x.double(), w)
    p = [_weight(l) @ xn for l in b.projections]
    if b.layout == SWQ_DELTA_SPLIT:
        mixed, z, beta, alpha = p
    else:
        q, k, v, z = p[0].reshape(nk, -1).split([dk, dk, rep * dv, rep * dv], dim=1)
        mixed, z = torch.cat([t.reshape(-1) for t in (q, k, v)]), z.reshape(-1)
        beta, alpha = (t.reshape(-1) for t in p[1].reshape(nk, 2 * rep).split([rep, rep], dim=1))
    ring, rec = (t.double().clone() for t in b.state_views(state))
    ring[position % taps] = mixed
    order = [(position + 1 + j) % taps for j in range(taps)]
    c = _silu((ring[order].t() * b.conv_weight.double().reshape(conv_dim, taps)).sum(1))
    q = _rms(c[:key].reshape(nk, dk), None, 1e-6) / dk
    k = _rms(c[key:2 * key].reshape(nk, dk), None, 1e-6) / math.sqrt(dk)
    q, k = q.repeat_interleave(rep, 0).unsqueeze(1), k.repeat_interleave(rep, 0).unsqueeze(1)
    v = c[2 * key:].reshape(nv, dv)
    decay = torch.exp(-torch.exp(b.a_log.double()) * torch.nn.functional.softplus(alpha + b.dt_bias.double()))
    rec = rec * decay.reshape(nv, 1, 1)
    delta = (v - (rec * k).sum(-1)) * torch.sigmoid(beta).unsqueeze(1)
    rec = rec + delta.unsqueeze(-1) * k
    y = _rms((rec * q).sum(-1), b.norm_weight).reshape(-1) * _silu(z)
    return _weight(b.out_proj) @ y, ring, rec


def _attention_exact(b, x, cache, position, w):
    """One block in 64 bits: (output, the new k row, the new v row)."""
    H, KVH, hd, rot, theta = ATTN
    xn = _rms(x.double(), w)
    q, k, v = (_weight(l) @ xn for l in b.projections)
    q, gate = q.reshape(H, 2 * hd).split([hd, hd], dim=1)
    q, k, v = _rms(q, b.q_norm), _rms(k.reshape(KVH, hd), b.k_norm), v.reshape(KVH, hd)
    # angles as the model's code has them, in 32 bits: at a long context 64-bit angles are others
    j = torch.arange(rot // 2, dtype=torch.float64)
    inv = torch.pow(torch.tensor(float(theta), dtype=torch.float64), (-(2 * j).float() / rot).double()).float()
    ang = (torch.tensor(float(position)) * inv).double().to(x.device)
    cs, sn = torch.cos(ang), torch.sin(ang)

    def rope(t):
        lo, hi = t[:, :rot // 2], t[:, rot // 2:rot]
        return torch.cat([lo * cs - hi * sn, hi * cs + lo * sn, t[:, rot:]], dim=1)

    q, k = rope(q), rope(k)
    ck, cv = b.cache_views(cache)
    out = []
    for n in range(KVH):
        keys = torch.cat([ck[:position, n].double(), k[n:n + 1]])
        vals = torch.cat([cv[:position, n].double(), v[n:n + 1]])
        hs = q[n * (H // KVH):(n + 1) * (H // KVH)]
        out.append(torch.softmax(hs @ keys.t() / math.sqrt(hd), dim=1) @ vals)
    y = torch.cat(out) * torch.sigmoid(gate)
    return _weight(b.o_proj) @ y.reshape(-1), k, v


def _logits_exact(head, h, w):
    xn = _rms(h.double(), w)
    out = []
    for lo in range(0, VOCAB, 31040):
        part = GPULinear(head.w[lo * HIDDEN // 2:(lo + 31040) * HIDDEN // 2], head.scales[lo * HIDDEN // 32:(lo + 31040) * HIDDEN // 32],
                         head.biases[lo * HIDDEN // 32:(lo + 31040) * HIDDEN // 32], 31040, HIDDEN, GROUP, 4, head.scales_type)
        out.append(_weight(part) @ xn)
    return torch.cat(out)


def exact(case, seed):
    """What run() returns on a new state, from the same stored inputs by plain torch in 64 bits."""
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "moe":
        res = [_moe_exact(l, x.double()) for l, x in zip(s["layers"], s["x"])]
        return {"out": [r[0] for r in res], "ids": [r[1] for r in res], "weights": [r[2] for r in res]}
    if kind == "moe_norm":
        h, res = s["h"].double(), []
        for l, r, w in zip(s["layers"], s["r"], s["w"]):
            h = h + r.double()
            y, ids, wts = _moe_exact(l, _rms(h, w).unsqueeze(0))
            h = h + y[0]
            res.append((h, ids, wts))
        return {"out": [r[0] for r in res], "ids": [r[1] for r in res], "weights": [r[2] for r in res]}
    if kind == "prefill":
        out, ids, wts = _moe_exact(s["layer"], s["x"].double())
        return {"out": out, "ids": ids, "weights": wts}
    if kind == "delta":
        res = [_delta_exact(b, x, st, s["position"], w) for b, x, st, w in zip(s["blocks"], s["x"], s["states"], s["w"])]
        return {"out": [r[0] for r in res], "state": [[r[1], r[2]] for r in res]}
    if kind == "attention":
        res = [_attention_exact(b, x, c, case["position"], w) for b, x, c, w in zip(s["blocks"], s["x"], s["caches"], s["w"])]
        return {"out": [r[0] for r in res], "new_rows": [[r[1], r[2]] for r in res]}
    if kind == "tail":
        return {"logits": _logits_exact(s["head"], s["h"], s["w_final"]), "token": None}
    h, hidden = s["h"].double(), []
    for b, st, w_in, w_post, moe in zip(s["blocks"], s["states"], s["w_in"], s["w_post"], s["moe"]):
        r = (_delta_exact if isinstance(b, DeltaNetGPU) else _attention_exact)(b, h, st, case["position"], w_in)[0]
        h = h + r
        h = h + _moe_exact(moe, _rms(h, w_post).unsqueeze(0))[0][0]
        hidden.append(h)
    logits = _logits_exact(s["head"], h, s["w_final"])
    return {"logits": logits, "hidden": hidden, "token": int(logits.argmax())}
