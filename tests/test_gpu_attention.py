"""Gated GQA attention decode on the device (swq_attention_step) against the
oracle (oracle/attention_ref.py, QwenCPUModel.attentionForward + applyRope,
QwenCPUModel.swift:285-367).

Bar: fp32, sums and the softmax in another order (split positions, online
maxima) — each token's output within 1e-5 of the oracle's (max abs error
over max abs value); the cache rows the step appends within the same bound
(normalised, rotated k; v bit-exact).  Cases: the tiny model's attention
shape (hd 16, 4 heads over 2 kv heads, 4 rotary dims) token by token; the
35B / 80B shape (16 heads over 2 kv heads, hd 256, 64 rotary dims, theta
1e7) token by token over five splits of 16 positions, and single steps
at positions 1000 and 5000 over a random cache (splits of one tile, and of
more); and the reference's tiny 4-bit qwen3_next model run
entirely on the device — embedding rows, every norm, DeltaNet and attention
block (input norm fused into the projections' launch), MoE block and the
lm_head — against mlx's logits (2e-3,
FixtureForwardTests.swift:94-95) and greedy ids."""

import json
from pathlib import Path

import numpy as np
import pytest

from oracle import attention_ref as A
from oracle.qwen_tiny import TinyQwen
from swiftlet_amd.attention import AttentionGPU, attention_from_checkpoint

pytestmark = pytest.mark.gpu

G = Path(__file__).resolve().parent / "golden" / "swiftlet_fixtures"
f32 = np.float32


def _rel(got, want):
    return float(np.abs(np.asarray(got) - want).max() / max(np.abs(want).max(), 1e-30))


def _block(prm, max_positions):
    return AttentionGPU(prm["H"], prm["KVH"], prm["hd"], prm["rot"], prm["theta"], prm["eps"], max_positions,
                        prm["q_norm_w"], prm["k_norm_w"])


def _sequence(prm, S, seed):
    import torch
    rng = np.random.default_rng(seed)
    H, KVH, hd = prm["H"], prm["KVH"], prm["hd"]
    blk = _block(prm, 256)
    cache, ws = blk.new_cache(), blk.new_workspace()
    q = rng.standard_normal((S, H * 2 * hd)).astype(f32)
    k = rng.standard_normal((S, KVH * hd)).astype(f32)
    v = rng.standard_normal((S, KVH * hd)).astype(f32)
    want, ck, cv = A.attention_core(q, k, v, **prm)
    worst = 0.0
    for s in range(S):
        out = blk.step(*(torch.from_numpy(t[s]).cuda() for t in (q, k, v)), cache, ws, s)
        torch.cuda.synchronize()
        worst = max(worst, _rel(out.cpu().numpy(), want[s]))
    gk, gv = blk.cache_views(cache)
    assert _rel(gk[:S].cpu().numpy(), ck) < 1e-5
    assert np.array_equal(gv[:S].cpu().numpy(), cv)
    return worst


def test_tiny_model_shape():
    err = _sequence(TinyQwen(G / "tiny-model-q4").attention_params(3), S=12, seed=2)
    print(f"tiny: {err:.2e}", flush=True)
    assert err < 1e-5


def _big_params(rng):
    return dict(q_norm_w=(1 + 0.2 * rng.standard_normal(256)).astype(f32),
                k_norm_w=(1 + 0.2 * rng.standard_normal(256)).astype(f32),
                H=16, KVH=2, hd=256, rot=64, theta=1e7, eps=1e-6)


def test_real_shape_sequence_across_splits():
    err = _sequence(_big_params(np.random.default_rng(3)), S=70, seed=4)
    print(f"35B shape, 70 tokens: {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("position", [1000, 5000])
def test_real_shape_long_cache(position):
    import torch
    rng = np.random.default_rng(position)
    prm = _big_params(rng)
    blk = _block(prm, 6000)
    cache, ws = blk.new_cache(), blk.new_workspace()
    gk, gv = blk.cache_views(cache)
    # a cache of unit-scale rows, as normalised keys are
    ck = (rng.standard_normal((position, 2, 256)) * 0.5).astype(f32)
    cv = rng.standard_normal((position, 2, 256)).astype(f32)
    gk[:position].copy_(torch.from_numpy(ck))
    gv[:position].copy_(torch.from_numpy(cv))
    q = rng.standard_normal((1, 16 * 2 * 256)).astype(f32)
    k = rng.standard_normal((1, 2 * 256)).astype(f32)
    v = rng.standard_normal((1, 2 * 256)).astype(f32)
    want, _, _ = A.attention_core(q, k, v, cache_k=ck, cache_v=cv, **prm)
    print(f"position {position}", flush=True)
    out = blk.step(*(torch.from_numpy(t[0]).cuda() for t in (q, k, v)), cache, ws, position)
    torch.cuda.synchronize()
    err = _rel(out.cpu().numpy(), want[0])
    print(f"error {err:.2e}", flush=True)
    assert err < 1e-5


@pytest.mark.parametrize("H,KVH,hd,rot,position", [
    (1, 1, 16, 4, 0), (16, 1, 16, 16, 15), (6, 2, 32, 8, 16), (3, 3, 64, 0, 17), (16, 1, 128, 32, 31),
    (16, 2, 256, 64, 32), (16, 2, 256, 2, 4094), (16, 2, 256, 2, 4095), (16, 2, 256, 2, 4096), (5, 1, 64, 2, 8191),
    (16, 2, 256, 2, 8191), (16, 2, 256, 2, 8192), (16, 8, 128, 2, 2113)])
def test_split_edges(H, KVH, hd, rot, position):
    """Positions at the edges of a 16-position tile, of a split of one tile (512 / KVH of them,
    at most 512) and of a step of two tiles; every head size, groups of 1 to 16.  Rows of the
    cache past the position hold NaN, as does the new row before the step.  From position 2,000
    on two dims rotate: their angle is the position itself, while theta^(-2j/rot), j > 0, may
    differ in its last bit from NumPy's float32 power, which moves the angle by up to position *
    2^-24 (2e-4 at 4,094), in any order of the sums.  Bar: that of the
    other cases, 1e-5 of the largest output (sums of up to 8,193 fp32 products in blocks:
    ~2^-24 * sqrt(8193) = 5e-6)."""
    import torch
    rng = np.random.default_rng(1000 * H + position)
    prm = dict(q_norm_w=(1 + 0.2 * rng.standard_normal(hd)).astype(f32), k_norm_w=(1 + 0.2 * rng.standard_normal(hd)).astype(f32),
               H=H, KVH=KVH, hd=hd, rot=rot, theta=1e7, eps=1e-6)
    blk = _block(prm, position + 40)
    cache, ws = blk.new_cache(), blk.new_workspace()
    gk, gv = blk.cache_views(cache)
    ck = (rng.standard_normal((position, KVH, hd)) * 0.5).astype(f32)
    cv = rng.standard_normal((position, KVH, hd)).astype(f32)
    gk[position:].fill_(float("nan"))
    gv[position:].fill_(float("nan"))
    gk[:position].copy_(torch.from_numpy(ck))
    gv[:position].copy_(torch.from_numpy(cv))
    q, k, v = (rng.standard_normal((1, n)).astype(f32) for n in (H * 2 * hd, KVH * hd, KVH * hd))
    want, wk, wv = A.attention_core(q, k, v, cache_k=ck, cache_v=cv, **prm)
    print(f"H {H} KVH {KVH} hd {hd} position {position}", flush=True)
    out = blk.step(*(torch.from_numpy(t[0]).cuda() for t in (q, k, v)), cache, ws, position)
    torch.cuda.synchronize()
    assert _rel(out.cpu().numpy(), want[0]) < 1e-5
    assert _rel(gk[position].cpu().numpy(), wk[-1]) < 1e-5
    assert np.array_equal(gv[position].cpu().numpy(), wv[-1])
    assert torch.isnan(gk[position + 1:]).all() and np.array_equal(gk[:position].cpu().numpy(), ck)


@pytest.mark.parametrize("H,KVH,hd,position", [(32, 8, 128, 33000), (16, 2, 256, 33000), (8, 8, 64, 8200)])
def test_long_sums_against_64_bits(H, KVH, hd, position):
    """A split's value sums stay as exact over hundreds of positions as over one tile's.  A chain of m
    equal steps rounds by about 3.4e-8 (2^-24 / sqrt(3)) of its partial sums at each, 3.4e-8 *
    sqrt(m / 2) of the result: blocks of 16 and 16 steps of two of them 1e-7 each, with the scores'
    and the merge's roundings 1.9e-7 measured; one chain of a split's 516 positions 5e-7 (4.3e-7
    measured).  Bar: 3e-7 relative 2-norm."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(position + hd)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    qw, kw, eps = 1 + 0.1 * r(hd), 1 + 0.1 * r(hd), 1e-6
    blk = AttentionGPU(H, KVH, hd, 0, 1e7, eps, position + 1, qw, kw)
    cache, ws = blk.new_cache(), blk.new_workspace()
    ck, cv = blk.cache_views(cache)
    ck[:position].normal_(0.0, 0.5, generator=g)
    cv[:position].normal_(generator=g)
    q, k, v = r(H, 2, hd), r(KVH, hd), r(KVH, hd)
    print(f"H {H} KVH {KVH} hd {hd} position {position}", flush=True)
    out = blk.step(q.reshape(-1), k.reshape(-1), v.reshape(-1), cache, ws, position)
    norm = lambda x, w: x / (x.pow(2).mean(-1, keepdim=True) + eps).sqrt() * w.double()  # noqa: E731
    qn = norm(q[:, 0].double(), qw)
    ck[position].copy_(norm(k.double(), kw).float())
    want = []
    for h in range(H):
        p = ((ck[:, h * KVH // H].double() @ qn[h]) / hd ** 0.5).softmax(0)
        want.append(p @ cv[:, h * KVH // H].double() * torch.sigmoid(q[h, 1].double()))
    want = torch.stack(want).reshape(-1)
    err = float((out.double() - want).norm() / want.norm())
    print(f"  error {err:.2e}", flush=True)
    assert err < 3e-7, err


def test_tiny_q4_model_entirely_on_the_device_matches_mlx():
    import torch
    from safetensors.numpy import load_file
    from swiftlet_amd.checkpoint import Checkpoint, moe_layer_from_checkpoint
    from swiftlet_amd.deltanet import deltanet_from_checkpoint
    from swiftlet_amd.engine import HipEngine
    eng = HipEngine()
    d = G / "tiny-model-q4"
    cfg = json.loads((d / "config.json").read_text())
    ck = Checkpoint(d)
    eps = cfg["rms_norm_eps"]
    fx = load_file(str(G / "tiny_forward_q4.safetensors"))
    toks = fx["input_ids"][0]
    S = len(toks)
    emb = ck.gpu_linear("model.embed_tokens")
    hd = torch.cat([eng.dequantize(emb, int(t), 1) for t in toks])
    interval = cfg["full_attention_interval"]
    for i in range(cfg["num_hidden_layers"]):
        p = f"model.layers.{i}."
        w_in = ck.load(p + "input_layernorm.weight")  # the input norm runs inside the projections' launch
        if (i + 1) % interval != 0:
            blk = deltanet_from_checkpoint(ck, i, cfg)
            state = blk.new_state()
            att = torch.stack([blk.forward_token(eng, hd[t], state, t, norm_weight=w_in, eps=eps) for t in range(S)])
        else:
            blk = attention_from_checkpoint(ck, i, cfg, max_positions=64)
            cache, ws = blk.new_cache(), blk.new_workspace()
            att = torch.stack([blk.forward_token(eng, hd[t], cache, ws, t, norm_weight=w_in, eps=eps)
                               for t in range(S)])
        x2 = eng.rms_norm(hd, ck.load(p + "post_attention_layernorm.weight"), eps, residual=att.contiguous())
        moe_layer_from_checkpoint(ck, i, cfg).decode(x2, out=hd, accumulate=True)
        torch.cuda.synchronize()
    hn = eng.rms_norm(hd, ck.load("model.norm.weight"), eps)
    head = ck.gpu_linear("lm_head")
    logits = torch.empty((S, head.out_dim), dtype=torch.float32, device="cuda")
    for t in range(S):
        eng.encode_gemv(head, hn[t], logits[t])
    torch.cuda.synchronize()
    got = logits.cpu().numpy()
    diff = np.abs(got - fx["logits"][0]).max()
    print(f"max |logit - mlx| = {diff:.3g}", flush=True)
    assert diff < 2e-3, diff
    want = json.loads((G / "tiny_forward_q4.json").read_text())["greedy_next_tokens"]
    assert np.argmax(got, axis=-1).tolist() == want
