"""Ragged MoE prefill on the device (swq_moe_prefill) against the oracle
(QwenCPUModel.moeForward for S tokens, QwenCPUModel.swift:500-569), at the
benchmark shapes, at odd shapes, and at the 512-token skewed-load workload.

Bar: expert ids equal the oracle's wherever the router's k-th/(k+1)-th
logit gap exceeds 1e-3; combine weights within 1e-5; layer output within
1e-3 relative L2 of the f32 oracle, and within 1e-5 (fp32 accumulation on
exact bf16 operands: the observed error is ~1e-6).  At 512 tokens the oracle
runs on a sample of tokens, and size-independent properties cover the rest:
each token's row is the same bit for bit whatever other tokens share the
call (rows never mix in the matrix cores), and repeated calls agree."""

import numpy as np
import pytest

from oracle import moe_ref as R
from swiftlet_amd import moe, synth
from tests import helpers

pytestmark = pytest.mark.gpu

REL_L2_BAR = 1e-3
TIGHT = 1e-5
MARGIN = 1e-3
ZIPF_SEED = 2024


def _x(seed, T, H, dtype="bf16"):
    import torch
    xb = synth.activations_bf16(seed, T, H)
    xf = synth.bf16_to_f32(xb)
    x = helpers.bf16_bits_to_torch(xb) if dtype == "bf16" else torch.from_numpy(xf).cuda()
    return x, xf


def _check(shape, xf, out, ids, w, rows=None, seed=helpers.SEED, layer=0, bias=None, ref_layer=None):
    """Compare rows `rows` (default all) of a prefill result with the oracle."""
    import torch
    rows = np.arange(xf.shape[0]) if rows is None else np.asarray(rows)
    ref_layer = ref_layer or helpers.ref_layer(shape, seed, layer)
    ref_out, picks, ref_w = R.moe_forward(xf[rows], ref_layer, logit_bias=bias)
    margin = R.router_margin(xf[rows], ref_layer, logit_bias=bias)
    checked = 0
    for i, t in enumerate(rows):
        if margin[i] > MARGIN:
            assert list(ids[t]) == [e for e, _ in picks[i]], (t, ids[t], picks[i])
            assert np.allclose(w[t], ref_w[i], rtol=1e-5, atol=1e-7), t
            checked += 1
    assert checked >= len(rows) - 1  # margins below 1e-3 are rare at these shapes
    if out.dtype == torch.bfloat16:
        got = R.bf16_bits_to_f32(helpers.torch_bf16_to_bits(out))[rows]
        # each element is the bf16 rounding of an f32 value within 1e-5 rms of the oracle's
        ulp = np.exp2(np.floor(np.log2(np.maximum(np.abs(ref_out), 1e-30))) - 7)
        rms = np.sqrt(np.mean(ref_out.astype(np.float64) ** 2))
        assert np.all(np.abs(got - ref_out) <= ulp + TIGHT * rms)
        assert R.rel_l2(got, R.bf16_bits_to_f32(R.f32_to_bf16_bits_rne(ref_out))) < REL_L2_BAR
    else:
        err = R.rel_l2(out.cpu().numpy()[rows], ref_out)
        print(f"rel_l2 vs oracle: {err:.3g}", flush=True)
        assert err < REL_L2_BAR, err
        assert err < TIGHT, err


@pytest.mark.parametrize("name,T,rows", [
    ("qwen3.6-35b-a3b-q4", 64, [0, 17, 40, 63]),
    ("qwen3-next-80b-a3b-q4", 40, [1, 22, 39]),
    ("qwen3.6-35b-a3b-q8", 33, [0, 16, 32]),
])
def test_prefill_matches_oracle(name, T, rows):
    import torch
    shape = synth.SHAPES[name]
    print(f"prefill vs oracle: {name} T={T}", flush=True)
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    x, xf = _x(helpers.SEED + 500 + T, T, shape.hidden)
    out, ids, w = gpu.prefill(x)
    torch.cuda.synchronize()
    _check(shape, xf, out, ids.cpu().numpy(), w.cpu().numpy(), rows=rows)


@pytest.mark.parametrize("E,K,I,Is,H,bits,norm,T", [
    (8, 2, 128, 128, 128, 4, True, 50),       # few experts: long tiles
    (60, 4, 128, 256, 256, 8, False, 70),     # E not a multiple of 16; Is != I; no renorm
    (1024, 16, 128, 128, 128, 4, True, 20),   # widest top-k table: mostly 1-row tiles
    (128, 1, 256, 128, 384, 4, True, 130),    # top-1; 6 groups per row
])
def test_prefill_odd_shapes(E, K, I, Is, H, bits, norm, T):
    import torch
    shape = synth.MoEShape("odd", H, E, K, I, Is, expert_bits=bits, router_bits=8, group=64,
                           norm_topk_prob=norm)
    print(f"prefill odd: E={E} K={K} I={I} Is={Is} H={H} q{bits} T={T}", flush=True)
    gpu = moe.synth_layer(shape, 77, 0)
    x, xf = _x(78, T, H)
    out, ids, w = gpu.prefill(x)
    torch.cuda.synchronize()
    _check(shape, xf, out, ids.cpu().numpy(), w.cpu().numpy(), seed=77)


def test_prefill_without_shared_expert():
    """has_shared = 0: no shared tiles, no shared-gate logit (QwenCPUModel.swift:559-566)."""
    import torch
    shape = synth.MoEShape("no-shared", 2048, 256, 8, 512, 0, 4)
    print("prefill without a shared expert, T=24", flush=True)
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    x, xf = _x(helpers.SEED + 77, 24, shape.hidden)
    out, ids, w = gpu.prefill(x)
    torch.cuda.synchronize()
    _check(shape, xf, out, ids.cpu().numpy(), w.cpu().numpy(), rows=[0, 11, 23])


@pytest.mark.parametrize("T", [1, 7, 100])
def test_prefill_single_expert_layer(T):
    """One routed expert and no shared expert (the single-expert workload): a
    one-column router, every pair on expert 0 with weight 1, and tiles of one
    expert over all the tokens."""
    import torch
    shape = synth.SHAPES["single-expert-q4"]
    print(f"prefill of the single-expert layer, T={T}", flush=True)
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    x, xf = _x(helpers.SEED + 5 + T, T, shape.hidden)
    out, ids, w = gpu.prefill(x)
    torch.cuda.synchronize()
    assert (ids.cpu().numpy() == 0).all() and (w.cpu().numpy() == 1.0).all()
    _check(shape, xf, out, ids.cpu().numpy(), w.cpu().numpy())


def test_prefill_f32_x_bf16_out():
    import torch
    shape = synth.SHAPES["qwen3.6-35b-a3b-q4"]
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    x, xf = _x(helpers.SEED + 9, 24, shape.hidden, dtype="f32")
    out, ids, w = gpu.prefill(x, out_dtype=torch.bfloat16)
    torch.cuda.synchronize()
    _check(shape, xf, out, ids.cpu().numpy(), w.cpu().numpy(), rows=[0, 11, 23])


def test_prefill_skewed_512_tokens():
    """The benchmark workload: 512 tokens, Zipf(1.1)-skewed expert load.
    Routing checked for every token, and every row whose k-th / (k+1)-th
    logit gap exceeds 1e-3 (510 of the 512) against the oracle; rows also
    equal those of a smaller call holding only some of the tokens.  The
    oracle's pass over the rows takes ~15 s on one core."""
    import torch
    shape = synth.SHAPES["qwen3.6-35b-a3b-q4"]
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    bias = synth.zipf_logit_bias(ZIPF_SEED, shape.experts)
    bias_t = torch.from_numpy(bias).cuda()
    x, xf = _x(helpers.SEED + 4242, 512, shape.hidden)
    ws = gpu.new_prefill_workspace(512)
    out, ids, w = gpu.prefill(x, ws=ws, logit_bias=bias_t)
    out, ids, w = out.clone(), ids.clone(), w.clone()
    torch.cuda.synchronize()
    ids_np, w_np = ids.cpu().numpy(), w.cpu().numpy()
    counts = np.bincount(ids_np.ravel(), minlength=shape.experts)
    assert counts.sum() == 512 * 8 and counts.max() <= 512
    assert counts.max() > 200  # skewed: the top expert takes a large share
    ref_layer = helpers.ref_layer(shape, helpers.SEED, 0)
    # routing of every token
    logits = xf @ ref_layer.router_dense.T + bias
    margin = R.router_margin(xf, ref_layer, logit_bias=bias)
    for t in range(512):
        if margin[t] > MARGIN:
            p = R.softmax_row(logits[t].astype(np.float32))
            picks = R.topk_insertion(p, 8)
            assert list(ids_np[t]) == [e for e, _ in picks], t
    # outputs of every margin-safe row
    safe = [t for t in range(512) if margin[t] > MARGIN]
    assert len(safe) >= 500
    print(f"oracle over {len(safe)} rows", flush=True)
    _check(shape, xf, out, ids_np, w_np, rows=safe, bias=bias, ref_layer=ref_layer)
    # repeat: identical
    out2, ids2, w2 = gpu.prefill(x, ws=ws, logit_bias=bias_t)
    torch.cuda.synchronize()
    assert torch.equal(out, out2) and torch.equal(ids, ids2) and torch.equal(w, w2)
    # each row equals the row of a call that holds only some of the tokens
    sub = [3, 100, 511, 7]
    o_sub, i_sub, w_sub = gpu.prefill(x[sub].contiguous(), logit_bias=bias_t)
    torch.cuda.synchronize()
    assert torch.equal(o_sub, out[sub]) and torch.equal(i_sub, ids[sub]) and torch.equal(w_sub, w[sub])


def test_prefill_matches_decode():
    """A token's prefill row against the decode step on that token alone:
    the same routing and, both within 1e-5 of the oracle, outputs within 2e-5."""
    import torch
    shape = synth.SHAPES["qwen3.6-35b-a3b-q4"]
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    x, xf = _x(helpers.SEED + 31, 12, shape.hidden)
    out, ids, w = gpu.prefill(x)
    ws = gpu.new_workspace(1)
    margin = R.router_margin(xf, helpers.ref_layer(shape, helpers.SEED, 0))
    for t in range(12):
        od, idd, wd = gpu.decode(x[t:t + 1], ws=ws)
        torch.cuda.synchronize()
        if margin[t] > MARGIN:
            assert torch.equal(idd[0], ids[t]), t
            assert torch.allclose(wd[0], w[t], rtol=1e-5, atol=1e-7), t
            # each path is within TIGHT of the oracle
            assert R.rel_l2(out[t].cpu().numpy(), od[0].cpu().numpy()) < 2 * TIGHT, t


def test_prefill_accumulate():
    import torch
    shape = synth.SHAPES["qwen3.6-35b-a3b-q4"]
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    x, _ = _x(5, 40, shape.hidden)
    ws = gpu.new_prefill_workspace(40)
    o1, _, _ = gpu.prefill(x, ws=ws)
    o1 = o1.clone()
    resid = torch.randn_like(o1)
    acc = resid.clone()
    gpu.prefill(x, out=acc, ws=ws, accumulate=True)
    torch.cuda.synchronize()
    assert torch.allclose(acc, resid + o1, rtol=0, atol=1e-5)


def test_prefill_single_token_and_workspace_reuse():
    """T = 1, then larger calls on a workspace sized for the largest: the
    counters the grouping leaves at zero serve every later call."""
    import torch
    shape = synth.SHAPES["qwen3.6-35b-a3b-q4"]
    gpu = moe.synth_layer(shape, helpers.SEED, 0)
    ws = gpu.new_prefill_workspace(96)
    for T in (1, 96, 17, 1):
        x, xf = _x(900 + T, T, shape.hidden)
        out, ids, w = gpu.prefill(x, ws=ws)
        fresh, ids_f, w_f = gpu.prefill(x)
        torch.cuda.synchronize()
        assert torch.equal(out, fresh) and torch.equal(ids, ids_f) and torch.equal(w, w_f), T
    _check(shape, xf, out, ids.cpu().numpy(), w.cpu().numpy())


@pytest.mark.parametrize("name,x_dtype", [
    ("qwen3.6-35b-a3b-q4", "bf16"),
    ("qwen3.6-35b-a3b-q4", "f32"),
    ("qwen3.6-35b-a3b-q8", "bf16"),
])
def test_prefill_f32_scales_equal_f16_scales(name, x_dtype):
    """f32 scales and biases (exact widenings of the fp16 ones) take the
    GEMMs' 4-byte-scale kernels: the same outputs, ids and weights bit for
    bit as the fp16 layer."""
    import torch
    print(f"prefill f32 scales vs f16: {name} x {x_dtype}", flush=True)
    shape = synth.SHAPES[name]
    a = moe.synth_layer(shape, helpers.SEED, 0)
    b = helpers.widen_layer(a)
    x, _ = _x(4242, 40, shape.hidden, x_dtype)
    oa, ia, wa = a.prefill(x)
    ob, ib, wb = b.prefill(x)
    torch.cuda.synchronize()
    assert torch.equal(ia, ib) and torch.equal(wa, wb) and torch.equal(oa, ob)


def test_prefill_router_scales_two_bytes_past_a_word():
    """2-byte router scales and biases that start 2 bytes past a 4-byte
    boundary (a layer swq_moe_decode takes) give the same prefill, bit for
    bit, as the same values on aligned words."""
    import torch
    from swiftlet_amd.engine import GPULinear
    shape = synth.SHAPES["qwen3.6-35b-a3b-q4"]
    layer = moe.synth_layer(shape, helpers.SEED, 0)
    x, _ = _x(helpers.SEED + 90, 24, shape.hidden)
    ref_out, ref_ids, ref_w = layer.prefill(x)
    r = layer.router

    def shifted(t):
        buf = torch.zeros(t.numel() + 8, dtype=torch.uint8, device=t.device)
        buf[2:2 + t.numel()].copy_(t)
        return buf

    r2 = GPULinear(r.w, shifted(r.scales), shifted(r.biases), r.out_dim, r.in_dim, r.group_size, r.bits,
                   r.scales_type, w_off=r.w_off, s_off=r.s_off + 2, b_off=r.b_off + 2)
    assert (r2.scales.data_ptr() + r2.s_off) % 4 == 2
    layer2 = moe.MoELayerGPU(r2, layer.gate, layer.up, layer.down, layer.shared_gate, layer.shared_up,
                             layer.shared_down, layer.shared_expert_gate, layer.top_k, layer.norm_topk_prob)
    out, ids, w = layer2.prefill(x)
    torch.cuda.synchronize()
    assert torch.equal(ids, ref_ids)
    assert torch.equal(w, ref_w)
    assert torch.equal(out, ref_out)


@pytest.mark.parametrize("H,I,Is,bits,x_dtype,f32_scales", [
    (2048, 512, 512, 4, "bf16", False), (384, 384, 128, 4, "bf16", False), (128, 640, 256, 4, "f32", False),
    (640, 128, 384, 8, "bf16", False), (256, 896, 0, 8, "f32", False), (384, 256, 128, 4, "bf16", True),
    (256, 384, 128, 8, "f32", True), (128, 128, 128, 4, "bf16", True), (2048, 256, 128, 4, "bf16", True)])
def test_few_tokens_equal_many(H, I, Is, bits, x_dtype, f32_scales):
    """The GEMM over 16-row tiles (up to six tokens per expert on average: 90 tokens of 60 experts,
    top 4) gives the bits of the one over 64-row tiles: the rows of calls of 1, 8, 9, 16, 17 and 90
    tokens equal those of a call of 91.  Group counts that fill its stages and ones that do not
    (6, 10, 14 groups), both activation forms, 2- and 4-byte scales; 4-byte ones with 2, 6 and 32
    groups under the 64-row kernel's deeper ring."""
    import torch
    shape = synth.MoEShape("few", H, 60, 4, I, Is, expert_bits=bits, router_bits=8, group=64, norm_topk_prob=True)
    gpu = moe.synth_layer(shape, 4000 + H + I, 0)
    if f32_scales:
        gpu = helpers.widen_layer(gpu)
    x, _ = _x(77 + H, 91, H)
    if x_dtype == "f32":
        x = x.float() * 1.1
    print(f"few tokens: H {H} I {I} Is {Is} q{bits} x {x_dtype} f32 scales {f32_scales}", flush=True)
    want, want_ids, want_w = gpu.prefill(x)
    for T in (1, 8, 9, 16, 17, 90):
        out, ids, w = gpu.prefill(x[:T].contiguous())
        torch.cuda.synchronize()
        assert torch.equal(ids, want_ids[:T]) and torch.equal(w, want_w[:T]) and torch.equal(out, want[:T]), T


@pytest.mark.parametrize("I,x_dtype", [(128, "bf16"), (128, "f32"), (256, "f32"), (256, "bf16")])
def test_short_down_rows_equal_on_either_side(I, x_dtype):
    """Where down's rows fit one stage of the 16-row kernel's ring the tiles change size at 1,536 pairs
    already (but for 256 inputs with bf16 x, at six rows per expert): 192 tokens of top 8 have those
    tiles, 193 the 64-row ones, 390 and 391 stand on the other line, and every row has the same bits."""
    import torch
    shape = synth.MoEShape("short", 256, 520, 8, I, 128, expert_bits=4, router_bits=8, group=64, norm_topk_prob=True)
    gpu = moe.synth_layer(shape, 4400 + I, 0)
    x, _ = _x(78 + I, 391, 256)
    if x_dtype == "f32":
        x = x.float() * 1.1
    print(f"short down rows: I {I} x {x_dtype}", flush=True)
    ws = gpu.new_prefill_workspace(391)
    want, want_ids, want_w = gpu.prefill(x, ws=ws)
    for T in (191, 192, 193, 390):
        out, ids, w = gpu.prefill(x[:T].contiguous(), ws=ws)
        torch.cuda.synchronize()
        assert torch.equal(ids, want_ids[:T]) and torch.equal(w, want_w[:T]) and torch.equal(out, want[:T]), T


@pytest.mark.parametrize("E,K,T,x_dtype", [(60, 9, 911, "bf16"), (256, 8, 1024, "f32"), (256, 8, 1025, "bf16"),
                                           (513, 5, 2049, "bf16"), (256, 8, 3073, "bf16"), (520, 16, 1311, "f32")])
def test_many_tokens_equal_few(E, K, T, x_dtype):
    """The router's 32-token tiles (from 1,024 tokens) and the grouping over several workgroups
    (from 8,193 pairs): routing and outputs of every token equal, bit for bit, those of calls of at most 500 of the
    tokens, which take none of them.  The expert loads are skewed; the pairs of the last share and
    the last tiles are ragged."""
    import torch
    shape = synth.MoEShape("many", 512, E, K, 128, 128, expert_bits=4, router_bits=8, group=64, norm_topk_prob=True)
    gpu = moe.synth_layer(shape, 5000 + E, 0)
    bias = torch.from_numpy(synth.zipf_logit_bias(ZIPF_SEED, E)).cuda()
    x, _ = _x(31 + T, T, 512)
    if x_dtype == "f32":
        x = x.float() * 1.1
    print(f"many tokens: E {E} K {K} T {T} x {x_dtype}", flush=True)
    ws = gpu.new_prefill_workspace(T)
    for _ in range(2):
        out, ids, w = gpu.prefill(x, ws=ws, logit_bias=bias)
        for lo in range(0, T, 500):
            o, i, ww = gpu.prefill(x[lo:lo + 500].contiguous(), logit_bias=bias)
            torch.cuda.synchronize()
            n = o.shape[0]
            assert torch.equal(i, ids[lo:lo + n]) and torch.equal(ww, w[lo:lo + n]) and torch.equal(o, out[lo:lo + n]), lo
