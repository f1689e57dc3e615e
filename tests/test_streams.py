"""Calls that are given a stream: what they allocate for themselves belongs to that stream.

Without a device, on stand-ins for torch and the library that record which stream is current at
each allocation; on a device, against the call on the current stream while that stream allocates
and overwrites blocks of the same size."""

import pytest

from swiftlet_amd import attention, deltanet, engine, moe
from tests import fakes


@pytest.fixture
def fake(monkeypatch):
    f = fakes.FakeTorch()
    for m in (engine, deltanet, attention, moe):
        monkeypatch.setattr(m, "_torch", lambda: f)
    return f


@pytest.mark.parametrize("cls,entry", [(deltanet.DeltaNetGPU, "swq_deltanet_token"),
                                       (attention.AttentionGPU, "swq_attention_token")])
def test_token_scratch_is_allocated_on_the_given_stream(fake, cls, entry):
    lib = fakes.FakeLib()
    _, token = fakes.block(cls, lib)
    eng = fakes.hip_engine(lib)
    token(eng)
    assert fake.log == ["default"] * 2 and lib.calls == [(entry, "default")]
    token(eng, fakes.SIDE)
    assert fake.log == ["default"] * 2 + ["side"] * 2 and lib.calls[1:] == [(entry, "side")]
    assert fake.current.cuda_stream == "default"


def test_prefill_workspace_is_allocated_on_the_given_stream(fake):
    """A prefill without a workspace makes one and lets go of it on return."""
    layer = moe.MoELayerGPU.__new__(moe.MoELayerGPU)
    lib = fakes.FakeLib()
    layer._c, layer.lib, layer.router, layer.hidden, layer.top_k = moe.MoELayer(), lib, fakes.linear(), 64, 2
    buf = fakes.tensor()
    buf.shape, buf.dim = (1, 64), lambda: 2
    given = dict(out=buf, topk_ids=buf, topk_weights=buf)
    layer.prefill(buf, **given)
    layer.prefill(buf, stream=fakes.SIDE, **given)
    assert fake.log == ["default", "side"]
    assert lib.calls == [(n, s) for s in ("default", "side") for n in ("swq_moe_workspace_init", "swq_moe_prefill")]


def test_current_stream_without_torchs_private_entry(fake):
    """The raw current stream where this torch lacks the entry that returns it directly."""
    assert engine._stream_handle(None) == "default"
    del fake._C._cuda_getCurrentRawStream
    assert engine._stream_handle(None) == "default" and engine._stream_handle(fakes.SIDE) == "side"


@pytest.mark.gpu
def test_token_on_a_side_stream_while_the_current_one_reuses_memory():
    """Both blocks on a side stream that is still busy when the call returns, while the current
    stream takes blocks of the scratch's sizes and fills them with NaN for as long as the side
    stream works: the results are those of the current stream alone."""
    import torch
    from swiftlet_amd._lib import SWQ_DELTA_SPLIT
    from swiftlet_amd.moe import synth_linear
    eng = engine.HipEngine()
    g = torch.Generator(device="cuda").manual_seed(5)
    r = lambda *s: torch.randn(s, generator=g, device="cuda")  # noqa: E731
    lin = lambda seed, rows, cols: synth_linear(seed, 0, "router", None, rows, cols, 4, 64)  # noqa: E731
    nk, nv, dk, dv, K, H = 2, 4, 16, 32, 4, 256
    conv, val = 2 * nk * dk + nv * dv, nv * dv
    delta = deltanet.DeltaNetGPU(nk, nv, dk, dv, K, SWQ_DELTA_SPLIT, 1e-6, r(conv * K), r(nv), r(nv), r(dv),
                                 projections=[lin(i, n, H) for i, n in enumerate((conv, val, nv, nv))],
                                 out_proj=lin(9, H, val))
    heads, kvh, hd = 4, 2, 32
    att = attention.AttentionGPU(heads, kvh, hd, 8, 1e4, 1e-6, 40, r(hd), r(hd),
                                 projections=[lin(20 + i, n, H) for i, n in enumerate((2 * heads * hd, kvh * hd, kvh * hd))],
                                 o_proj=lin(30, H, heads * hd))
    x, ws = r(H), att.new_workspace()
    busy = r(2048, 2048)
    side = torch.cuda.Stream()
    for name, call, new in (("delta", lambda st, s: delta.forward_token(eng, x, st, 3, stream=s), delta.new_state),
                            ("attention", lambda st, s: att.forward_token(eng, x, st, ws, 0, stream=s), att.new_cache)):
        a, b = new(), new()
        want = call(a, None)
        n = delta._scratch if name == "delta" else att.lib.swq_attention_scratch_floats(
            engine.ctypes.byref(att._c), att._projs.of(att.projections))
        torch.cuda.synchronize()
        print(f"side stream: {name}", flush=True)
        with torch.cuda.stream(side):
            for _ in range(20):
                busy @ busy
        got = call(b, side)
        done = side.record_event()
        fills = 0
        while not done.query() and fills < 100000:
            for m in (n, H):
                torch.full((m,), float("nan"), device="cuda")
            fills += 1
        torch.cuda.synchronize()
        assert fills > 0 and torch.equal(got, want) and torch.equal(a, b), name
