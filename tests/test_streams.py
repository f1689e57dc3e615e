"""Calls that are given a stream: what they allocate for themselves belongs to that stream.

Without a device, on stand-ins for torch and the library that record which stream is current at
each allocation; on a device, against the call on the current stream while that stream allocates
and overwrites blocks of the same size."""

import contextlib
import types

import pytest

from swiftlet_amd import attention, deltanet, engine, moe


class FakeTorch:
    """empty() and the current stream of torch; `log` holds the stream of each allocation."""

    float32, bfloat16, int32, uint8 = "f32", "bf16", "i32", "u8"

    def __init__(self):
        self.current, self.log = types.SimpleNamespace(cuda_stream="default"), []
        self.cuda = types.SimpleNamespace(current_stream=lambda: self.current, stream=self._stream,
                                          current_device=lambda: 0)
        self._C = types.SimpleNamespace(_cuda_getCurrentRawStream=lambda device: self.current.cuda_stream)

    @contextlib.contextmanager
    def _stream(self, s):
        before, self.current = self.current, s
        yield
        self.current = before

    def empty(self, n, dtype=None, device=None):
        self.log.append(self.current.cuda_stream)
        return types.SimpleNamespace(data_ptr=lambda: 0x1000, dtype=dtype, numel=lambda: n)


class FakeLib:
    """Every entry returns success; `streams` holds the last argument of the token and prefill calls."""

    def __init__(self):
        self.streams = []

    def __getattr__(self, name):
        def call(*args):
            if name.endswith(("_token", "_prefill")):
                self.streams.append(args[-1])
            return 64 if name.endswith(("_floats", "_bytes")) else 0
        return call


def _lin():
    t = types.SimpleNamespace(data_ptr=lambda: 0x2000)
    return engine.GPULinear(t, t, t, 64, 64, 64, 4, 0)


def _block(cls, **fields):
    blk = cls.__new__(cls)
    blk._c = (deltanet.DeltaNetLayer if cls is deltanet.DeltaNetGPU else attention.AttentionLayer)()
    blk.lib, blk._projs, blk._scratch = FakeLib(), engine.DescArray(), 64
    for k, v in fields.items():
        setattr(blk, k, v)
    return blk


@pytest.mark.parametrize("kind", ["delta", "attention"])
def test_token_scratch_is_allocated_on_the_given_stream(kind, monkeypatch):
    fake = FakeTorch()
    for m in (engine, deltanet, attention):
        monkeypatch.setattr(m, "_torch", lambda: fake)
    eng = engine.HipEngine.__new__(engine.HipEngine)
    buf = types.SimpleNamespace(data_ptr=lambda: 0x3000, device="cuda", numel=lambda: 64, dtype="f32")
    if kind == "delta":
        blk = _block(deltanet.DeltaNetGPU, projections=(_lin(),) * 4, out_proj=_lin())
        call = lambda s: blk.forward_token(eng, buf, buf, 0, stream=s)  # noqa: E731
    else:
        blk = _block(attention.AttentionGPU, projections=(_lin(),) * 3, o_proj=_lin())
        call = lambda s: blk.forward_token(eng, buf, buf, buf, 0, stream=s)  # noqa: E731
    call(None)
    assert fake.log == ["default"] * 2 and blk.lib.streams == ["default"]
    call(types.SimpleNamespace(cuda_stream="side"))
    assert fake.log == ["default"] * 2 + ["side"] * 2 and blk.lib.streams == ["default", "side"]
    assert fake.current.cuda_stream == "default"


def test_prefill_workspace_is_allocated_on_the_given_stream(monkeypatch):
    """A prefill without a workspace makes one and lets go of it on return."""
    fake = FakeTorch()
    for m in (engine, moe):
        monkeypatch.setattr(m, "_torch", lambda: fake)
    layer = moe.MoELayerGPU.__new__(moe.MoELayerGPU)
    layer._c, layer.lib, layer.router, layer.hidden, layer.top_k = moe.MoELayer(), FakeLib(), _lin(), 64, 2
    layer.router.w.device = "cuda"
    buf = types.SimpleNamespace(data_ptr=lambda: 0x3000, device="cuda", dtype="f32", shape=(1, 64), dim=lambda: 2)
    given = dict(out=buf, topk_ids=buf, topk_weights=buf)
    layer.prefill(buf, **given)
    assert fake.log == ["default"] and layer.lib.streams == ["default"]
    layer.prefill(buf, stream=types.SimpleNamespace(cuda_stream="side"), **given)
    assert fake.log == ["default", "side"] and layer.lib.streams == ["default", "side"]


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
