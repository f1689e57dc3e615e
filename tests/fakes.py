"""Stand-ins for torch and the library that record what a call allocates and which entry points
it takes, for tests of the Python layer without a device."""

import contextlib
import types

from swiftlet_amd import attention, deltanet, engine

SIDE = types.SimpleNamespace(cuda_stream="side")  # a stream that is not the current one


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
        return tensor(n, dtype)


class FakeLib:
    """Every entry returns success; `calls` holds the names of those that launch and the last
    argument, the stream, of each."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            if name.endswith(("_floats", "_bytes")):
                return 64
            self.calls.append((name, args[-1]))
            return 0
        return call


def tensor(n=64, dtype="f32"):
    return types.SimpleNamespace(data_ptr=lambda: 0x3000, device="cuda", dtype=dtype, numel=lambda: n)


def linear():
    return engine.GPULinear(tensor(), tensor(), tensor(), 64, 64, 64, 4, 0)


def hip_engine(lib, cls=engine.HipEngine):
    eng = cls.__new__(cls)
    eng.lib = lib
    return eng


def block(cls, lib):
    """A DeltaNetGPU or AttentionGPU (or a subclass's) of the stand-ins, and its forward_token as a
    function of the engine and the stream."""
    blk = cls.__new__(cls)
    delta = issubclass(cls, deltanet.DeltaNetGPU)
    blk._c = deltanet.DeltaNetLayer() if delta else attention.AttentionLayer()
    blk.lib, blk._projs, blk._scratch = lib, engine.DescArray(), 64
    blk.layout, blk.conv_dim, blk.value_dim, blk.nv, blk.H, blk.hd = 0, 4, 4, 1, 1, 16
    blk.projections = (linear(),) * (4 if delta else 3)
    blk.out_proj = blk.o_proj = linear()
    t = tensor()
    state = (t,) if delta else (t, t)
    return blk, lambda eng, stream=None: blk.forward_token(eng, t, *state, 0, stream=stream)
