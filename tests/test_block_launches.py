"""forward_token's one native call, and the launches one by one for programs that override them."""

import pytest

from swiftlet_amd import attention, deltanet, engine
from tests import fakes

BLOCKS = [(deltanet.DeltaNetGPU, "swq_deltanet"), (attention.AttentionGPU, "swq_attention")]


@pytest.fixture(autouse=True)
def fake(monkeypatch):
    f = fakes.FakeTorch()
    for m in (engine, deltanet, attention):
        monkeypatch.setattr(m, "_torch", lambda: f)
    return f


def _names(lib):
    return [n for n, _ in lib.calls]


def _one_by_one(prefix):
    return ["swq_encode_gemv_multi", prefix + "_step", "swq_encode_gemv"]


@pytest.mark.parametrize("cls,prefix", BLOCKS)
def test_one_native_call(cls, prefix):
    lib = fakes.FakeLib()
    _, token = fakes.block(cls, lib)
    token(fakes.hip_engine(lib))
    assert _names(lib) == [prefix + "_token"]


@pytest.mark.parametrize("cls,prefix", BLOCKS)
def test_overridden_step_is_called(cls, prefix):
    """In a subclass, on an instance, and with the class's own in its place again."""
    steps = []

    class Sub(cls):
        def step(self, *args, **kwargs):
            steps.append("subclass")
            return super().step(*args, **kwargs)

    lib = fakes.FakeLib()
    _, token = fakes.block(Sub, lib)
    token(fakes.hip_engine(lib))
    assert steps == ["subclass"] and _names(lib) == _one_by_one(prefix)

    lib = fakes.FakeLib()
    blk, token = fakes.block(cls, lib)
    blk.step = lambda *args, **kwargs: steps.append("instance") or cls.step(blk, *args, **kwargs)
    token(fakes.hip_engine(lib))
    assert steps[1:] == ["instance"] and _names(lib) == _one_by_one(prefix)
    del blk.step
    token(fakes.hip_engine(lib))
    assert _names(lib)[3:] == [prefix + "_token"]


@pytest.mark.parametrize("method", ["encode_gemv", "encode_gemv_multi"])
@pytest.mark.parametrize("cls,prefix", BLOCKS)
def test_overridden_engine_launch_is_called(cls, prefix, method, monkeypatch):
    """In a subclass, on an instance, and in the class itself."""
    seen = []
    own = getattr(engine.HipEngine, method)

    def counted(self, *args, **kwargs):
        seen.append(method)
        return own(self, *args, **kwargs)

    lib = fakes.FakeLib()
    _, token = fakes.block(cls, lib)
    sub = type("Sub", (engine.HipEngine,), {method: counted})
    token(fakes.hip_engine(lib, sub))
    inst = fakes.hip_engine(lib)
    setattr(inst, method, lambda *args, **kwargs: counted(inst, *args, **kwargs))
    token(inst)
    monkeypatch.setattr(engine.HipEngine, method, counted)
    token(fakes.hip_engine(lib))
    assert seen == [method] * 3 and _names(lib) == _one_by_one(prefix) * 3


@pytest.mark.parametrize("cls,prefix", BLOCKS)
def test_overridden_forward_token_runs_once(cls, prefix, fake):
    """Also where the base class runs itself again under the given stream."""
    calls = []

    class Sub(cls):
        def forward_token(self, *args, **kwargs):
            calls.append(1)
            return super().forward_token(*args, **kwargs)

    lib = fakes.FakeLib()
    _, token = fakes.block(Sub, lib)
    token(fakes.hip_engine(lib), fakes.SIDE)
    assert calls == [1] and lib.calls == [(prefix + "_token", "side")]
