"""Where hpt_amd._calls cannot be loaded (another interpreter, a tree in which only the library was built) every call goes through ctypes:
memory goes back to the allocator, and results and errors are the same."""
import ctypes as C
import sys
import warnings

import numpy as np
import pytest


@pytest.fixture
def without(hpt, monkeypatch):
    from hpt_amd import _ffi
    monkeypatch.setitem(sys.modules, "hpt_amd._calls", None)
    monkeypatch.delattr(hpt, "_calls", raising=False)
    monkeypatch.setattr(_ffi, "_calls", None)
    with pytest.warns(RuntimeWarning, match="_calls cannot be loaded"):
        assert _ffi.calls() is _ffi._ThroughCtypes
    return _ffi


@pytest.mark.parametrize("pending,entry", [({0}, "hpt_hip_free_ordered"), (set(), "hpt_hip_free"), ({0, 7}, "hpt_hip_free")])
def test_blocks_are_freed(without, monkeypatch, pending, entry):
    from hpt_amd import tensor
    calls = []

    class Lib:
        def __getattr__(self, name):
            return lambda *a: calls.append((name, *(x.value if isinstance(x, C.c_void_p) else x for x in a))) or 0

    monkeypatch.setattr(without, "lib", Lib)
    st = tensor._DeviceStorage.adopt(0, 4096, 640, 0)
    st.pending = set(pending)
    del st
    assert calls[-1] == (entry, 0, 4096, 640, tensor.ALIGN), calls


def test_the_warning_as_an_error(without):
    without._calls = None
    with pytest.raises(RuntimeWarning), warnings.catch_warnings():
        warnings.simplefilter("error")
        without.calls()
    assert without.calls() is without._ThroughCtypes


def test_errors(hpt, without):
    t = hpt.Tensor.from_raw(1 << 40, [4, 5, 6], hpt.f32)
    with pytest.raises(hpt.HptError, match="out of range"):
        t.sum([3])


@pytest.mark.gpu
def test_results_and_memory(hpt, dev, without):
    rng = np.random.default_rng(2)
    x = rng.standard_normal((64, 96)).astype(np.float32)
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    g = hpt.Tensor.from_numpy(np.ones(96, np.float32)).to_hip(dev)
    calls = (lambda: t.sum([0]), lambda: t.argmax(1, True), lambda: t.softmax(1), lambda: t.layernorm([96], g, g), lambda: t.add_layernorm(t, [96], g, g),
             lambda: t.softmax_causal(0.5, 32))
    got = [f().numpy().tobytes() for f in calls]

    def live():
        n = [C.c_uint64() for _ in range(3)]
        assert hpt.lib().hpt_hip_alloc_stats(dev, *(C.byref(u) for u in n)) == 0
        return n[0].value

    before = live()
    for f in calls:
        f()
    assert live() == before  # nothing of theirs stays allocated
    without._calls = None
    del sys.modules["hpt_amd._calls"]
    assert without.calls() is not without._ThroughCtypes
    assert [f().numpy().tobytes() for f in calls] == got


def test_build_without_a_compiler(monkeypatch, tmp_path, capsys):
    from hpt_amd import build
    monkeypatch.setattr(build, "CALLS", tmp_path / "_calls.so")
    monkeypatch.setenv("CXX", str(tmp_path / "no-such-compiler"))
    assert build.build_calls(force=True) is None and not build.CALLS.exists()
    assert "calls go through ctypes" in capsys.readouterr().err
