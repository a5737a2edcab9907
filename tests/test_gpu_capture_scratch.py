"""Calls that want scratch while a stream is being captured: scratch is not allocated then. A call that cannot do without is
refused; a small column reduction and the unaligned transposed rows, which are split for speed alone, run in their form
without scratch - recorded on the captured stream, and eagerly beside it where the reservation is refused."""
import ctypes as C

import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL

pytestmark = pytest.mark.gpu

P = C.c_void_p
GLOBAL, THREAD_LOCAL, RELAXED = 0, 1, 2


@pytest.fixture()
def hip():
    h = C.CDLL("libamdhip64.so")
    h.hipStreamCreateWithFlags.argtypes = [C.POINTER(P), C.c_uint]
    h.hipStreamBeginCapture.argtypes = [P, C.c_int]
    h.hipStreamEndCapture.argtypes = [P, C.POINTER(P)]
    h.hipGraphInstantiate.argtypes = [C.POINTER(P), P, P, P, C.c_size_t]
    h.hipGraphLaunch.argtypes = [P, P]
    for f in (h.hipStreamSynchronize, h.hipGraphExecDestroy, h.hipGraphDestroy, h.hipStreamDestroy):
        f.argtypes = [P]
    return h


@pytest.fixture()
def streams(hpt, dev, hip):
    """Two streams of their own, not ordered with the default stream; no scratch has been reserved for any stream."""
    from hpt_amd import _ffi
    _ffi.check(hpt.lib().hpt_hip_cache_clear(dev))
    made = [P(), P()]
    for s in made:
        assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    yield made
    for s in made:
        hip.hipStreamDestroy(s)


def _mallocs_and_cached(hpt, dev):
    from hpt_amd import _ffi
    v = [C.c_uint64() for _ in range(3)]
    _ffi.check(hpt.lib().hpt_hip_alloc_stats(dev, *[C.byref(x) for x in v]))
    return v[2].value, v[1].value


def _cases(hpt, dev):
    """(name, call into a given output on a stream, output, expected) of the two kinds that have a form without scratch"""
    rng = np.random.default_rng(31)
    a = rng.integers(-99, 100, (12608, 128)).astype(np.int32)
    ta = hpt.Tensor.from_numpy(a).to_hip(dev)
    assert "split=1 " not in hpt.reduce_plan(ta, hpt.SUM, [0]) + " "
    x = rng.standard_normal((5003, 131)).astype(np.float32)
    tx = hpt.Tensor.from_numpy(x).to_hip(dev).permute([1, 0])
    assert hpt.normalize_plan(tx, 1).startswith("transposed-unaligned")
    oa, ox = hpt.Tensor.empty([128], hpt.i32, dev), hpt.Tensor.empty([131, 5003], hpt.f32, dev)
    e = np.exp(x.T.astype(np.float64))
    return [("sum", lambda st: ta.sum_([0], False, True, oa, stream=st), oa, a.sum(0, dtype=np.int32)),
            ("softmax", lambda st: tx.softmax(1, out=ox, stream=st), ox, (e / e.sum(1, keepdims=True)).astype(np.float32))]


def _check(got, want, what):
    if want.dtype == np.int32:
        assert np.array_equal(got, want), what
    else:
        assert_close(got, want, F32_RTOL, F32_ATOL, what)


@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL])
def test_scratch_is_not_allocated_for_a_recorded_call(hpt, dev, hip, streams, mode):
    from hpt_amd import _ffi
    x = np.random.default_rng(30).integers(-99, 100, (4096, 4096)).astype(np.int32)
    t, out = hpt.Tensor.from_numpy(x).to_hip(dev), hpt.Tensor.empty([1], hpt.i32, dev)
    kept = hpt.Tensor.empty([1234567], hpt.f32, dev)
    del kept  # a cached block: a refusal is no reason to give it up
    hpt.synchronize(dev)
    before = _mallocs_and_cached(hpt, dev)
    assert before[1] >= 1
    assert hip.hipStreamBeginCapture(streams[0], mode) == 0
    try:
        with pytest.raises(_ffi.HptError):
            t.sum_([0, 1], False, True, out, stream=streams[0])
    finally:
        graph = P()
        hip.hipStreamEndCapture(streams[0], C.byref(graph))
        hip.hipGetLastError()  # (the refusal may have ended the capture: the error of this test's own call)
    if graph.value:
        hip.hipGraphDestroy(graph)
    assert _mallocs_and_cached(hpt, dev) == before
    # (the runtime may leave the stream whose capture has failed unusable: another one)
    t.sum_([0, 1], False, True, out, stream=streams[1])
    assert hip.hipStreamSynchronize(streams[1]) == 0
    assert out.numpy()[0] == x.sum(), "the same call afterwards"


@pytest.mark.parametrize("mode", [GLOBAL, THREAD_LOCAL, RELAXED])
def test_forms_without_scratch_are_recorded(hpt, dev, hip, streams, mode):
    for name, call, out, want in _cases(hpt, dev):
        hpt.synchronize(dev)
        before = _mallocs_and_cached(hpt, dev)
        assert hip.hipStreamBeginCapture(streams[0], mode) == 0
        try:
            call(streams[0])
        finally:
            graph, gexec = P(), P()
            rc = hip.hipStreamEndCapture(streams[0], C.byref(graph))
        assert rc == 0 and graph.value, name
        assert _mallocs_and_cached(hpt, dev) == before, name
        assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
        for _ in range(3):
            assert hip.hipGraphLaunch(gexec, streams[0]) == 0 and hip.hipStreamSynchronize(streams[0]) == 0
            _check(out.numpy(), want, f"{name}, replayed")
            call(None)  # eagerly in between, the form with scratch
            _check(out.numpy(), want, f"{name}, eager")
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)


def test_forms_without_scratch_where_it_is_refused(hpt, dev, hip, streams):
    """While one stream is being captured, memory is refused to calls on another one too."""
    cases = _cases(hpt, dev)
    hpt.synchronize(dev)
    before = _mallocs_and_cached(hpt, dev)
    assert hip.hipStreamBeginCapture(streams[0], GLOBAL) == 0
    try:
        for _, call, _, _ in cases:
            call(streams[1])
    finally:
        graph = P()
        hip.hipStreamEndCapture(streams[0], C.byref(graph))
        hip.hipGetLastError()  # (the refusal may have ended the capture: the error of this test's own call)
    if graph.value:
        hip.hipGraphDestroy(graph)
    assert _mallocs_and_cached(hpt, dev) == before, "the reservation was meant to be refused"
    assert hip.hipStreamSynchronize(streams[1]) == 0
    for name, _, out, want in cases:
        _check(out.numpy(), want, name)
