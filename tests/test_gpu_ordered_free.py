"""Results that only the default stream has used are freed without a wait: the block may be handed out again while work
that uses it is queued, to calls on the same stream at once and to anybody else only when that work is over."""
import ctypes as C
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

P = C.c_void_p


@pytest.fixture()
def hip():
    h = C.CDLL("libamdhip64.so")
    h.hipStreamCreateWithFlags.argtypes = [C.POINTER(P), C.c_uint]
    h.hipStreamBeginCapture.argtypes = [P, C.c_int]
    h.hipStreamEndCapture.argtypes = [P, C.POINTER(P)]
    h.hipGraphInstantiate.argtypes = [C.POINTER(P), P, P, P, C.c_size_t]
    h.hipGraphLaunch.argtypes = [P, P]
    for f in (h.hipStreamQuery, h.hipStreamSynchronize, h.hipGraphExecDestroy, h.hipGraphDestroy, h.hipStreamDestroy):
        f.argtypes = [P]
    return h


def _blocks(hpt, dev):
    from hpt_amd import _ffi
    v = [C.c_uint64() for _ in range(3)]
    _ffi.check(hpt.lib().hpt_hip_alloc_stats(dev, *[C.byref(x) for x in v]))
    return [x.value for x in v]


def _busy(hpt, dev):
    """Half a millisecond of work queued on the default stream; returns what has to stay alive meanwhile."""
    big = hpt.Tensor.empty([1 << 27], hpt.f32, dev)
    for _ in range(8):
        big.add_(big, out=big)
    return big


def test_blocks_handed_on(hpt, dev, hip):
    from hpt_amd import _ffi
    l, n = hpt.lib(), 12345 * 64
    p, q, r = P(), P(), P()
    _ffi.check(l.hpt_hip_cache_clear(dev))
    _ffi.check(l.hpt_hip_alloc_ordered(dev, n, 64, C.byref(p)))
    keep = _busy(hpt, dev)
    _ffi.check(l.hpt_hip_free_ordered(dev, p, n, 64))
    _ffi.check(l.hpt_hip_alloc_ordered(dev, n, 64, C.byref(q)))
    assert q.value == p.value  # at once, whatever the stream is doing
    _ffi.check(l.hpt_hip_free_ordered(dev, q, n, 64))
    _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(r)))
    assert hip.hipStreamQuery(None) == 0, "an ordinary allocation was handed a block that is still in use"
    assert r.value == p.value
    _ffi.check(l.hpt_hip_free(dev, r, n, 64))
    # an idle block is preferred to waiting
    _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(r)))
    _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(p)))
    _ffi.check(l.hpt_hip_free(dev, p, n, 64))
    keep.add_(keep, out=keep)
    _ffi.check(l.hpt_hip_free_ordered(dev, r, n, 64))
    _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(q)))
    assert q.value == p.value
    _ffi.check(l.hpt_hip_free(dev, q, n, 64))
    for bad in (lambda: l.hpt_hip_alloc_ordered(dev, n, 48, C.byref(q)), lambda: l.hpt_hip_alloc_ordered(99, n, 64, C.byref(q)),
                lambda: l.hpt_hip_free_ordered(dev, P(64), n, 64)):
        with pytest.raises(_ffi.HptError):
            _ffi.check(bad())
    _ffi.check(l.hpt_hip_cache_clear(dev))
    assert _blocks(hpt, dev)[1] == 0


def test_results_dropped_in_flight(hpt, orc, dev, hip):
    """A loop whose results are dropped at once, calls on a stream of the caller's between them, and a second thread."""
    rng = np.random.default_rng(8)
    a, b = (rng.integers(-1000, 1000, (512, 3000)).astype(np.int32) for _ in range(2))
    ta, tb = hpt.Tensor.from_numpy(a).to_hip(dev), hpt.Tensor.from_numpy(b).to_hip(dev)
    hpt.synchronize(dev)
    s = P()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
    bad = []

    def loop(stream):
        for k in range(20):
            keep = _busy(hpt, dev) if stream is None and k % 5 == 0 else None
            x = ta.add(tb, stream=stream)
            y = x.sub(tb, stream=stream)
            del x  # its block is the next result's
            z = y.add(ta, stream=stream)
            got = z.sum([1], stream=stream).numpy()
            if not np.array_equal(got, (2 * a).sum(1, dtype=np.int32)) or not np.array_equal(y.numpy(), a):
                bad.append((stream, k))
            del keep

    loop(s)
    threads = [threading.Thread(target=loop, args=(st,)) for st in (None, s, None)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    hip.hipStreamSynchronize(s)
    hip.hipStreamDestroy(s)
    assert not bad


def test_allocation_under_capture_beside_a_busy_block(hpt, dev, hip):
    """A captured call allocates its result while the only cached block of that size is in use by the default stream."""
    x = np.random.default_rng(9).standard_normal((300, 1000)).astype(np.float32)
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    want = t.softmax(1).numpy()
    s, graph, gexec = P(), P(), P()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    r = t.softmax(1)
    del r
    assert hip.hipStreamBeginCapture(s, 0) == 0  # global
    try:
        out = t.softmax(1, stream=s)
    finally:
        rc = hip.hipStreamEndCapture(s, C.byref(graph))
    assert rc == 0 and graph.value
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
    for _ in range(3):
        assert hip.hipGraphLaunch(gexec, s) == 0 and hip.hipStreamSynchronize(s) == 0
        assert np.array_equal(out.numpy(), want)
        assert np.array_equal(t.softmax(1).numpy(), want)
    hip.hipGraphExecDestroy(gexec)
    hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(s)


def test_a_waiting_allocation_holds_nobody_up(hpt, dev, hip):
    """An ordinary allocation that finds only a block in use waits for the default stream; meanwhile other threads take and
    give back blocks."""
    import time
    from hpt_amd import _ffi
    l, n, m = hpt.lib(), 23456 * 64, 34567 * 64
    p, q, r = P(), P(), P()
    _ffi.check(l.hpt_hip_cache_clear(dev))
    _ffi.check(l.hpt_hip_alloc_ordered(dev, n, 64, C.byref(p)))
    _ffi.check(l.hpt_hip_alloc_ordered(dev, m, 64, C.byref(q)))
    _ffi.check(l.hpt_hip_free_ordered(dev, q, m, 64))
    keep = hpt.Tensor.empty([1 << 28], hpt.f32, dev)
    keep.add_(keep, out=keep)
    hpt.synchronize(dev)
    for _ in range(200):  # about a tenth of a second
        keep.add_(keep, out=keep)
    _ffi.check(l.hpt_hip_free_ordered(dev, p, n, 64))
    waiting = threading.Thread(target=lambda: _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(r))))
    waiting.start()
    time.sleep(0.01)
    for _ in range(20):
        _ffi.check(l.hpt_hip_alloc_ordered(dev, m, 64, C.byref(q)))
        _ffi.check(l.hpt_hip_free_ordered(dev, q, m, 64))
    busy = hip.hipStreamQuery(None) != 0
    hip.hipGetLastError()  # (not ready)
    still = waiting.is_alive()
    waiting.join()
    assert hip.hipStreamQuery(None) == 0 and r.value == p.value
    assert busy and still, "allocations on another thread waited for the default stream too"
    _ffi.check(l.hpt_hip_free(dev, r, n, 64))
    _ffi.check(l.hpt_hip_cache_clear(dev))


def test_idle_blocks_are_left_for_those_who_need_one(hpt, dev, hip):
    from hpt_amd import _ffi
    l, n = hpt.lib(), 45678 * 64
    p, q, r = P(), P(), P()
    _ffi.check(l.hpt_hip_cache_clear(dev))
    for x in (p, q):
        _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(x)))
    keep = _busy(hpt, dev)
    _ffi.check(l.hpt_hip_free_ordered(dev, p, n, 64))
    _ffi.check(l.hpt_hip_free(dev, q, n, 64))  # idle, and freed last
    _ffi.check(l.hpt_hip_alloc_ordered(dev, n, 64, C.byref(r)))
    assert r.value == p.value
    _ffi.check(l.hpt_hip_free_ordered(dev, r, n, 64))
    _ffi.check(l.hpt_hip_alloc(dev, n, 64, 0, C.byref(r)))
    assert r.value == q.value
    _ffi.check(l.hpt_hip_alloc_ordered(dev, n, 64, C.byref(q)))
    assert q.value == p.value
    for x in (r, q):
        _ffi.check(l.hpt_hip_free_ordered(dev, x, n, 64))
    del keep
    _ffi.check(l.hpt_hip_cache_clear(dev))
