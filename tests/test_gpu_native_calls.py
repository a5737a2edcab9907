"""The calls that return a fresh tensor go through one native crossing where the stream is None or an integer, and step by step
through ctypes where it is a ctypes pointer: both give the same bits, shapes, strides, stream records and errors."""
import ctypes as C
import gc
import threading

import numpy as np
import pytest

LONG = C.c_void_p(0)  # the default stream in the form that only ctypes takes


def _same_error(f, *args, **kw):
    got = []
    for stream in (None, LONG):
        with pytest.raises(Exception) as e:
            f(*args, stream=stream, **kw)
        got.append((type(e.value), str(e.value)))
    assert got[0] == got[1], got
    return got[0][1]


def test_errors_before_a_device_is_touched(hpt):
    t = hpt.Tensor.from_raw(1 << 40, [4, 5, 6], hpt.f32)
    assert "out of range" in _same_error(t.sum, [3])
    assert "duplicated" in _same_error(t.sum, [1, 1])
    assert "exactly one axis" in _same_error(t.argmax, [0, 1])
    assert "out of range" in _same_error(t.argmin, -4)
    assert "normalized dims" in _same_error(t.layernorm, [5])
    deep = hpt.Tensor.from_raw(1 << 40, [1] * 33, hpt.f32)  # more dims than either way takes
    _same_error(deep.sum, [0])
    with pytest.raises(NotImplementedError):
        hpt.Tensor.from_numpy(np.zeros((2, 2), np.float32)).sum([0])


def _both(f, *args, **kw):
    a, b = f(*args, **kw), f(*args, stream=LONG, **kw)
    assert (a.shape, a.strides, a.dtype, a.backend, a.device, a.parent) == (b.shape, b.strides, b.dtype, b.backend, b.device, b.parent)
    assert a._storage.nbytes == b._storage.nbytes and a._storage.pending == b._storage.pending == {0}
    assert a.numpy().tobytes() == b.numpy().tobytes()
    return a


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["bool", "u8", "i16", "i32", "i64", "f16", "bf16", "f32", "f64"])
def test_both_ways_agree(hpt, dev, dtype):
    rng = np.random.default_rng(3)
    x = rng.integers(0, 3, (6, 5, 32)) if dtype in ("bool", "u8", "i16", "i32", "i64") else rng.standard_normal((6, 5, 32))
    if dtype == "bf16":
        t = hpt.Tensor.from_numpy(hpt.f32_to_bf16_bits(x.astype(np.float32)), hpt.bf16).to_hip(dev)
    else:
        t = hpt.Tensor.from_numpy(x.astype({"bool": np.bool_, "u8": np.uint8, "i16": np.int16, "i32": np.int32, "i64": np.int64, "f16": np.float16,
                                            "f32": np.float32, "f64": np.float64}[dtype])).to_hip(dev)
    t._storage.wait()
    for v in (t, t.permute([2, 0, 1]), t[:, ::2, 1:30], t[:, :, ::-1]):
        for keep in (False, True):
            for axes in ([0], [0, 2], (1,), np.int64(2), [-1], [0, 1, 2]):
                _both(v.max, axes, keep)
            _both(v.sum, [1], keep)
            _both(v.mean, [0, 1], keep)
            _both(v.argmax, 1, keep)
        _both(v.softmax, 1)
        _both(v.log_softmax, -1)
        n = v.shape[-1]
        ft = v._float_binary_type()
        g, b = hpt.Tensor.full(0.5, [n], ft, dev), hpt.Tensor.full(0.25, [n], ft, dev)
        for gb in ((g, b), (g, None), (None, b), (None, None)):
            _both(v.layernorm, [n], *gb)
        if ft is v.dtype:
            c = v.contiguous()
            _both(c.add_layernorm, c, [n], g, b, 1e-3)
            _both(c.softmax_causal, 0.5, 1)
    assert t._storage.pending == {0}  # the input's use is on record too
    _same_error(t.softmax, 7)
    if dtype in ("f32", "f64"):
        _same_error(t.layernorm, [32], hpt.Tensor.full(1, [31], t.dtype, dev), None)  # refused after the result has been allocated
    else:
        _same_error(t.softmax_causal, log=False, causal_offset=0) if dtype in ("u8", "i32") else None


@pytest.mark.gpu
def test_memory_goes_back(hpt, dev):
    """Results, and those of calls that are refused, return to the allocator; from other threads too."""
    def live():
        n = C.c_uint64()
        hpt._ffi.check(hpt.lib().hpt_hip_alloc_stats(dev, C.byref(n), None, None))
        return n.value
    t = hpt.Tensor.full(1, [64, 48], hpt.f32, dev)
    bad = hpt.Tensor.full(1, [47], hpt.f32, dev)
    t.sum([1]), t.softmax(1)
    gc.collect()  # (tensors that errors of other tests still hold)
    before = live()

    def work():
        for _ in range(200):
            t.sum([0]), t.softmax(0), t.argmax(1), t.layernorm([48])
            with pytest.raises(hpt.HptError):
                t.layernorm([48], bad, None)
    threads = [threading.Thread(target=work) for _ in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    gc.collect()
    assert live() == before
    kept = [t.sum([0]) for _ in range(5)]
    assert live() == before + 5
    assert all(np.array_equal(k.numpy(), np.full(48, 64, np.float32)) for k in kept)
