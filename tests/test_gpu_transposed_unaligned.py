"""Normalisation along the strided axis of a transposed view whose rows or columns are not whole, aligned vectors: the
register tiles and the three passes with unaligned vectors, at the edges of vectors, tiles and wavefronts, against the
oracle; and the same call under capture, where the form without scratch runs."""
import ctypes as C

import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu

# (stored shape [.., columns, rows], first stored row and element left out). Column and row counts one below, at and
# one above vectors, the 64-row and 16-column tiles, and the 4096 columns that fit one workgroup's registers.
SHAPES = [
    ((64, 65), 0, 0), ((65, 64), 0, 0), ((79, 8193), 0, 0), ((81, 4095), 0, 0), ((367, 4099), 0, 0), ((1000, 2049), 0, 0),
    ((257, 16391), 0, 0), ((4095, 2051), 0, 0), ((4097, 130), 0, 0), ((5003, 1001), 0, 0), ((3, 131, 1027), 0, 0), ((5, 1000, 71), 0, 0),
    ((129, 4097), 1, 1), ((1024, 2049), 0, 1), ((72, 4104), 0, 3),
]
DTYPES = ["f32", "f16", "bf16", "f64"]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape,skip_cols,skip_rows", SHAPES, ids=lambda v: str(v).replace(" ", ""))
def test_transposed_unaligned(hpt, orc, dev, shape, skip_cols, skip_rows, dtype):
    rng = np.random.default_rng(37)
    x = (rng.standard_normal(shape) * 2 + rng.uniform(-3, 3, shape[:-2] + (1, shape[-1]))).astype(np.float32)
    ident = lambda v: v
    cv, tof, dt, odt, bits, acc = {
        "f32": (ident, ident, None, None, 0, orc.ACC_F64),
        "f64": (lambda v: v.astype(np.float64), ident, None, None, 0, orc.ACC_F64),
        "f16": (lambda v: v.astype(np.float16), lambda v: v.astype(np.float32), None, None, 11, orc.ACC_F32),
        "bf16": (hpt.f32_to_bf16_bits, hpt.bf16_bits_to_f32, hpt.bf16, orc.BF16, 8, orc.ACC_F32),
    }[dtype]
    a = cv(x)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
    if len(shape) == 2:
        t, a = t[skip_cols:, skip_rows:], a[skip_cols:, skip_rows:]
    t = t.permute([1, 0] if len(shape) == 2 else [0, 2, 1])
    a = np.ascontiguousarray(a.swapaxes(-1, -2))
    axis, n = a.ndim - 1, a.shape[-1]
    plan = hpt.normalize_plan(t, axis)
    print(plan, flush=True)
    if n >= 128 and a.shape[-2] >= 128:
        assert plan.startswith("transposed"), plan
    g, b = cv(rng.normal(1, 0.1, n + 1).astype(np.float32)), cv(rng.normal(0, 0.1, n + 1).astype(np.float32))
    # gamma and beta start one element off too
    tg, tb = (hpt.Tensor.from_numpy(v, dt).to_hip(dev)[1:] for v in (g, b))

    def check(got, want, what):
        got, want = tof(got), tof(want)
        if bits:
            assert_close(got, want, HALF_RTOL, max(half_atol(want, bits), 6e-8 if bits == 11 else 0), f"{what} {shape} {dtype}")
        else:
            assert_close(got, want, F32_RTOL, F32_ATOL, f"{what} {shape} {dtype}")

    check(t.softmax(axis).numpy(), orc.softmax(a, axis, acc=acc, dtype=odt), "softmax")
    check(t.log_softmax(axis).numpy(), orc.softmax(a, axis, log=True, acc=acc, dtype=odt), "log_softmax")
    check(t.layernorm([n], tg, tb, 1e-5).numpy(), orc.layernorm(a, 1, g[1:], b[1:], 1e-5, acc=acc, dtype=odt), "layernorm")
    check(t.layernorm([n], None, None, 1e-5).numpy(), orc.layernorm(a, 1, None, None, 1e-5, acc=acc, dtype=odt), "layernorm alone")


@pytest.mark.parametrize("shape", [(131, 4099), (4099, 203)], ids=str)
def test_transposed_unaligned_special_rows(hpt, dev, shape):
    """Masked rows, a row of -inf only, a row with one +inf: what a row held twice or a column counted once must not change."""
    cols, rows = shape
    x = np.full(shape, -np.inf, np.float32)
    x[cols - 1, 0] = 2.0                         # one finite entry, in the last column
    x[:, 1] = np.arange(cols) % 97
    x[:, rows - 1] = (np.arange(cols) % 89) - 40
    x[:, 3] = np.float32(np.finfo(np.float32).min)
    x[cols - 2, 4] = np.inf
    t = hpt.Tensor.from_numpy(x).to_hip(dev).permute([1, 0])
    s = t.softmax(1).numpy()
    assert s[0, cols - 1] == 1.0 and s[0].sum() == 1.0
    assert np.all(np.isnan(s[2])) and np.isnan(s[4]).any()
    for r in (1, 3, rows - 1):
        e = np.exp(x[:, r].astype(np.float64) - x[:, r].max())
        assert_close(s[r], e / e.sum(), F32_RTOL, F32_ATOL, f"row {r}")


def test_transposed_unaligned_captured(hpt, dev):
    """Five thousand columns take three passes and scratch; under capture, where no scratch may be allocated, the call
    runs in the form without, and every replay gives the eager result."""
    hip = C.CDLL("libamdhip64.so")
    P = C.c_void_p
    hip.hipStreamCreateWithFlags.argtypes = [C.POINTER(P), C.c_uint]
    hip.hipStreamBeginCapture.argtypes = [P, C.c_int]
    hip.hipStreamEndCapture.argtypes = [P, C.POINTER(P)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(P), P, P, P, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [P, P]
    for f in (hip.hipStreamSynchronize, hip.hipGraphExecDestroy, hip.hipGraphDestroy, hip.hipStreamDestroy):
        f.argtypes = [P]
    x = np.random.default_rng(3).standard_normal((5003, 131)).astype(np.float32)
    t = hpt.Tensor.from_numpy(x).to_hip(dev).permute([1, 0])
    assert hpt.normalize_plan(t, 1).startswith("transposed-unaligned")
    want = t.softmax(1).numpy()
    out = hpt.Tensor.empty([131, 5003], hpt.f32, dev)
    s, graph, gexec = P(), P(), P()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
    hpt.synchronize(dev)
    assert hip.hipStreamBeginCapture(s, 2) == 0  # relaxed
    try:
        t.softmax(1, stream=s, out=out)
    finally:
        rc = hip.hipStreamEndCapture(s, C.byref(graph))
    assert rc == 0 and graph.value
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
    try:
        for _ in range(3):
            assert hip.hipGraphLaunch(gexec, s) == 0 and hip.hipStreamSynchronize(s) == 0
            assert_close(out.numpy(), want, F32_RTOL, F32_ATOL, "replay")
            assert np.array_equal(t.softmax(1).numpy(), want), "eager between the replays"
    finally:
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)
        hip.hipStreamDestroy(s)


@pytest.mark.parametrize("dtype,rows,cols", [("f64", 17, 2097121), ("f64", 16, 2097152), ("f32", 33, 4194241)])
def test_transposed_of_millions_of_columns(hpt, dev, dtype, rows, cols):
    """Just past 65535 column blocks of the last pass (32 eight-byte columns each, 64 four-byte ones)."""
    np_dtype = np.float64 if dtype == "f64" else np.float32
    x = np.random.default_rng(21).random((cols, rows), dtype=np_dtype)
    t = hpt.Tensor.from_numpy(x).to_hip(dev).permute([1, 0])
    assert hpt.normalize_plan(t, 1).startswith("transposed"), hpt.normalize_plan(t, 1)
    e = np.exp(x.T.astype(np.float64))
    # (results of 5e-7: compared as shares of the largest; f64 sums of cols terms in any order are 1e-10 apart at most)
    got = t.softmax(1).numpy()
    assert_close(got * cols, e / e.sum(1, keepdims=True) * cols, 1e-9 if dtype == "f64" else F32_RTOL, F32_ATOL, "softmax")
    del e, got
    d = x.T.astype(np.float64)
    d -= d.mean(1, keepdims=True)
    d /= np.sqrt((d * d).mean(1, keepdims=True) + 1e-5)
    assert_close(t.layernorm([cols], None, None, 1e-5).numpy(), d, 1e-9 if dtype == "f64" else F32_RTOL, F32_ATOL, "layernorm")
