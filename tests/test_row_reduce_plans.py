"""Row reductions of few outputs: how many threads share an output and whether one launch does, either side of each line of the rule (plans alone, no device),
and the results there against the oracle."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL

SUM, MAX, ARGMAX = 0, 2, 14

# (type, shape, op, threads per output, launches)
PLANS = [
    # one launch up to 16384 vectors per output and 4 MiB in all, off the vector grid too; 8192 of one-byte argmin / argmax
    ("f32", (1, 65536), SUM, 1024, 1), ("f32", (1, 65540), SUM, 256, 2), ("f32", (16, 65536), SUM, 1024, 1), ("f32", (17, 65536), SUM, 256, 2), ("f32", (1, 65539), SUM, 1024, 1), ("f32", (1, 65543), SUM, 256, 2),
    ("u8", (1, 131072), ARGMAX, 1024, 1), ("u8", (1, 131088), ARGMAX, 256, 2), ("u8", (1, 204894), ARGMAX, 256, 2), ("u8", (1, 204894), MAX, 1024, 1), ("u8", (2, 131072), ARGMAX, 1024, 1),
    ("bf16", (1, 131072), ARGMAX, 1024, 1),
    # four vectors per thread; eight where some lanes would have four and most of the others three
    ("u8", (300, 3072), ARGMAX, 64, 1), ("u8", (300, 3088), ARGMAX, 32, 1), ("u8", (300, 3584), ARGMAX, 32, 1), ("u8", (300, 3600), ARGMAX, 64, 1),
    ("f32", (100, 800), SUM, 32, 1), ("f32", (100, 3200), SUM, 128, 1), ("f32", (100, 3588), SUM, 256, 1), ("f32", (100, 4096), SUM, 256, 1), ("f32", (100, 6400), SUM, 512, 1), ("f32", (7, 6400), SUM, 512, 1), ("f32", (5, 13200), SUM, 1024, 1),
    # and where up to four workgroups would become more
    ("f32", (128, 68), SUM, 8, 1), ("f32", (129, 68), SUM, 4, 1), ("f32", (256, 68), SUM, 4, 1), ("f32", (257, 68), SUM, 8, 1), ("bf16", (30, 2048), ARGMAX, 32, 1), ("f32", (7, 4092), SUM, 128, 1),
]


def _args(p):
    return pytest.mark.parametrize("dtype,shape,op,tpr,launches", p, ids=lambda v: str(v).replace(" ", ""))


@_args(PLANS)
def test_row_reduce_plans(hpt, dtype, shape, op, tpr, launches):
    plan = hpt.reduce_plan(hpt.Tensor.from_raw(1 << 40, list(shape), getattr(hpt, dtype)), op, [len(shape) - 1])
    assert plan.startswith("row") and f" tpr={tpr} " in plan and (" split=1(" in plan) == (launches == 1), plan


@pytest.mark.gpu
@_args([p for p in PLANS if p[0] != "bf16"])
def test_row_reduce_results(hpt, orc, dev, dtype, shape, op, tpr, launches):
    rng = np.random.default_rng(shape[-1])
    a = rng.standard_normal(shape).astype(np.float32) if dtype == "f32" else rng.integers(0, 200, shape).astype(np.uint8)
    axis = len(shape) - 1
    for at in (0, shape[-1] // 2, shape[-1] - 1):  # the largest of all in the first, a middle and the last vector
        b = a.copy()
        b[..., at] = 250
        t = hpt.Tensor.from_numpy(b).to_hip(dev)
        assert np.array_equal(t.argmax(axis).numpy(), orc.argreduce(True, b, axis))
        assert np.array_equal(t.max([axis]).numpy(), b.max(axis))
    s = t.sum([axis]).numpy()
    if dtype == "f32":
        assert_close(s, orc.reduce(orc.SUM, b, [axis], acc=orc.ACC_F64), F32_RTOL, F32_ATOL, "sum")
    else:
        assert np.array_equal(s, orc.reduce(orc.SUM, b, [axis]))


@pytest.mark.gpu
def test_captured_argmax_takes_no_scratch(hpt, dev):
    """One-byte argmax of 8193 ... 16384 vectors is split for speed alone: recorded, on a stream that has no scratch, it is one node."""
    import ctypes as C

    from hpt_amd import _ffi
    hip, P = C.CDLL("libamdhip64.so"), C.c_void_p
    hip.hipStreamCreateWithFlags.argtypes = [C.POINTER(P), C.c_uint]
    hip.hipStreamBeginCapture.argtypes = [P, C.c_int]
    hip.hipStreamEndCapture.argtypes = [P, C.POINTER(P)]
    hip.hipGraphGetNodes.argtypes = [P, P, C.POINTER(C.c_size_t)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(P), P, P, P, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [P, P]
    for f in (hip.hipStreamSynchronize, hip.hipGraphExecDestroy, hip.hipGraphDestroy, hip.hipStreamDestroy):
        f.argtypes = [P]
    a = np.random.default_rng(4).integers(0, 200, (2, 204896)).astype(np.uint8)
    a[0, 204895], a[1, 3] = 250, 250
    t, out = hpt.Tensor.from_numpy(a).to_hip(dev), hpt.Tensor.empty([2], hpt.i64, dev)
    assert "split=1(" not in hpt.reduce_plan(t, ARGMAX, [1])
    s, graph, gexec, n = P(), P(), P(), C.c_size_t()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0
    vin, k1 = t._c_view()
    vout, k2 = out._c_view()
    hpt.synchronize(dev)
    assert hip.hipStreamBeginCapture(s, 0) == 0
    try:
        rc = _ffi.lib().hpt_hip_argreduce(dev, s, 1, C.byref(vin), 1, C.byref(vout))
    finally:
        ended = hip.hipStreamEndCapture(s, C.byref(graph))
    assert rc == 0 and ended == 0 and hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0 and n.value == 1
    assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
    for _ in range(3):
        assert hip.hipGraphLaunch(gexec, s) == 0 and hip.hipStreamSynchronize(s) == 0
        assert np.array_equal(out.numpy(), [204895, 3])
        assert np.array_equal(t.argmax(1).numpy(), [204895, 3])  # eagerly, in two launches
    hip.hipGraphExecDestroy(gexec)
    hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(s)
