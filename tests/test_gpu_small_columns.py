"""Column reductions of small inputs (below 8 MiB): narrow column blocks, unaligned vectors whose last lane is taken
from the row's end backwards, and rows dealt over workgroups with a second launch - at the sizes where each begins and
ends, against the oracle. Sums that accumulate into `out` and swapped kept dims go the same ways."""
import ctypes as C

import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_acc, half_atol

pytestmark = pytest.mark.gpu

# (shape, reduced axis, view): around one vector more than a lane, two lanes, the row count from which unaligned vectors
# are taken (64), thousands of rows, which are split (2048 and 2049, where that begins, are in test_small_column_plans.py), odd and whole rows, stepped
# rows, a swapped kept dim
SHAPES = [
    ((6135, 287), 0, None), ((12608, 128), 0, None), ((1536, 128), 0, None), ((1537, 128), 0, None), ((34112, 40), 0, None), ((5440, 45), 0, None), ((37446, 16), 0, None),
    ((63, 4099), 0, None), ((64, 4099), 0, None), ((3073, 8), 0, None), ((3073, 9), 0, None), ((9000, 3), 0, None), ((20001, 1), 0, None),
    ((4000, 17), 0, None), ((4000, 15), 0, None), ((3, 472, 21, 21), 1, None), ((2, 64, 13, 7), 1, None), ((1578, 2101), 0, "step"),
    ((3136, 176), 0, "step"), ((40, 5000, 7), 1, None), ((33, 700, 130), 2, "permute"), ((33, 701, 131), 2, "permute"),
]
DTYPES = [np.float32, np.float16, np.int32, np.uint8, np.float64]


@pytest.mark.parametrize("dtype", DTYPES, ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape,axis,view", SHAPES, ids=lambda v: str(v).replace(" ", ""))
def test_small_columns(hpt, orc, dev, shape, axis, view, dtype):
    rng = np.random.default_rng(91)
    if np.issubdtype(dtype, np.floating):
        a = rng.standard_normal(shape).astype(dtype)
    else:
        a = rng.integers(0, 100, shape).astype(dtype)
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    if view == "step":
        t, a = t[:, ::2], a[:, ::2]
    elif view == "permute":  # the contiguous kept dim comes first, the reduced one last
        t, a, axis = t.permute([2, 0, 1]), a.transpose(2, 0, 1), 2
    print(hpt.reduce_plan(t, hpt.SUM, [axis]), flush=True)
    assert np.array_equal(t.max([axis]).numpy(), a.max(axis))
    assert np.array_equal(t.argmin(axis).numpy(), orc.argreduce(False, a, axis))
    s = t.sum([axis])
    if dtype == np.float16:
        want = orc.reduce(orc.SUM, a, [axis], acc=half_acc(orc, a.shape[axis])).astype(np.float32)
        assert_close(s.numpy().astype(np.float32), want, HALF_RTOL, half_atol(want, 11), "sum")
    elif dtype in (np.float32, np.float64):
        rtol, atol = (F32_RTOL, F32_ATOL) if dtype == np.float32 else (1e-12, 1e-11)
        assert_close(s.numpy(), orc.reduce(orc.SUM, a, [axis], acc=orc.ACC_F64), rtol, atol, "sum")
    else:
        assert np.array_equal(s.numpy(), orc.reduce(orc.SUM, a, [axis]))
    if dtype in (np.int32, np.uint8):  # accumulate: every output is added to exactly once
        t.sum_([axis], False, False, s)
        assert np.array_equal(s.numpy(), orc.reduce(orc.SUM, a, [axis]) * np.dtype(dtype).type(2))


def test_static_and_captured_calls_take_no_scratch(hpt, dev):
    """The entry whose partials live in one array shared by all streams, and calls that are recorded, keep small inputs in one
    launch: one node in the graph, where a split reduction has two."""
    hip, P = C.CDLL("libamdhip64.so"), C.c_void_p
    hip.hipStreamCreateWithFlags.argtypes = [C.POINTER(P), C.c_uint]
    hip.hipStreamBeginCapture.argtypes = [P, C.c_int]
    hip.hipStreamEndCapture.argtypes = [P, C.POINTER(P)]
    hip.hipGraphGetNodes.argtypes = [P, P, C.POINTER(C.c_size_t)]
    hip.hipGraphInstantiate.argtypes = [C.POINTER(P), P, P, P, C.c_size_t]
    hip.hipGraphLaunch.argtypes = [P, P]
    for f in (hip.hipStreamSynchronize, hip.hipGraphExecDestroy, hip.hipGraphDestroy, hip.hipStreamDestroy):
        f.argtypes = [P]
    a = np.random.default_rng(5).integers(-99, 100, (12608, 128)).astype(np.int32)
    b = np.random.default_rng(6).integers(-99, 100, (20000, 1024)).astype(np.int32)  # large: split in any case
    t, u = hpt.Tensor.from_numpy(a).to_hip(dev), hpt.Tensor.from_numpy(b).to_hip(dev)
    for x in (t, u):
        assert "split=1 " not in hpt.reduce_plan(x, hpt.SUM, [0]) + " "
        assert np.array_equal(x.sum([0], static_scratch=True).numpy(), x.numpy().sum(0, dtype=np.int32))
    s = P()
    assert hip.hipStreamCreateWithFlags(C.byref(s), 1) == 0  # non-blocking
    for x, static, nodes in ((t, True, 1), (t, False, 1), (u, True, 2)):
        want, out = x.numpy().sum(0, dtype=np.int32), hpt.Tensor.empty([x.shape[1]], hpt.i32, dev)
        graph, gexec, n = P(), P(), C.c_size_t()
        hpt.synchronize(dev)
        assert hip.hipStreamBeginCapture(s, 0) == 0
        try:
            x.sum_([0], False, True, out, stream=s, static_scratch=static)
        finally:
            rc = hip.hipStreamEndCapture(s, C.byref(graph))
        assert rc == 0 and hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
        assert n.value == nodes, (x.shape, static)
        assert hip.hipGraphInstantiate(C.byref(gexec), graph, None, None, 0) == 0
        for _ in range(3):
            assert hip.hipGraphLaunch(gexec, s) == 0 and hip.hipStreamSynchronize(s) == 0
            assert np.array_equal(out.numpy(), want), (x.shape, static)
            assert np.array_equal(x.sum([0]).numpy(), want)  # eagerly, in two launches
        hip.hipGraphExecDestroy(gexec)
        hip.hipGraphDestroy(graph)
    hip.hipStreamDestroy(s)
