"""Column reductions below 8 MiB: the lanes of a column block, the thread rows that share it and the workgroups that its rows are dealt over, either side of
each line of the rule (plans alone, no device), and the results there against the oracle."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_acc, half_atol

SUM, ARGMAX = 0, 14

# (type, shape, every second element, op, lanes, thread rows, workgroups)
PLANS = [
    # eight lanes from 769 rows on, whole vectors and not, stepped, up to 2048 rows in one launch
    ("f32", (768, 500), False, SUM, 16, 64, 1), ("f32", (769, 500), False, SUM, 8, 128, 1), ("f32", (2048, 512), False, SUM, 8, 128, 1), ("f32", (2049, 512), False, SUM, 16, 16, 11),
    ("f16", (768, 501), False, SUM, 16, 64, 1), ("f16", (769, 501), False, SUM, 8, 128, 1), ("f16", (2048, 501), False, SUM, 8, 128, 1), ("f16", (2049, 501), False, SUM, 16, 16, 11),
    ("f32", (768, 1000), True, SUM, 16, 64, 1), ("f32", (2048, 800), True, SUM, 8, 128, 1), ("f32", (2049, 800), True, SUM, 16, 16, 11),
    # up to 7 MiB, above that up to 1536 rows
    ("f16", (2000, 1835), False, SUM, 8, 128, 1), ("f16", (2000, 1836), False, SUM, 16, 16, 11), ("f32", (2000, 917), False, SUM, 8, 128, 1), ("f32", (2000, 918), False, SUM, 16, 16, 11),
    ("f16", (1536, 2400), False, SUM, 8, 128, 1), ("f16", (1537, 2400), False, SUM, 16, 16, 9),
    # up to 1536 rows of whole vectors that do not start on cache lines
    ("f32", (1536, 500), False, SUM, 8, 128, 1), ("f32", (1537, 500), False, SUM, 16, 16, 9), ("f16", (1536, 600), False, SUM, 8, 128, 1), ("f16", (1537, 600), False, SUM, 16, 16, 9),
    ("f32", (1537, 900), True, SUM, 16, 16, 9),
    # accumulators of eight bytes: argmax of two bytes up to 1536 rows, of one byte 64 thread rows and up to 1024 rows
    ("f16", (1536, 501), False, ARGMAX, 8, 128, 1), ("f16", (1537, 501), False, ARGMAX, 16, 16, 9), ("f32", (2048, 501), False, ARGMAX, 8, 128, 1), ("u8", (768, 500), False, ARGMAX, 16, 32, 1), ("u8", (769, 500), False, ARGMAX, 8, 64, 1), ("u8", (1024, 500), False, ARGMAX, 8, 64, 1),
    ("u8", (1025, 500), False, ARGMAX, 16, 16, 6), ("u8", (2048, 500), False, ARGMAX, 16, 16, 11), ("u8", (2048, 500), False, SUM, 8, 128, 1), ("i8", (1200, 900), False, ARGMAX, 16, 16, 7),
]


def _args(p):
    return pytest.mark.parametrize("dtype,shape,step,op,bx,by,split", p, ids=lambda v: str(v).replace(" ", ""))


@_args(PLANS)
def test_small_column_plans(hpt, dtype, shape, step, op, bx, by, split):
    t = hpt.Tensor.from_raw(1 << 40, list(shape), getattr(hpt, dtype))
    plan = hpt.reduce_plan(t[:, ::2] if step else t, op, [0])
    assert f" bx={bx} by={by} " in plan and f" split={split} " in plan, plan


@pytest.mark.gpu
@_args(PLANS)
def test_small_column_results(hpt, orc, dev, dtype, shape, step, op, bx, by, split):
    rng = np.random.default_rng(shape[0])
    npdt = {"f32": np.float32, "f16": np.float16, "u8": np.uint8, "i8": np.int8}[dtype]
    a = rng.standard_normal(shape).astype(npdt) if dtype in ("f32", "f16") else rng.integers(0, 100, shape).astype(npdt)
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    if step:
        t, a = t[:, ::2], a[:, ::2]
    if op == ARGMAX:
        assert np.array_equal(t.argmax(0).numpy(), orc.argreduce(True, a, 0))
        assert np.array_equal(t.argmin(0).numpy(), orc.argreduce(False, a, 0))
        return
    s = t.sum([0]).numpy()
    if dtype == "f16":
        want = orc.reduce(orc.SUM, a, [0], acc=half_acc(orc, a.shape[0])).astype(np.float32)
        assert_close(s.astype(np.float32), want, HALF_RTOL, half_atol(want, 11), "sum")
    elif dtype == "f32":  # (sums near zero: the error follows the terms, at most eps sqrt(n) of their size here, not the result)
        assert_close(s, orc.reduce(orc.SUM, a, [0], acc=orc.ACC_F64), F32_RTOL, max(F32_ATOL, 6e-8 * a.shape[0] ** 0.5), "sum")
    else:
        assert np.array_equal(s, orc.reduce(orc.SUM, a, [0]))
