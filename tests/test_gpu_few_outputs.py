"""Reductions whose time is a chain of dependent loads: rows of few outputs that stay in one launch of up to 1024 threads (around the
16384 vectors and the 4 MiB where a second launch begins), runs of one outer dim walked as one range, and the columns' remainders of one
to seven rows per lane with one to sixteen wavefronts to fold, against the oracle."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_acc, half_atol

pytestmark = pytest.mark.gpu

CASES = (
    # rows: one output and several, the last one-launch length and the first split one, off the vector grid, 1 ... 5 vectors per thread
    [((1, n), (1,)) for n in (65536, 65537, 65540, 1020, 1028, 4099, 8191)]
    + [((k, n), (1,)) for k, n in ((16, 65536), (17, 65536), (64, 16384), (65, 16384), (3, 20484), (7, 33333), (500, 2051))]
    # batch-norm runs: one outer dim, runs of fewer and of more vectors than threads, 1 ... 7 pairs per lane, several outer dims
    + [((b, c, h), (0, 2)) for b, c, h in ((3, 5, 49), (12, 6, 2401), (40, 28, 676), (2, 64, 676), (17, 3, 1000), (33, 9, 7), (9, 4, 5000))]
    + [((3, 4, 5, 6, 77), (0, 2, 4)), ((64, 2, 3136), (0, 2))]
    # columns: remainders after whole batches of eight, 1 ... 16 wavefronts
    + [((r, c), (0,)) for r in (7, 15, 64 * 8 + 65, 64 * 11, 64 * 13 + 1, 64 * 15 + 3) for c in (24, 64, 260)]
    + [((8 * 9 + 5, 3000), (0,)), ((1100, 5, 33), (0, 2)), ((300, 8200), (0,))]
)


@pytest.mark.parametrize("dtype", [np.float32, np.float16, np.int32, np.uint8, np.float64], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape,axes", CASES, ids=lambda v: str(v).replace(" ", ""))
def test_few_outputs(hpt, orc, dev, shape, axes, dtype):
    rng = np.random.default_rng(17)
    a = rng.standard_normal(shape).astype(dtype) if np.issubdtype(dtype, np.floating) else rng.integers(0, 100, shape).astype(dtype)
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    axes = list(axes)
    n = int(np.prod([shape[i] for i in axes]))
    plan = hpt.reduce_plan(t, hpt.SUM, axes)
    print(plan, flush=True)
    vectors = -(-n // (16 // a.itemsize))
    if axes != [0]:  # rows: one launch up to 16384 vectors per output and 4 MiB in all
        assert plan.startswith("row"), plan
        if vectors <= 16384 and a.size * a.itemsize <= 4 << 20:
            assert " split=1(" in plan, plan
    else:
        assert plan.startswith("col"), plan
    assert np.array_equal(t.max(axes).numpy(), a.max(tuple(axes)))
    if len(axes) == 1:
        assert np.array_equal(t.argmax(axes[0]).numpy(), orc.argreduce(True, a, axes[0]))
    s = t.sum(axes).numpy()
    if dtype == np.float16:
        want = orc.reduce(orc.SUM, a, axes, acc=half_acc(orc, n)).astype(np.float32)
        assert_close(s.astype(np.float32), want, HALF_RTOL, half_atol(want, 11), "sum")
    elif dtype in (np.float32, np.float64):
        # (sums near zero: the error follows the terms, at most eps sqrt(n) of their size here, not the result)
        rtol, atol = (F32_RTOL, max(F32_ATOL, 6e-8 * n ** 0.5)) if dtype == np.float32 else (1e-12, 1e-11)
        assert_close(s, orc.reduce(orc.SUM, a, axes, acc=orc.ACC_F64), rtol, atol, "sum")
    else:
        assert np.array_equal(s, orc.reduce(orc.SUM, a, axes))


# columns whose partials a second launch folds, 16 thread rows per output: 51 and 64 partials are up to four per thread, 129 and 141 up to nine, 235 fifteen, 256
# sixteen (eight loads in flight, then four)
PARTIALS = [((9000, 260), 51), ((4100, 1000), 64), ((16600, 127), 129), ((17000, 130), 141), ((30000, 100), 235), ((100000, 200), 256), ((200000, 33), 256)]


@pytest.mark.parametrize("dtype", [np.float32, np.int32], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape,split", PARTIALS, ids=lambda v: str(v).replace(" ", ""))
def test_partials_of_columns(hpt, orc, dev, shape, split, dtype):
    rng = np.random.default_rng(split)
    a = rng.standard_normal(shape).astype(dtype) if dtype == np.float32 else rng.integers(-1000, 1001, shape).astype(dtype)
    a[rng.integers(0, shape[0], shape[1]), np.arange(shape[1])] = 2000  # the largest of every column somewhere
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    plan = hpt.reduce_plan(t, hpt.SUM, [0])
    assert f" split={split} " in plan, plan
    assert np.array_equal(t.max([0]).numpy(), a.max(0))
    assert np.array_equal(t.argmax(0).numpy(), orc.argreduce(True, a, 0))
    s = t.sum([0]).numpy()
    if dtype == np.float32:  # (around 2000 and, as above, at most eps sqrt(n) of the terms)
        assert_close(s, orc.reduce(orc.SUM, a, [0], acc=orc.ACC_F64), F32_RTOL, 6e-8 * shape[0] ** 0.5, "sum")
    else:
        assert np.array_equal(s, a.sum(0, dtype=np.int32))


# argmin / argmax over the last axis of a view whose kept dims do not merge: one-byte rows of fewer than 64 vectors walk a lane's remainder together, longer ones
# one by one; and sixteen wavefronts of eight-byte pairs, which meet four at a time
@pytest.mark.parametrize("dtype", [np.uint8, np.int8, np.float64, np.int64], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("shape,axis", [((30, 8, 160), 2), ((30, 8, 1008), 2), ((30, 8, 1024), 2), ((30, 8, 1040), 2), ((30, 8, 4111), 2), ((600, 4, 40), 0), ((1025, 4, 130), 0)], ids=str)
def test_argreduce_of_views(hpt, orc, dev, shape, axis, dtype):
    rng = np.random.default_rng(23)
    a = rng.integers(-100 if np.issubdtype(dtype, np.signedinteger) else 0, 100, shape).astype(dtype)
    t, v = hpt.Tensor.from_numpy(a).to_hip(dev)[:, :3], a[:, :3]
    print(hpt.reduce_plan(t, 14, [axis]), flush=True)
    assert np.array_equal(t.argmax(axis).numpy(), orc.argreduce(True, np.ascontiguousarray(v), axis))
    assert np.array_equal(t.argmin(axis).numpy(), orc.argreduce(False, np.ascontiguousarray(v), axis))
