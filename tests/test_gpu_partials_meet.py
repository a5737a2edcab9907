"""Softmax whose statistics are partials of several wavefronts and workgroups: long rows shared by workgroups with one to nine vectors per thread, and
transposed views of few, long rows on both sides of where eight wavefronts share a slice, with rows whose maximum lies in one partial only,
rows that are all -inf but for one element, and infinities and NaN, against 64 bits."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu

# rows of 16384 elements and more, whole vectors and not: slices of 1024 vectors and more, the last one short; stored [columns, rows]
ROWS = [(3, 32768), (1, 32772), (2, 40001), (5, 36868), (1, 300007), (100, 16389), (2, 147456)]
COLUMNS = [(8191, 100), (8192, 100), (8195, 101), (16383, 130), (16400, 129), (6208, 163), (12000, 400), (8195, 160), (8192, 130), (12000, 101), (8192, 8192)]
# what they take: (f32, f16) wavefronts of a slice, none where a group of lanes per row is ahead of few two-byte rows
WAVEFRONTS = {(8191, 100): (8, None), (8192, 100): (8, None), (8195, 101): (8, None), (16400, 129): (4, 4), (8192, 8192): (4, 4)}


def _values(shape, dtype, axis, seed):
    rng = np.random.default_rng(seed)
    x = (rng.standard_normal(shape) * 3).astype(dtype)
    v = np.moveaxis(x, axis, -1)  # (a view: one row per leading index)
    n = v.shape[-1]
    v[0, n - 1] = 40  # one partial holds what counts
    if v.shape[0] > 3:
        v[1, :] = -np.inf
        v[1, n // 2] = 1
        v[2, : n // 2] = -np.inf
        v[3, 7] = np.nan
    return x


@pytest.mark.parametrize("dtype", [np.float32, np.float16], ids=lambda d: np.dtype(d).name)
@pytest.mark.parametrize("kind,shape", [("rows", s) for s in ROWS] + [("transposed", s) for s in COLUMNS], ids=str)
def test_partials_meet(hpt, dev, kind, shape, dtype):
    x = _values(shape, dtype, 1 if kind == "rows" else 0, 5)
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    if kind == "transposed":
        t, x = t.permute([1, 0]), x.T
    plan = hpt.normalize_plan(t, 1)
    print(plan, flush=True)
    if kind == "rows":
        assert plan.startswith("rowsplit"), plan
    else:
        waves = WAVEFRONTS.get(shape, (8, 8))[dtype == np.float16]
        assert plan.startswith("transposed") and f" tpr={waves} " in plan if waves else plan.startswith("generic "), plan
    v = x.astype(np.float64)
    d = v - v.max(1, keepdims=True)
    e = np.exp(d)
    for log in (False, True):
        got = (t.log_softmax(1) if log else t.softmax(1)).numpy().astype(np.float64)
        want = d - np.log(e.sum(1, keepdims=True)) if log else e / e.sum(1, keepdims=True)
        ok = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), ok) and np.array_equal(np.isnan(got), np.isnan(want))
        if dtype == np.float16:
            assert_close(got[ok], want[ok], HALF_RTOL, max(half_atol(want[ok], 11), 6e-8), f"log={log}")
        else:
            assert_close(got[ok], want[ok], F32_RTOL, F32_ATOL, f"log={log}")
