"""A NaN anywhere in a row makes every result of a softmax row NaN, in every form the launches take: alone in a lane's first elements, in whole vectors,
among -inf, first, last. Statistics that are kept as (maximum so far, sum) must not drop it while there is no maximum yet."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu

# (shape, view, axis, form, types): "T" the stored tensor transposed, an integer: every so many elements of a row, "off" rows from their second element on
FORMS = [
    ((64, 1000), None, 1, "rowreg ", "f32 f16"), ((16, 4104), None, 1, "rowreg ", "f32 f16"), ((64, 1001), None, 1, "rowreg-shift ", "f32 f16"),
    ((300, 16392), None, 1, "rowreg-lds ", "f32 f16"), ((300, 17001), None, 1, "rowreg-lds-shift ", "f32 f16"),
    ((4937, 505), None, 1, "rowreg-shift+tile ", "f32 f16"), ((40000, 33), None, 1, "rowreg+tile ", "f32"), ((64, 2000), 2, 1, "rowreg-step2 ", "f32 f16"),
    ((16, 36001), 2, 1, "rowstream ", "f32 f16"), ((16, 40000), 3, 1, "rowstream ", "f32 f16"), ((16, 10217), "off", 1, "rowstream ", "f64"), ((16, 4231), None, 1, "rowstream-shift ", "f64"),
    ((139, 21002), None, 1, "rowstream ", "f64"), ((300, 140001), None, 1, "rowstream-shift ", "f32"),
    ((16, 40960), None, 1, "rowsplit ", "f32 f16 f64"), ((16, 40001), None, 1, "rowsplit-unaligned ", "f32 f16"),
    ((8191, 100), "T", 1, "generic ", "f16"), ((9, 4097), "T", 1, "generic ", "f32 f16"), ((4163, 275), "T", 1, "transposed-unaligned ", "f32 f16"), ((8192, 128), "T", 1, "transposed ", "f32 f16"),
    ((500, 184), "T", 1, "transposed-tile ", "f32"), ((501, 187), "T", 1, "transposed-tile-unaligned ", "f32"),
    ((128, 184), "T", 1, "transposed-tile ", "f16"), ((67, 69), "T", 1, "transposed-tile-unaligned ", "f16"),
    ((3000, 400), None, 0, "col-split ", "f32 f16"), ((3000, 401), None, 0, "col-split-unaligned ", "f32"), ((3000, 401), None, 0, "col-split ", "f16"), ((2000, 1001), None, 0, "col-split-unaligned ", "f16"), ((87407, 24), None, 0, "col-split-flat ", "f32"), ((180000, 24), None, 0, "col-split-flat ", "f16"),
    ((30, 808, 44), None, 1, "col-split-flat ", "f64"), ((3, 1161, 634), None, 1, "col-split-flat-unaligned ", "f32"),
    ((3, 109, 2000), None, 1, "col-reg ", "f32 f16"), ((3, 109, 2001), None, 1, "col-reg-unaligned ", "f32 f16"), ((40, 512, 512), None, 1, "col-reg ", "f32 f16"),
    ((9, 109, 3), None, 1, "col-slab ", "f32 f16"), ((60000, 16, 2), None, 1, "col-group-tile ", "f32"), ((1200, 500, 2), None, 1, "rowreg-interleaved ", "f32"),
    ((900, 1000, 3), None, 1, "rowreg-modular ", "f16"), ((300, 1092, 5), None, 1, "rowreg-modular ", "f32"),
]


def _spoil(v):
    """Rows 0 ... 6 of [rows, n] hold a NaN each, row 7 does not."""
    n = v.shape[-1]
    v[0, 0] = np.nan
    v[1, n - 1] = np.nan
    v[2, : max(1, min(64, n // 2))] = np.nan
    v[3] = -np.inf
    v[3, n // 2] = np.nan
    v[4] = -np.inf
    v[4, n // 2] = np.nan
    v[4, 0] = 1
    v[5, max(0, n // 2 - 20) : n // 2 + 20] = -np.inf
    v[5, n // 2] = np.nan
    v[6] = np.nan
    v[7, : n // 2] = -np.inf


@pytest.mark.parametrize("shape,view,axis,form,dtype", [(s, v, a, f, d) for s, v, a, f, ds in FORMS for d in ds.split()], ids=lambda p: str(p).replace(" ", ""))
def test_softmax_keeps_every_nan(hpt, dev, shape, view, axis, form, dtype):
    npdt = {"f32": np.float32, "f16": np.float16, "f64": np.float64}[dtype]
    stored = (np.random.default_rng(9).standard_normal(shape) * 3).astype(npdt)
    cut = {"T": lambda a: a.T if isinstance(a, np.ndarray) else a.permute([1, 0]), "off": lambda a: a[:, 1:], None: lambda a: a}.get(view) or (lambda a: a[:, ::view])
    x = cut(stored)
    rows = np.moveaxis(x, axis, -1)
    _spoil(rows if rows.ndim == 2 else rows[1] if rows.shape[1] >= 8 else rows[:, 0])
    t = cut(hpt.Tensor.from_numpy(stored).to_hip(dev))
    plan = hpt.normalize_plan(t, axis)
    print(plan, flush=True)
    assert plan.startswith(form), plan
    v = np.moveaxis(x, axis, -1).astype(np.float64)
    with np.errstate(invalid="ignore"):
        d = v - np.fmax.reduce(v, -1, keepdims=True)
    e = np.exp(d)
    for log in (False, True):
        got = np.moveaxis((t.log_softmax(axis) if log else t.softmax(axis)).numpy(), axis, -1).astype(np.float64)
        want = d - np.log(e.sum(-1, keepdims=True)) if log else e / e.sum(-1, keepdims=True)
        lost = np.argwhere(np.isnan(got) != np.isnan(want))
        assert not lost.size, f"log={log}: NaN pattern differs in rows {sorted({tuple(i[:-1].tolist()) for i in lost})[:9]}"
        ok = np.isfinite(want)
        assert np.array_equal(got[~ok & ~np.isnan(want)], want[~ok & ~np.isnan(want)])
        if dtype == "f16":
            assert_close(got[ok], want[ok], HALF_RTOL, max(half_atol(want[ok], 11), 6e-8), f"log={log}")
        else:
            assert_close(got[ok], want[ok], F32_RTOL, F32_ATOL, f"log={log}")


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("shape", [(2, 9, 700), (2, 9, 9001), (2, 9, 70000), (3, 9, 160001)], ids=str)
def test_causal_softmax_keeps_every_nan(hpt, dev, shape, dtype):
    x = (np.random.default_rng(9).standard_normal(shape) * 3).astype(np.float32 if dtype == "f32" else np.float16)
    q, k = shape[1:]
    _spoil(x[1])
    x[0, 0, -1] = np.nan  # never read: beyond the first query's keys
    live = np.arange(k)[None, :] <= np.arange(q)[:, None] + (k - q)
    got = hpt.Tensor.from_numpy(x).to_hip(dev).softmax_causal(1.0, k - q).numpy()
    want = np.isnan(np.where(live, x, 0)).any(-1)
    assert np.array_equal(np.isnan(got).any(-1), want)
    assert np.array_equal((np.isnan(got) | ~live).all(-1), want)
