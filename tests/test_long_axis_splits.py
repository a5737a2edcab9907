"""The statistics pass over a long axis and over the columns of transposed rows: into how many slices an axis is dealt, and the columns that are
left after a wavefront's whole batches, which are loaded together and folded as four, two and one of them."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol


def _split(hpt, t, *args):
    return int(hpt.normalize_plan(t, *args).split("split=")[1].split()[0])


# One workgroup per compute unit of 256, or two if they fill the units better: never more, or the scratch of a call outgrows what a
# capture of before found there. Single elements: two, 64 partials per row of all but long axes.
@pytest.mark.parametrize("dtype,cols,inner,slices", [
    ("f32", 8190, 4097, 15), ("f64", 1344, 8248, 7), ("f32", 1977, 16400, 7), ("f32", 1300, 40004, 3), ("f16", 2047, 4097, 28), ("f16", 2056, 271, 64),
    ("f16", 4270, 268, 64), ("f32", 7353, 79, 64), ("f32", 13675, 122, 128), ("f32", 4100, 63, 64), ("f32", 138341, 11, 256), ("f64", 49999, 15, 128), ("f16", 18232, 536, 128)])
def test_slices_of_a_long_axis(hpt, dtype, cols, inner, slices):
    t = hpt.Tensor.from_raw(1 << 40, [cols, inner], getattr(hpt, dtype))
    assert hpt.normalize_plan(t, 0).startswith("col-split") and _split(hpt, t, 0) == slices


@pytest.mark.parametrize("dtype,cols,rows,softmax,layernorm", [
    ("f32", 8192, 8192, 8, 8), ("f16", 8192, 8192, 32, 16), ("bf16", 5001, 4001, 32, 32), ("f64", 5001, 1001, 32, 32), ("f32", 16384, 1024, 64, 64),
    ("f32", 5000, 40000, 3, 3)])
def test_slices_of_transposed_rows(hpt, dtype, cols, rows, softmax, layernorm):
    t = hpt.Tensor.from_raw(1 << 40, [cols, rows], getattr(hpt, dtype)).permute([1, 0])
    assert hpt.normalize_plan(t, 1).startswith("transposed")
    assert (_split(hpt, t, 1), _split(hpt, t, 0, 1)) == (softmax, layernorm)


# 256 wavefronts share an axis of 64 slices: eight columns each and `left` more, some wavefronts one more still
@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("left", range(8))
def test_columns_left_over(hpt, dev, dtype, left):
    inner = {"f32": 255, "f16": 512}[dtype]
    cols = 2048 + 256 * left + 5
    rng = np.random.default_rng(left)
    x = (rng.standard_normal((cols, inner)) * 3).astype(np.float32)
    x[-300:, ::3] += 6  # what is left over counts
    x[:, 5] = -np.inf
    x[cols - 1, 5] = 1
    a = x.astype(np.float16) if dtype == "f16" else x
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    assert _split(hpt, t, 0) == 64
    v = a.astype(np.float64)
    d = v - v.max(0)
    for log in (False, True):
        got = (t.log_softmax(0) if log else t.softmax(0)).numpy().astype(np.float64)
        want = d - np.log(np.exp(d).sum(0)) if log else np.exp(d) / np.exp(d).sum(0)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin)
        if dtype == "f16":
            assert_close(got[fin], want[fin], HALF_RTOL, max(half_atol(want[fin], 11), 6e-8), f"{dtype} {left} log={log}")
        else:
            assert_close(got[fin], want[fin], F32_RTOL, F32_ATOL, f"{dtype} {left} log={log}")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f64"])
@pytest.mark.parametrize("left", [0, 1, 3, 4, 6, 7])
def test_transposed_columns_left_over(hpt, dev, dtype, left):
    rows = {"f32": 1024, "bf16": 2048, "f64": 511}[dtype]
    cols = 8192 + 256 * left + 3
    rng = np.random.default_rng(left + 100)
    x = (rng.standard_normal((cols, rows), dtype=np.float32) + np.linspace(-3, 3, rows, dtype=np.float32))
    x[-300:] += 2
    a, dt = (hpt.f32_to_bf16_bits(x), hpt.bf16) if dtype == "bf16" else (x.astype({"f32": np.float32, "f64": np.float64}[dtype]), None)
    back = hpt.bf16_bits_to_f32 if dtype == "bf16" else (lambda u: u)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev).permute([1, 0])
    assert hpt.normalize_plan(t, 0, 1).startswith("transposed") and _split(hpt, t, 0, 1) == 64
    v = back(a).astype(np.float64).T
    d = v - v.mean(1, keepdims=True)
    want = d / np.sqrt((d * d).mean(1, keepdims=True) + 1e-5)
    got = back(t.layernorm([cols], None, None, 1e-5).numpy())
    if dtype == "bf16":
        assert_close(got, want, HALF_RTOL, half_atol(want, 8), f"{dtype} {left}")
    else:
        assert_close(got, want, 1e-12 if dtype == "f64" else F32_RTOL, 1e-12 if dtype == "f64" else F32_ATOL, f"{dtype} {left}")
