"""Softmax over a long axis that is not the last: the statistics pass folds the columns of a wavefront in batches, two in
flight, then four, then one at a time, and the last pass walks the axis from its end. Column counts either side of every
batch, inner lengths either side of a wavefront of vectors, against numpy in float64."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

gpu = pytest.mark.gpu


def _reference(x, log):
    x = x.astype(np.float64)
    d = x - x.max(0, keepdims=True)
    e = np.exp(d)
    return d - np.log(e.sum(0, keepdims=True)) if log else e / e.sum(0, keepdims=True)


# One wavefront's columns: cols / (slices * wavefronts). With `inner` of one group of vectors the slices are min(256, max(64,
# cols / 64)), so these run from less than one batch to two batches, four and one more column per wavefront.
@gpu
@pytest.mark.parametrize("dtype,cols,inner", [
    ("f32", 1025, 256), ("f32", 2047, 255), ("f32", 2049, 257), ("f32", 4095, 256), ("f32", 4097, 300), ("f32", 5121, 1025), ("f32", 2304, 2052),
    ("f32", 20000, 64), ("f32", 21001, 63), ("f16", 1031, 512), ("f16", 4099, 520), ("f16", 8200, 511), ("f16", 20001, 320), ("bf16", 6148, 1001),
    ("bf16", 3000, 2432), ("f64", 1100, 2050), ("f64", 1027, 2049)])
def test_long_axis(hpt, dev, dtype, cols, inner):
    rng = np.random.default_rng(cols * 31 + inner)
    x = (rng.standard_normal((cols, inner)) * 3).astype(np.float32)
    x[:, 1] = -np.inf
    x[cols // 2, 1] = 0.5  # one finite entry
    x[:, inner - 1] += np.linspace(-40, 40, cols, dtype=np.float32)  # the running maximum rises to the very end
    bits = {"f16": 11, "bf16": 8}.get(dtype, 0)
    a = hpt.f32_to_bf16_bits(x) if dtype == "bf16" else x.astype({"f16": np.float16, "f32": np.float32, "f64": np.float64}[dtype])
    tof = hpt.bf16_bits_to_f32 if dtype == "bf16" else (lambda v: v)
    t = hpt.Tensor.from_numpy(a, hpt.bf16 if dtype == "bf16" else None).to_hip(dev)
    plan = hpt.normalize_plan(t, 0)
    assert plan.startswith("col-split"), plan
    for log in (False, True):
        got = tof((t.log_softmax(0) if log else t.softmax(0)).numpy()).astype(np.float64)
        want = _reference(tof(a), log)
        fin = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), fin), plan
        if bits:
            assert_close(got[fin], want[fin], HALF_RTOL, max(half_atol(want[fin], bits), 6e-8), f"{plan} log={log}")
        elif dtype == "f64":
            assert_close(got[fin], want[fin], 1e-12, 1e-14, f"{plan} log={log}")
        else:
            assert_close(got[fin], want[fin], F32_RTOL, F32_ATOL, f"{plan} log={log}")


# where lanes along the inner dim take over from the flat walk (plans alone, no device)
@pytest.mark.parametrize("dtype,cols,inner,flat", [
    ("f32", 16384, 508, True), ("f32", 16384, 512, False), ("f32", 32768, 1024, True), ("f32", 32768, 1028, False), ("f32", 20000, 767, True),
    ("f32", 20000, 769, False), ("f16", 20000, 312, True), ("f16", 20000, 320, False), ("f16", 55924, 600, True), ("f16", 20000, 600, False),
    ("bf16", 20000, 767, True), ("bf16", 20000, 769, False), ("f64", 9000, 2048, True), ("f64", 9000, 2050, False)])
def test_where_the_flat_walk_ends(hpt, dtype, cols, inner, flat):
    plan = hpt.normalize_plan(hpt.Tensor.from_raw(1 << 40, [cols, inner], getattr(hpt, dtype)), 0)
    assert plan.startswith("col-split-flat") == flat and plan.startswith("col-split"), plan
