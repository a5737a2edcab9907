"""Reductions over axis 0 (and the middle axis of slabs) whose inner rows are no whole vectors and wider than a workgroup: the flat walk in
workgroups of 256 or 512 threads (large ones for several slabs), unaligned columns for shorter elements where enough is
reduced; either side of each line, against numpy."""
import numpy as np
import pytest

from conftest import assert_close

gpu = pytest.mark.gpu


@gpu
@pytest.mark.parametrize("dtype,shape,axis", [
    ("f32", (2050, 1027), 0), ("f32", (2051, 4097), 0), ("f32", (521, 8190), 0), ("f32", (67, 33001), 0), ("f32", (64, 32770), 0), ("f32", (3, 1031, 2051), 1),
    ("f32", (5, 255, 2051), 1), ("i32", (1501, 2051), 0), ("i32", (12, 128, 4225), 1), ("f64", (301, 4099), 0), ("f16", (1031, 5003), 0), ("f16", (255, 17001), 0),
    ("f16", (256, 17001), 0), ("u8", (4097, 2051), 0), ("u8", (255, 36001), 0)], ids=str)
def test_wide_columns(hpt, dev, dtype, shape, axis):
    rng = np.random.default_rng(sum(shape))
    npdt = {"f32": np.float32, "f64": np.float64, "f16": np.float16, "i32": np.int32, "u8": np.uint8}[dtype]
    a = rng.integers(0, 90, shape).astype(npdt)  # many ties; sums are exact in the accumulators of every type
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    got = t.sum([axis]).numpy()
    if dtype in ("i32", "u8"):
        assert np.array_equal(got, a.sum(axis, dtype=npdt))
    else:
        want = a.sum(axis, dtype=np.float64)
        assert_close(got.astype(np.float64), want, 2 ** -11 if dtype == "f16" else 2 ** -24, 0, f"{dtype} {shape}")  # one rounding
    assert np.array_equal(t.max([axis]).numpy(), a.max(axis))
    assert np.array_equal(t.argmax(axis).numpy(), a.argmax(axis))
    assert np.array_equal(t.argmin(axis).numpy(), a.argmin(axis))


# the plans alone, no device
@pytest.mark.parametrize("dtype,shape,axis,want", [
    ("f32", (8190, 4097), 0, "col-flat-wide vec=4 as=256x60"), ("f32", (700, 50257), 0, "col-flat-wide vec=4 as=512x20"), ("f32", (16, 512, 4097), 1, "col-flat-wide"), ("f16", (16, 512, 4097), 1, "col-unaligned"),
    ("i32", (12, 128, 4225), 1, "col-flat-wide"), ("f16", (8190, 4097), 0, "col-unaligned vec=8"), ("f16", (255, 17001), 0, "col-flat-wide"),
    ("u8", (8190, 4097), 0, "col-unaligned vec=16")], ids=str)
def test_plans(hpt, dtype, shape, axis, want):
    plan = hpt.reduce_plan(hpt.Tensor.from_raw(1 << 40, list(shape), getattr(hpt, dtype)), hpt.SUM, [axis])
    first, launched = want.partition(" as=")[::2]
    assert plan.startswith(first) and (" as=" + launched + " " in plan if launched else " as=" not in plan), plan
