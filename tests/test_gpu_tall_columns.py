"""Softmax over an axis of up to 1024 elements held in whole vectors by 512 or 1024 threads: axis lengths either side of what a
thread row, a vector more per thread and the next form hold, inner rows from one vector to odd lengths past a segment, few and
many segments (an odd number leaves one without its pair), views with wider pitches, and the call in place."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

gpu = pytest.mark.gpu

CASES = [
    # four bytes: up to 256 in 32 rows of 8 vectors and segments of 128 elements, up to 512 in 64 rows of 8, up to 1024 of 16
    ("f32", (1, 2, 4)), ("f32", (3, 31, 20)), ("f32", (5, 129, 127)), ("f32", (3, 255, 129)), ("f32", (7, 256, 100)), ("f32", (2, 256, 2044)),
    ("f32", (40, 257, 36)), ("f32", (9, 300, 65)), ("f32", (3, 511, 1023)), ("f32", (33, 512, 68)), ("f32", (17, 513, 1000)), ("f32", (13, 1024, 1001)),
    # two bytes: 32 rows of 8 and 16 vectors, 64 rows of 16, segments of 128 elements
    ("f16", (1, 3, 8)), ("f16", (5, 65, 127)), ("bf16", (3, 128, 136)), ("f16", (7, 255, 129)), ("bf16", (9, 256, 100)), ("f16", (31, 257, 72)),
    ("bf16", (5, 511, 1023)), ("f16", (11, 512, 200)), ("f16", (100, 513, 150)), ("bf16", (97, 1024, 128)), ("f16", (20, 1000, 801)),
]


def _values(shape, dtype, hpt):
    rng = np.random.default_rng(sum(shape))
    x = (rng.standard_normal(shape) * 3).astype(np.float32)
    x[..., -1] += 25 * np.linspace(-1, 1, shape[1], dtype=np.float32)
    x[0, :, 0] = -np.inf
    x[0, shape[1] // 2, 0] = 0.25   # one finite entry
    x[-1, :, 1] = -np.inf           # none
    a = hpt.f32_to_bf16_bits(x) if dtype == "bf16" else x.astype({"f16": np.float16, "f32": np.float32}[dtype])
    return a, hpt.bf16 if dtype == "bf16" else None


def _check(hpt, got, a, dtype, log, what):
    tof = hpt.bf16_bits_to_f32 if dtype == "bf16" else (lambda v: v)
    got, x = tof(got).astype(np.float64), tof(a).astype(np.float64)
    with np.errstate(invalid="ignore"):
        d = x - x.max(1, keepdims=True)
        s = np.exp(d).sum(1, keepdims=True)
        want = d - np.log(s) if log else np.exp(d) / s
    assert np.array_equal(np.isnan(got), np.isnan(want)), what
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin), what
    if dtype == "f32":
        assert_close(got[fin], want[fin], F32_RTOL, F32_ATOL, what)
    else:
        assert_close(got[fin], want[fin], HALF_RTOL, max(half_atol(want[fin], 8 if dtype == "bf16" else 11), 6e-8), what)


@gpu
@pytest.mark.parametrize("dtype,shape", CASES, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_tall_columns(hpt, dev, dtype, shape):
    a, dt = _values(shape, dtype, hpt)
    for log in (False, True):
        t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
        plan = hpt.normalize_plan(t, 1)
        assert plan.startswith("col-reg"), plan
        run = t.log_softmax if log else t.softmax
        fresh = run(1).numpy()
        _check(hpt, fresh, a, dtype, log, f"{dtype} {shape} log={log} {plan}")
        run(1, out=t)  # in place: no workgroup reads what another has written
        assert np.array_equal(t.numpy(), fresh, equal_nan=dtype != "bf16"), plan


# pitches of the axis and of the slabs that are wider than the inner rows, on and off the vector grid
@gpu
@pytest.mark.parametrize("dtype,shape,cut", [("f32", (5, 300, 140), (4, 132)), ("f32", (5, 200, 141), (1, 130)), ("f16", (6, 200, 152), (8, 144)),
                                             ("bf16", (4, 333, 150), (3, 140))], ids=str)
def test_tall_columns_of_views(hpt, dev, dtype, shape, cut):
    a, dt = _values(shape, dtype, hpt)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)[:, :, cut[0]:cut[1]]
    v = a[:, :, cut[0]:cut[1]]
    plan = hpt.normalize_plan(t, 1)
    assert plan.startswith("col-reg"), plan
    for log in (False, True):
        _check(hpt, (t.log_softmax(1) if log else t.softmax(1)).numpy(), v, dtype, log, f"{dtype} {shape}[{cut}] log={log}")


# the plans alone, no device: (thread rows, vectors per thread) of the form, or None for the plan of before
@pytest.mark.parametrize("dtype,shape,want", [
    ("f32", (8, 128, 1000), None), ("f32", (8, 129, 1000), (32, 8)), ("f32", (8, 256, 1000), (32, 8)), ("f32", (8, 256, 1024), None),
    ("f32", (8, 257, 1000), (64, 8)), ("f32", (16, 512, 2048), None), ("f32", (64, 512, 1024), (64, 8)), ("f32", (1, 512, 262144), None), ("f32", (8, 512, 1001), (64, 8)),
    ("f32", (16, 512, 1001), None), ("f32", (32, 512, 1001), (64, 8)), ("f32", (24, 321, 1001), None), ("f32", (24, 320, 1001), (64, 8)), ("f32", (16, 512, 1000), (64, 8)), ("f32", (256, 512, 65), (64, 8)),
    ("f32", (8, 513, 4000), (64, 16)), ("f32", (2, 513, 1000), None), ("f32", (8, 1025, 4000), None), ("f32", (2, 40, 30), (32, 8)), ("f32", (1, 300, 259), None),
    ("f16", (8, 64, 10000), None), ("f16", (8, 65, 1000), (32, 8)), ("f16", (8, 257, 1000), (32, 16)), ("bf16", (64, 256, 2048), None), ("f16", (16, 1000, 2048), (64, 16)),
    ("bf16", (1, 513, 58050), None), ("f16", (4, 777, 1000), None), ("f64", (8, 200, 1000), None),
    # the work-items of one launch: 1024 threads per 128 elements of an inner row
    ("f32", (511, 200, (1 << 20) + 4), (32, 8)), ("f32", (512, 200, (1 << 20) + 4), None)], ids=str)
def test_plans(hpt, dtype, shape, want):
    plan = hpt.normalize_plan(hpt.Tensor.from_raw(1 << 40, list(shape), getattr(hpt, dtype)), 1)
    tall = plan.startswith("col-reg") and f" tpr={want[0]} " in plan and f" nchunk={want[1]} " in plan if want else False
    if want:
        assert tall, plan
    else:
        assert not (plan.startswith("col-reg") and (" tpr=32 " in plan or " tpr=64 " in plan)), plan
