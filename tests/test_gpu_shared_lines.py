"""Softmax over an axis whose inner rows do not start on cache lines: neighbouring workgroups share the lines between them, and the launches
number them so that neighbours run on one XCD and choose how results are stored by the size of the result. Sizes on both sides of each of
those lines, with counts of workgroups that leave the last run partly filled, against numpy in 64 bits."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu


def _softmax64(x, axis):
    e = np.exp(x - x.max(axis, keepdims=True))
    return e / e.sum(axis, keepdims=True)


# (shape, dtype): equal shares below 48 MiB, runs of 32 workgroups above; results through the cache from 20 to 48 MiB and from 96 MiB on for four
# bytes, from 48 (aligned) or 96 MiB on for two
MIDDLE = [((5, 129, 45), "f32"), ((1, 257, 61), "f32"), ((52, 300, 301), "f32"), ((64, 300, 301), "f32"), ((46, 512, 600), "f32"), ((83, 512, 600), "f32"),
          ((83, 513, 598), "f32"), ((3, 70, 1001), "f32"), ((101, 64, 2001), "f32"), ((7, 513, 36), "f32"),
          ((66, 512, 1000), "f16"), ((99, 512, 1001), "f16"), ((40, 200, 1001), "f16"), ((3, 66, 75), "f16")]


@pytest.mark.parametrize("shape,dtype", MIDDLE, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_softmax_over_the_middle_axis(hpt, dev, shape, dtype):
    rng = np.random.default_rng(71)
    x = (rng.standard_normal(shape, dtype=np.float32) * 3).astype(np.float32 if dtype == "f32" else np.float16)
    x[0, :, 0] = -50
    x[-1, -1, -1] = 40  # the last element of all dominates its column
    want = _softmax64(x.astype(np.float64), 1)
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    got = t.softmax(1).numpy().astype(np.float64)
    half = dtype == "f16"
    assert_close(got, want, HALF_RTOL if half else F32_RTOL, max(half_atol(want, 11), 6e-8) if half else F32_ATOL, f"{shape} {dtype}")
    if x.size < 4 << 20:
        got = t.log_softmax(1).numpy().astype(np.float64)
        log = x.astype(np.float64) - x.max(1, keepdims=True)
        log -= np.log(np.exp(log).sum(1, keepdims=True))
        assert_close(got, log, HALF_RTOL if half else F32_RTOL, half_atol(log, 11) if half else F32_ATOL, f"log {shape} {dtype}")


# a long axis 0, three launches: vectors whose rows do not start on lines, eight equal parts from 16 MiB on (with one and several batches)
LONG = [((2047, 2051), "f32"), ((2048, 2048), "f32"), ((1100, 4100), "f32"), ((1031, 1030), "f32"), ((2, 1500, 1502), "f32"), ((4099, 2051), "f16"), ((2500, 4100), "f16")]


@pytest.mark.parametrize("shape,dtype", LONG, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_softmax_over_a_long_axis(hpt, dev, shape, dtype):
    axis = len(shape) - 2
    x = (np.random.default_rng(72).standard_normal(shape, dtype=np.float32) * 3).astype(np.float32 if dtype == "f32" else np.float16)
    x[..., -1, -1] = 40
    want = _softmax64(x.astype(np.float64), axis)
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    half = dtype == "f16"
    for inplace in (False, True):
        got = t.softmax(axis, out=t if inplace else None).numpy().astype(np.float64)
        assert_close(got, want, HALF_RTOL if half else F32_RTOL, max(half_atol(want, 11), 6e-8) if half else F32_ATOL, f"{shape} {dtype} inplace={inplace}")


# stored [columns, rows], normalised along the columns: three launches with unaligned vectors beyond 4096 columns (column blocks of 64 or 128, the last
# one partly filled; one and two batches), register tiles below; aligned tiles that run eight in a row on an XCD
TRANSPOSED = [((4500, 701), "f32"), ((4101, 1030), "f16"), ((2, 4200, 259), "f32"), ((1001, 2603), "f32"), ((900, 5003), "f16"), ((3500, 4112), "f32"), ((2048, 8256), "f16")]


@pytest.mark.parametrize("shape,dtype", TRANSPOSED, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_transposed_rows(hpt, dev, shape, dtype):
    x = (np.random.default_rng(73).standard_normal(shape, dtype=np.float32) * 3).astype(np.float32 if dtype == "f32" else np.float16)
    x[..., -1, -1] = 40
    perm = [0, 2, 1][-len(shape):] if len(shape) == 3 else [1, 0]
    v = x.astype(np.float64).transpose(perm)
    t = hpt.Tensor.from_numpy(x).to_hip(dev).permute(perm)
    half = dtype == "f16"
    for name, want, got in [("softmax", _softmax64(v, -1), t.softmax(len(shape) - 1)),
                            ("layernorm", (v - v.mean(-1, keepdims=True)) / np.sqrt(v.var(-1, keepdims=True) + 1e-5), t.layernorm([shape[-2]]))]:
        assert_close(got.numpy().astype(np.float64), want, HALF_RTOL if half else F32_RTOL, max(half_atol(want, 11), 6e-8) if half else F32_ATOL, f"{name} {shape} {dtype}")


# held by 512 and 1024 threads, either side of where results begin to leave through the caches: whole vectors of four bytes from 20 MiB, of two from 48; unaligned ones of
# four bytes from 34 MiB (26 of more than 256 elements of the axis), where a segment of 128 (64) elements is a part of an inner row, of 48 to 96 MiB from an axis of 160 on
STORED = [((43, 300, 404), "f32"), ((44, 300, 404), "f32"), ((26, 1000, 500), "f32"), ((59, 300, 1400), "f16"), ((60, 300, 1400), "f16"), ((84, 300, 2001), "f16"),
          ((56, 300, 402), "f32"), ((57, 300, 402), "f32"), ((330, 300, 71), "f32"), ((330, 300, 73), "f32"), ((44, 200, 1001), "f32"), ((45, 200, 1001), "f32"),
          ((320, 200, 143), "f32"), ((320, 200, 145), "f32"), ((100, 159, 801), "f32"), ((99, 160, 801), "f32"), ((129, 150, 1301), "f32"), ((129, 200, 1001), "f32")]


@pytest.mark.parametrize("log", [False, True], ids=["softmax", "log_softmax"])
@pytest.mark.parametrize("shape,dtype", STORED, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_results_through_the_caches(hpt, dev, shape, dtype, log):
    x = (np.random.default_rng(74).standard_normal(shape, dtype=np.float32) * 3).astype(np.float32 if dtype == "f32" else np.float16)
    x[-1, -1, -1] = 40
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    plan = hpt.normalize_plan(t, 1)
    assert plan.startswith("col-reg") and (" tpr=32 " in plan or " tpr=64 " in plan), plan
    run = t.log_softmax if log else t.softmax
    fresh = run(1).numpy()
    half = dtype == "f16"
    for b in (slice(0, 2), slice(shape[0] // 2, shape[0] // 2 + 1), slice(shape[0] - 2, shape[0])):  # (64 bits of the whole take seconds)
        d = x[b].astype(np.float64) - x[b].max(1, keepdims=True)
        e = np.exp(d)
        want = d - np.log(e.sum(1, keepdims=True)) if log else e / e.sum(1, keepdims=True)
        assert_close(fresh[b].astype(np.float64), want, HALF_RTOL if half else F32_RTOL, max(half_atol(want, 11), 6e-8) if half else F32_ATOL, f"{shape} {dtype}")
    if not log:
        assert abs(fresh.sum(1, dtype=np.float64) - 1).max() < (2.0 ** -10 if half else 1e-5)  # (every column: results are rounded to 2 ** -11 of themselves, and the sum to their statistics)
    run(1, out=t)
    assert np.array_equal(t.numpy(), fresh)


# held in registers, workgroups dealt to the XCDs and as they come: single elements and pairs of inner rows that a workgroup holds whole and does not, aligned pairs,
# vectors on cache lines, and rows on lines in batches that are not
REGISTERS = [((472, 176, 9), "f32", 1), ((36, 1000, 157), "f32", 1), ((600, 100, 13), "f16", 1), ((300, 60, 33), "f64", 1), ((8227, 43, 27), "f32", 2), ((40, 43, 301), "f32", 4),
             ((817, 13, 37), "f32", 2), ((28, 512, 510), "f32", 2), ((64, 40, 128), "f32", 4), ((500, 43, 20), "f32", 4)]


@pytest.mark.parametrize("shape,dtype,vec", REGISTERS, ids=lambda v: str(v).replace(" ", ""))
def test_register_columns(hpt, dev, shape, dtype, vec):
    x = (np.random.default_rng(75).standard_normal(shape) * 3).astype({"f32": np.float32, "f16": np.float16, "f64": np.float64}[dtype])
    x[0, :, 0] = -50
    x[-1, -1, -1] = 40
    t = hpt.Tensor.from_numpy(x).to_hip(dev)
    print(hpt.normalize_plan(t, 1), flush=True)
    half = dtype == "f16"
    want = _softmax64(x.astype(np.float64), 1)
    for inplace in (False, True):
        got = t.softmax(1, out=t if inplace else None).numpy().astype(np.float64)
        assert_close(got, want, HALF_RTOL if half else F32_RTOL, max(half_atol(want, 11), 6e-8) if half else F32_ATOL, f"{shape} {dtype} inplace={inplace}")


@pytest.mark.parametrize("axis_len", [21, 100])
@pytest.mark.parametrize("batch_step", [1, 2, 4, 32])
def test_register_columns_of_batches_off_the_lines(hpt, dev, axis_len, batch_step):
    """Inner rows of 256 bytes back to back, the batches a few elements apart: unaligned vectors with every row but the batches on cache lines."""
    b, length = 40000 // axis_len, 64
    step = axis_len * length + batch_step
    flat = (np.random.default_rng(76).standard_normal(b * step) * 3).astype(np.float32)
    base = hpt.Tensor.from_numpy(flat).to_hip(dev)
    t = hpt.Tensor.from_raw(base.ptr, [b, axis_len, length], hpt.f32, dev, strides=[step, length, 1])
    plan = hpt.normalize_plan(t, 1)
    assert plan.startswith("col-reg"), plan
    x = np.lib.stride_tricks.as_strided(flat, (b, axis_len, length), (step * 4, length * 4, 4)).astype(np.float64)
    assert_close(t.softmax(1).numpy().astype(np.float64), _softmax64(x, 1), F32_RTOL, F32_ATOL, plan)
