"""Normalisations in place whose last vector of a row is taken from the row's end backwards: every element has one writer, and
nothing is read by one workgroup after another has stored it. The same bits as into a fresh tensor."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _values(hpt, shape, dtype):
    x = (np.random.default_rng(12).standard_normal(shape) * 3).astype(np.float32)
    if dtype == "bf16":
        return hpt.f32_to_bf16_bits(x), hpt.bf16
    return x.astype({"f32": np.float32, "f16": np.float16, "f64": np.float64}[dtype]), None


# inner lengths a few elements past what a wavefront of vectors covers: the last vector is alone in its workgroup
COLUMNS = [("f32", (4100, 4097)), ("f32", (4100, 4099)), ("f32", (3, 2100, 4097)), ("f16", (4100, 4097)), ("bf16", (4100, 4103)), ("f64", (3000, 1025))]


@pytest.mark.parametrize("dtype,shape", COLUMNS, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
@pytest.mark.parametrize("log", [False, True])
def test_softmax_over_odd_columns_in_place(hpt, dev, dtype, shape, log):
    a, dt = _values(hpt, shape, dtype)
    axis = len(shape) - 2
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
    plan = hpt.normalize_plan(t, axis)
    assert plan.startswith("col-split-unaligned"), plan
    run = t.log_softmax if log else t.softmax
    want = run(axis).numpy()
    run(axis, out=t)
    assert np.array_equal(t.numpy(), want), plan


# the other forms with unaligned vectors: slabs in one workgroup's registers, register columns, the flat walk
MIDDLE = [("col-slab", (201, 1639, 5)), ("col-slab", (3, 4095, 7)), ("col-reg-unaligned", (16, 128, 3249)), ("col-split-flat-unaligned", (9, 2501, 1001))]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16"])
@pytest.mark.parametrize("plan,shape", MIDDLE, ids=lambda v: v if isinstance(v, str) else "x".join(map(str, v)))
def test_softmax_over_the_middle_axis_in_place(hpt, dev, dtype, plan, shape):
    a, dt = _values(hpt, shape, dtype)
    for log in (False, True):
        t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
        assert hpt.normalize_plan(t, 1).startswith(plan), hpt.normalize_plan(t, 1)
        run = t.log_softmax if log else t.softmax
        want = run(1).numpy()
        run(1, out=t)
        assert np.array_equal(t.numpy(), want), log


@pytest.mark.parametrize("dtype", ["f32", "f16", "f64"])
@pytest.mark.parametrize("shape", [(1, 1 << 22), (5, 1 << 20), (4, 300007), (100, 65539)], ids=lambda v: "x".join(map(str, v)))
def test_layernorm_of_shared_rows_in_place(hpt, dev, dtype, shape):
    a, dt = _values(hpt, shape, dtype)
    a[:, 0] = 50
    t, r = hpt.Tensor.from_numpy(a, dt).to_hip(dev), hpt.Tensor.from_numpy(a[:, ::-1].copy(), dt).to_hip(dev)
    plan = hpt.normalize_plan(t, 0, 1)
    assert plan.startswith("rowsplit"), plan
    n = [shape[1]]
    want, want_sum = t.layernorm(n, None, None, 1e-5).numpy(), t.layernorm(n, None, None, 1e-5, residual=r).numpy()
    u = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
    t.layernorm(n, None, None, 1e-5, out=t)
    assert np.array_equal(t.numpy(), want), plan
    u.layernorm(n, None, None, 1e-5, residual=r, out=u)
    assert np.array_equal(u.numpy(), want_sum), plan
