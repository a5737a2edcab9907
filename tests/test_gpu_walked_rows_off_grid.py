"""Layernorm rows off the vector grid, more of them than one round of workgroups holds, in each of their forms: unaligned vectors with gamma / beta in
registers and in LDS, every second element, aligned vectors that contain the row; x + residual, whose residual is off by another amount;
and the plans that choose among these. Against numpy in float64."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol


def _plan(hpt, t, *args):
    p = hpt.normalize_plan(t, *args)
    words = dict(w.split("=", 1) for w in p.split() if "=" in w)
    return p, "unaligned" in p.split(), int(words["vec"]), int(words["tpr"]), int(words["rpb"]), int(words["nchunk"]), int(words["max_blocks"])


def _check(hpt, dtype, got, x, g, b, what):
    """In blocks of rows: the float64 copies of a large case would be gigabytes."""
    for r in range(0, x.shape[0], 2048):
        v = x[r:r + 2048].astype(np.float64)
        v -= v.mean(1, keepdims=True)
        want = v / np.sqrt((v * v).mean(1, keepdims=True) + 1e-5) * g + b
        if dtype == "f32":
            assert_close(got[r:r + 2048], want, F32_RTOL, F32_ATOL, what)
        else:
            assert_close(got[r:r + 2048], want, HALF_RTOL, half_atol(want, 8 if dtype == "bf16" else 11), what)


def _codec(hpt, dtype):
    if dtype == "bf16":
        return hpt.f32_to_bf16_bits, hpt.bf16_bits_to_f32, hpt.bf16
    np_type = {"f16": np.float16, "f32": np.float32}[dtype]
    return (lambda v: v.astype(np_type)), (lambda v: v.astype(np.float32)), None


def _rows(hpt, owner, off, rows, cols):
    """Contiguous rows that start `off` elements into the memory of `owner`."""
    return hpt.Tensor.from_raw(owner.ptr + off * owner.dtype.size, [rows, cols], owner.dtype)


# (dtype, rows, stored columns, step, form of the plain layernorm, threads per row, vectors per thread, workgroups at most)
FORMS = [
    ("f16", 24601, 641, 1, "unaligned", 32, 3, 3072), ("bf16", 6200, 3011, 1, "unaligned", 128, 3, 3072), ("f16", 3100, 7001, 1, "unaligned", 256, 4, 3072),
    ("f16", 600, 12001, 1, "unaligned", 512, 3, 512), ("bf16", 530, 16377, 1, "unaligned", 512, 4, 512), ("f16", 4400, 1281, 2, "unaligned", 64, 4, 1024),
    ("bf16", 600, 12291, 2, "unaligned", 512, 4, 512), ("f16", 530, 32767, 2, "unaligned", 1024, 4, 512), ("f32", 1100, 4097, 1, "unaligned", 256, 5, 1024),
    ("f32", 600, 8301, 1, "unaligned", 512, 5, 512), ("f32", 530, 15001, 1, "unaligned", 1024, 4, 512), ("f32", 4500, 774, 1, "unaligned", 64, 4, 1024),
    ("f32", 4300, 750, 1, "unaligned", 64, 3, 1024), ("f32", 1100, 3090, 1, "unaligned", 256, 4, 1024),
    # few rows, a workgroup each
    ("f16", 121, 6149, 1, "unaligned", 512, 2, 0), ("bf16", 500, 3111, 1, "unaligned", 256, 2, 0), ("f32", 336, 4458, 1, "shift", 512, 3, 0), ("f32", 500, 3090, 1, "shift", 256, 4, 0),
    ("f16", 340, 1763, 2, "single", 256, 4, 0), ("f16", 600, 7001, 2, "unaligned", 256, 4, 0), ("bf16", 110, 23911, 2, "unaligned", 1024, 4, 0), ("f16", 530, 16387, 2, "unaligned", 1024, 4, 512)]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,rows,stored,step,form,threads,vectors,most", FORMS)
def test_walked_rows_off_the_grid(hpt, dev, dtype, rows, stored, step, form, threads, vectors, most):
    to, back, dt = _codec(hpt, dtype)
    rng = np.random.default_rng(rows + stored)
    x = rng.standard_normal((rows, stored), dtype=np.float32) + rng.uniform(-5, 5, (rows, 1)).astype(np.float32)
    a = to(x)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)[:, ::step]
    v = back(a)[:, ::step]
    cols = v.shape[1]
    plan, ua, vec, tpr, rpb, nchunk, blocks = _plan(hpt, t, 0, 1)
    assert (ua, vec > 1, tpr, nchunk) == (form == "unaligned", form != "single", threads, vectors), plan
    if most:
        assert -(-rows // rpb) > most and (most == 512 or blocks in (most, 768)), plan  # some workgroups have a second row
    (ag, ab, ar) = (to(u.astype(np.float32)) for u in (rng.normal(1, 0.1, cols + 1), rng.normal(0, 0.1, cols + 1), rng.standard_normal(rows * cols + 3)))
    tg, tb = (hpt.Tensor.from_numpy(u, dt).to_hip(dev)[1:] for u in (ag, ab))
    g, b = back(ag)[1:].astype(np.float64), back(ab)[1:].astype(np.float64)
    _check(hpt, dtype, back(t.layernorm([cols], tg, tb, 1e-5).numpy()), v, g, b, plan)
    owner = hpt.Tensor.from_numpy(ar, dt).to_hip(dev)
    for off in (0, 3):  # a residual that is off the grid like the output, and by another amount
        tr = _rows(hpt, owner, off, rows, cols)
        s = back(to(v + back(ar)[off:off + rows * cols].reshape(rows, cols)))
        _check(hpt, dtype, back(t.add_layernorm(tr, [cols], tg, tb, 1e-5).numpy()), s, g, b, f"{plan} residual off {off}")


# input and output off the grid by different amounts: the forms either side of single elements
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,rows,cols", [("f32", 9000, 97), ("f32", 8000, 160), ("f32", 8000, 215), ("f32", 4000, 263), ("f32", 400, 600), ("f32", 3000, 600),
                                             ("f16", 9000, 176), ("f16", 9000, 263), ("f16", 500, 900), ("bf16", 4000, 900), ("bf16", 200, 1100)])
def test_off_by_different_amounts(hpt, dev, dtype, rows, cols):
    to, back, dt = _codec(hpt, dtype)
    rng = np.random.default_rng(rows + cols)
    a = to(rng.standard_normal(rows * cols + 3).astype(np.float32) * 2)
    owner = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
    t = _rows(hpt, owner, 3, rows, cols)
    v = back(a)[3:].reshape(rows, cols)
    what = f"{dtype} {rows} x {cols} {hpt.normalize_plan(t, 0, 1)}"
    _check(hpt, dtype, back(t.layernorm([cols], None, None, 1e-5).numpy()), v, 1.0, 0.0, what)
    ar = to(rng.standard_normal((rows, cols)).astype(np.float32))
    s = back(to(v + back(ar)))
    _check(hpt, dtype, back(t.add_layernorm(hpt.Tensor.from_numpy(ar, dt).to_hip(dev), [cols], None, None, 1e-5).numpy()), s, 1.0, 0.0, what)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols", [(600, 9571), (530, 12531), (530, 16371), (100, 9571), (600, 9572), (600, 7335), (5000, 5121), (3500, 7335)])
def test_two_byte_softmax_of_long_odd_rows(hpt, dev, rows, cols):
    rng = np.random.default_rng(cols)
    a = (rng.standard_normal((rows, cols), dtype=np.float32) * 4).astype(np.float16)
    a[:, -1] += 5
    t = hpt.Tensor.from_numpy(a).to_hip(dev)
    plan = hpt.normalize_plan(t, 1)
    assert plan.startswith("rowreg-shift") and "unaligned" in plan.split(), plan
    for log in (False, True):
        got = (t.log_softmax(1) if log else t.softmax(1)).numpy()
        for r in range(0, rows, 1024):
            d = a[r:r + 1024].astype(np.float64)
            d -= d.max(1, keepdims=True)
            e = np.exp(d)
            want = d - np.log(e.sum(1, keepdims=True)) if log else e / e.sum(1, keepdims=True)
            assert_close(got[r:r + 1024], want, HALF_RTOL, max(half_atol(want, 11), 6e-8), f"{plan} log={log}")


# (plans alone, no device) rows, columns, elements that the input starts past a 16-byte boundary -> unaligned vectors, vector width
@pytest.mark.parametrize("dtype,rows,cols,off,unaligned,vec", [
    ("f32", 5000, 255, 0, True, 4), ("f32", 5000, 261, 0, True, 4), ("f32", 600, 4085, 0, True, 4), ("f32", 512, 261, 0, False, 4), ("f32", 600, 4097, 0, True, 4), ("f32", 512, 4097, 0, False, 4),
    ("f32", 512, 8185, 0, False, 4), ("f32", 512, 8195, 0, True, 4), ("f32", 90000, 127, 1, False, 1), ("f32", 90000, 130, 1, True, 4), ("f32", 90000, 215, 1, False, 1),
    ("f32", 90000, 263, 1, True, 4), ("f32", 2000, 390, 1, False, 1), ("f32", 100, 4100, 1, True, 4), ("f16", 2000, 600, 1, False, 1), ("f16", 3000, 600, 1, True, 8),
    ("f16", 100, 1100, 1, True, 8), ("f16", 3000, 133, 0, True, 8)])
def test_forms_of_layernorm_rows(hpt, dtype, rows, cols, off, unaligned, vec):
    size = {"f32": 4, "f16": 2}[dtype]
    t = hpt.Tensor.from_raw((1 << 40) + off * size, [rows, cols], getattr(hpt, dtype))
    plan, ua, v, *_ = _plan(hpt, t, 0, 1)
    assert (ua, v) == (unaligned, vec), plan
