"""Rows off the vector grid as unaligned vectors, the last one from the row's end backwards: softmax, log_softmax, layernorm, layernorm of
a sum and the causal softmax at row lengths either side of vectors, threads per row, vectors per thread and the forms that follow;
rows whose input and output are misaligned by different amounts; in place. Which of them are unaligned vectors and which masked aligned ones is the
plan's choice; test_gpu_walked_rows_off_grid.py asserts it, with more rows than one round of workgroups."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu

# (rows, stored columns, first column, columns)
SHAPES = [(7, 129, 0, 129), (33, 135, 0, 135), (5, 136, 1, 128), (9, 263, 2, 257), (3000, 519, 0, 519), (12, 639, 0, 639), (2100, 641, 0, 641), (9, 805, 0, 805),
          (17, 1030, 3, 1024), (5, 2202, 0, 2202), (3, 4097, 0, 4097), (2, 4105, 0, 4105), (3, 8191, 0, 8191), (130, 16377, 0, 16377), (130, 16385, 0, 16385)]


def _store(hpt, dtype, x):
    if dtype == "bf16":
        return hpt.f32_to_bf16_bits(x), hpt.bf16
    return x.astype({"f16": np.float16, "f32": np.float32}[dtype]), None


def _wide(hpt, dtype, a):
    return (hpt.bf16_bits_to_f32(a) if dtype == "bf16" else a).astype(np.float64)


def _check(hpt, dtype, got, want, what):
    got = _wide(hpt, dtype, got)
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan), what
    inf = np.isneginf(want)
    assert np.array_equal(np.isneginf(got), inf), what
    keep = ~(nan | inf)
    if dtype == "f32":
        assert_close(got[keep], want[keep], F32_RTOL, F32_ATOL, what)
    else:
        assert_close(got[keep], want[keep], HALF_RTOL, max(half_atol(want[keep], 8 if dtype == "bf16" else 11), 6e-8), what)


def _softmax(x, log):
    with np.errstate(invalid="ignore"):
        d = x - x.max(-1, keepdims=True)
        s = np.exp(d).sum(-1, keepdims=True)
        return d - np.log(s) if log else np.exp(d) / s


def _layernorm(x, g, b):
    d = x - x.mean(-1, keepdims=True)
    y = d / np.sqrt((d * d).mean(-1, keepdims=True) + 1e-5)
    return y * (1 if g is None else g) + (0 if b is None else b)


@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_unaligned_rows(hpt, dev, dtype, shape):
    rows, stored, first, cols = shape
    rng = np.random.default_rng(stored)
    x = (rng.standard_normal((rows, stored)) * 2 + rng.uniform(-3, 3, (rows, 1))).astype(np.float32)
    x[1, first] = 30          # the row's ends decide
    x[0, first + cols - 1] = 30
    a, dt = _store(hpt, dtype, x)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)[:, first:first + cols]
    v = _wide(hpt, dtype, a)[:, first:first + cols]
    what = f"{dtype} {shape}"
    for log in (False, True):
        _check(hpt, dtype, (t.log_softmax(1) if log else t.softmax(1)).numpy(), _softmax(v, log), f"{what} softmax log={log}")
    (ga, _), (ba, _) = (_store(hpt, dtype, rng.normal(m, 0.1, cols + 1).astype(np.float32)) for m in (1, 0))
    g, b = _wide(hpt, dtype, ga)[1:], _wide(hpt, dtype, ba)[1:]
    tg, tb = (hpt.Tensor.from_numpy(u, dt).to_hip(dev)[1:] for u in (ga, ba))  # off the grid themselves
    for gg, bb, p, q in ((tg, tb, g, b), (tg, None, g, None), (None, None, None, None)):
        _check(hpt, dtype, t.layernorm([cols], gg, bb, 1e-5).numpy(), _layernorm(v, p, q), f"{what} layernorm")
    ra, _ = _store(hpt, dtype, rng.standard_normal((rows, cols)).astype(np.float32))
    tr = hpt.Tensor.from_numpy(ra, dt).to_hip(dev)
    s = _wide(hpt, dtype, _store(hpt, dtype, (v + _wide(hpt, dtype, ra)).astype(np.float32))[0])
    _check(hpt, dtype, t.add_layernorm(tr, [cols], tg, tb, 1e-5).numpy(), _layernorm(s, g, b), f"{what} add_layernorm")
    if first == 0:  # in place, of the whole tensor
        for f, want in ((lambda u, o: u.softmax(1, out=o), t.softmax(1)), (lambda u, o: u.layernorm([cols], tg, tb, 1e-5, out=o), t.layernorm([cols], tg, tb, 1e-5))):
            u = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
            f(u, u)
            assert u.numpy().tobytes() == want.numpy().tobytes(), what


# every second element of the rows: odd pitches, odd first elements, the row's last element the last of the memory or not, 512 threads per
# row and more (whose workgroups walk the rows), aligned and not, and rows too long for the registers
@pytest.mark.parametrize("dtype", ["f16", "bf16", "f32"])
@pytest.mark.parametrize("rows,stored,first", [(5, 129, 0), (9, 130, 1), (33, 263, 0), (3, 1027, 2), (2100, 517, 1), (2100, 1279, 0), (9, 1281, 0), (600, 7897, 0), (5, 12287, 0), (5, 12291, 0), (3, 8190, 1), (530, 8192, 0), (2, 16385, 0),
                                               (2, 32767, 0), (2, 32770, 1)])
def test_every_second_element(hpt, dev, dtype, rows, stored, first):
    rng = np.random.default_rng(stored + first)
    x = (rng.standard_normal((rows, stored)) * 2).astype(np.float32)
    x[-1, -1] = x[-1, -2] = 25
    x[0, first] = 25
    a, dt = _store(hpt, dtype, x)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)[:, first::2]
    v = _wide(hpt, dtype, a)[:, first::2]
    cols = v.shape[1]
    what = f"{dtype} [{rows}, {stored}][:, {first}::2] {hpt.normalize_plan(t, 1)[:40]}"
    for log in (False, True):
        _check(hpt, dtype, (t.log_softmax(1) if log else t.softmax(1)).numpy(), _softmax(v, log), f"{what} softmax log={log}")
    (ga, _), (ba, _), (ra, _) = (_store(hpt, dtype, rng.normal(m, 0.1, n).astype(np.float32)) for m, n in ((1, cols), (0, cols), (0, (rows, cols))))
    tg, tb, tr = (hpt.Tensor.from_numpy(u, dt).to_hip(dev) for u in (ga, ba, ra))
    g, b = _wide(hpt, dtype, ga), _wide(hpt, dtype, ba)
    _check(hpt, dtype, t.layernorm([cols], tg, tb, 1e-5).numpy(), _layernorm(v, g, b), f"{what} layernorm")
    s = _wide(hpt, dtype, _store(hpt, dtype, (v + _wide(hpt, dtype, ra)).astype(np.float32))[0])
    _check(hpt, dtype, t.add_layernorm(tr, [cols], tg, tb, 1e-5).numpy(), _layernorm(s, g, b), f"{what} add_layernorm")
    got = t.softmax_causal(1.0, cols - rows if cols > rows else 3).numpy()
    kept = np.arange(cols)[None, :] <= np.arange(rows)[:, None] + (cols - rows if cols > rows else 3)
    _check(hpt, dtype, got, _softmax(np.where(kept, v, -np.inf), False), f"{what} causal")


@pytest.mark.parametrize("dtype", ["f16", "bf16"])
@pytest.mark.parametrize("heads,queries,keys", [(3, 40, 131), (2, 300, 301), (4, 9, 805), (1, 70, 2202), (2, 5, 4097), (1, 3, 9001)])
def test_causal_rows(hpt, dev, dtype, heads, queries, keys):
    rng = np.random.default_rng(keys)
    a, dt = _store(hpt, dtype, (rng.standard_normal((heads, queries, keys)) * 8).astype(np.float32))
    v = _wide(hpt, dtype, a)
    for offset in (keys - queries, 0, 5, -2):
        kept = np.arange(keys)[None, :] <= np.arange(queries)[:, None] + offset
        scaled = _wide(hpt, dtype, _store(hpt, dtype, (v * 0.25).astype(np.float32))[0])
        want = _softmax(np.where(kept, scaled, -np.inf), False)
        # nothing of what is masked may come in: those keys are NaN
        poisoned = _store(hpt, dtype, np.where(kept, v, np.nan).astype(np.float32))[0]
        got = hpt.Tensor.from_numpy(poisoned, dt).to_hip(dev).softmax_causal(0.25, offset).numpy()
        _check(hpt, dtype, got, want, f"{dtype} {heads}x{queries}x{keys} offset {offset}")
