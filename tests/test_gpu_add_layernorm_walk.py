"""layernorm(x + residual) of two-byte rows with gamma / beta in LDS: a workgroup loads the next row and its residual before it
normalises the current one. More rows than one round of workgroups, a last round that is partly empty, rows with idle
lanes, against numpy in float64; the result in place of x and in place of the residual."""
import numpy as np
import pytest

from conftest import assert_close
from util import HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu


# rows: workgroups are capped at 3072 (512 ... 1024 threads per row: the same), 8, 4, 2 or 1 rows each
@pytest.mark.parametrize("dtype,rows,cols", [
    ("f16", 24577, 648), ("f16", 3072 * 8 + 5, 1024), ("bf16", 12289, 1536), ("f16", 6143, 4096), ("bf16", 3073, 5120), ("f16", 3077, 5128),
    ("f16", 3090, 8192), ("bf16", 700, 16384), ("f16", 3, 5120), ("f16", 3100, 8200)])
def test_walked_rows(hpt, dev, dtype, rows, cols):
    rng = np.random.default_rng(rows + cols)
    x = (rng.standard_normal((rows, cols), dtype=np.float32) + rng.uniform(-5, 5, (rows, 1)).astype(np.float32))
    r = rng.standard_normal((rows, cols), dtype=np.float32)
    g, b = rng.normal(1, 0.1, cols).astype(np.float32), rng.normal(0, 0.1, cols).astype(np.float32)
    if dtype == "bf16":
        to, back, dt, bits = hpt.f32_to_bf16_bits, hpt.bf16_bits_to_f32, hpt.bf16, 8
    else:
        to, back, dt, bits = (lambda v: v.astype(np.float16)), (lambda v: v.astype(np.float32)), None, 11
    ax, ar, ag, ab = (to(v) for v in (x, r, g, b))
    s = back(to(back(ax) + back(ar))).astype(np.float64)  # x + residual is rounded to the dtype
    s -= s.mean(1, keepdims=True)
    want = s / np.sqrt((s * s).mean(1, keepdims=True) + 1e-5) * back(ag) + back(ab)
    tg, tb = (hpt.Tensor.from_numpy(v, dt).to_hip(dev) for v in (ag, ab))
    for place in ("fresh", "x", "residual"):
        tx, tr = hpt.Tensor.from_numpy(ax, dt).to_hip(dev), hpt.Tensor.from_numpy(ar, dt).to_hip(dev)
        out = tx.layernorm([cols], tg, tb, 1e-5, residual=tr, out={"fresh": None, "x": tx, "residual": tr}[place])
        assert_close(back(out.numpy()), want, HALF_RTOL, half_atol(want, bits), f"{dtype} {rows} x {cols}, {place}")


# f16 rows of three vectors per thread: from 7500 workgroups on 5120 of them walk the rows
@pytest.mark.parametrize("rows,cols", [(30001, 1032), (15001, 2056), (7505, 4104)])
def test_more_than_five_thousand_workgroups(hpt, dev, rows, cols):
    rng = np.random.default_rng(cols)
    ax, ar = (rng.standard_normal((rows, cols), dtype=np.float32).astype(np.float16) for _ in range(2))
    ag, ab = rng.normal(1, 0.1, cols).astype(np.float16), rng.normal(0, 0.1, cols).astype(np.float16)
    tx, tr, tg, tb = (hpt.Tensor.from_numpy(v).to_hip(dev) for v in (ax, ar, ag, ab))
    got = tx.add_layernorm(tr, [cols], tg, tb, 1e-5).numpy()
    for r in range(0, rows, 4096):
        s = (ax[r:r + 4096] + ar[r:r + 4096]).astype(np.float64)  # x + residual is rounded to the dtype
        s -= s.mean(1, keepdims=True)
        want = s / np.sqrt((s * s).mean(1, keepdims=True) + 1e-5) * ag.astype(np.float64) + ab
        assert_close(got[r:r + 4096], want, HALF_RTOL, half_atol(want, 11), f"{rows} x {cols}")
