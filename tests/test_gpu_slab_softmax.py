"""Softmax over the middle axis of contiguous [batch, C, L] with a narrow L, one workgroup per slab: lengths around whole
vectors (0 to 7 elements left over), around what a number of threads and vectors per thread hold, slabs off the 16-byte
grid, columns that share vectors in every way, against the oracle. One column has no finite entry."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol

pytestmark = pytest.mark.gpu

SHAPES = [(3, 64, 2), (5, 65, 3), (2, 66, 5), (7, 67, 7), (4, 128, 4), (9, 127, 6), (2, 191, 5), (300, 79, 3), (37, 512, 8), (11, 513, 4),
          (6, 681, 6), (5, 1365, 3), (3, 1366, 3), (8, 1639, 5), (3, 2340, 7), (2, 2341, 7), (2, 4096, 8), (2, 4095, 8), (3, 4095, 5), (300, 3071, 4),
          (1100, 216, 4), (1100, 341, 3), (5000, 125, 7)]


@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
@pytest.mark.parametrize("shape", SHAPES, ids=lambda v: "x".join(map(str, v)))
def test_slab_softmax(hpt, orc, dev, shape, dtype):
    x = (np.random.default_rng(55).standard_normal(shape) * 3).astype(np.float32)
    x[0, :, 1] = -np.inf
    x[-1, -1, -1] = 40  # the last element of all dominates its column
    ident = lambda v: v
    cv, tof, dt, odt, bits, acc = {
        "f32": (ident, ident, None, None, 0, orc.ACC_F64),
        "f64": (lambda v: v.astype(np.float64), ident, None, None, 0, orc.ACC_F64),
        "f16": (lambda v: v.astype(np.float16), lambda v: v.astype(np.float32), None, None, 11, orc.ACC_F32),
        "bf16": (hpt.f32_to_bf16_bits, hpt.bf16_bits_to_f32, hpt.bf16, orc.BF16, 8, orc.ACC_F32),
    }[dtype]
    a = cv(x)
    whole = hpt.Tensor.from_numpy(np.concatenate([a.reshape(-1)[:1], a.reshape(-1)]), dt).to_hip(dev)
    for off in (0, 1):  # on the 16-byte grid, and one element past it
        flat = hpt.Tensor.from_numpy(a.reshape(-1), dt).to_hip(dev) if off == 0 else whole[1:]
        t = hpt.Tensor.from_raw(flat.ptr, list(shape), flat.dtype, dev)
        plan = hpt.normalize_plan(t, 1)
        print(plan, flush=True)
        if shape[0] * shape[1] * shape[2] * flat.dtype.size < 4 << 20 and shape[1] * shape[2] * flat.dtype.size <= 112 << 10:  # (7 of 1024 threads' places may not take part)
            assert plan.startswith("col-slab"), plan
        for log in (False, True):
            got = tof((t.log_softmax(1) if log else t.softmax(1)).numpy())
            want = tof(orc.softmax(a, 1, log=log, acc=acc, dtype=odt))
            dead = np.isnan(want)
            assert dead[0, :, 1].all() and dead.sum() == shape[1] and np.isnan(got[dead]).all()
            ok = ~dead
            atol = max(half_atol(want[ok], bits), 6e-8 if bits == 11 else 0) if bits else F32_ATOL
            assert_close(got[ok], want[ok], HALF_RTOL if bits else F32_RTOL, atol, f"{shape} {dtype} log={log} off={off}")
