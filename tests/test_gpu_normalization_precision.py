"""Rows that a careless statistic gets wrong: layernorm rows whose first element lies far from the rest (nothing may be summed
around that element alone in 32 bits), and f16 log_softmax rows with a large common offset (nothing may round the offset
before it is subtracted). Against numpy in 64 bits or more."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL

pytestmark = pytest.mark.gpu


def _normalised(x):
    """layernorm over the last axis without weights, eps 1e-5, in long double."""
    x = x.astype(np.longdouble)
    d = x - x.mean(-1, keepdims=True)
    return d / np.sqrt((d * d).mean(-1, keepdims=True) + np.longdouble(1e-5))


def _check_layernorm(hpt, got, x, dtype, what, f64_units=16):
    """`x` holds the rows as they were stored, `got` what came back, both as floats. f64_units: what f64 rows may be off by,
    in units of 2^-53 - the roundings of the mean, of 1 / sqrt and of the product, and what a sum around a far element loses."""
    want = _normalised(x)
    err = np.linalg.norm((got.astype(np.longdouble) - want).astype(np.float64))
    size = np.linalg.norm(want.astype(np.float64))
    if dtype == "f32":
        # the project's gate for every element, and over all of them two roundings of an f32 (2^-24 each, 3e-8 rms)
        assert_close(got, want.astype(np.float64), F32_RTOL, F32_ATOL, what)
        assert err < 2.0 ** -22 * size, f"{what}: {err / size:g}"
    elif dtype == "f64":
        assert err < f64_units * 2.0 ** -53 * size, f"{what}: {err / size:g}"
    else:  # what rounding the exact result costs, and a twentieth more for the 32 bits in between
        w32 = want.astype(np.float32)
        rounded = w32.astype(np.float16).astype(np.float64) if dtype == "f16" else \
            hpt.bf16_bits_to_f32(hpt.f32_to_bf16_bits(w32)).astype(np.float64)
        assert err < 1.05 * np.linalg.norm(rounded - want.astype(np.float64)), f"{what}: {err / size:g}"


def _stored(hpt, x, dtype):
    """(what goes to the device, its dtype, the values it holds)"""
    if dtype == "bf16":
        bits = hpt.f32_to_bf16_bits(x.astype(np.float32))
        return bits, hpt.bf16, hpt.bf16_bits_to_f32(bits)
    a = x.astype({"f32": np.float32, "f16": np.float16, "f64": np.float64}[dtype])
    return a, None, a


# stored [(batch,) columns, rows]: several workgroups share the columns (off and on the vector grid), or one has them all
TRANSPOSED = [(shape, first) for shape in [(5001, 131), (5000, 136)] for first in (0, 20, 100, 1000, 30000)]
TRANSPOSED += [(shape, first) for shape in [(260, 4099, 65), (257, 4104, 64)] for first in (0, 1000)]


@pytest.mark.parametrize("shape,first", TRANSPOSED, ids=str)
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
def test_layernorm_of_transposed_rows_with_a_far_first_element(hpt, dev, shape, dtype, first):
    x = np.random.default_rng(3).standard_normal(shape)
    x[..., 0, :] += first
    a, dt, values = _stored(hpt, x, dtype)
    del x
    perm = list(range(len(shape) - 2)) + [len(shape) - 1, len(shape) - 2]
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev).permute(perm)
    plan = hpt.normalize_plan(t, 0, 1)
    assert plan.startswith("transposed ") or plan.startswith("transposed-unaligned "), plan
    got = t.layernorm([shape[-2]], None, None, 1e-5).numpy()
    if dtype == "bf16":
        got = hpt.bf16_bits_to_f32(got)
    some = slice(None) if len(shape) == 2 else slice(0, shape[0], 37)  # (batches: a sample)
    v = values.swapaxes(-1, -2)
    _check_layernorm(hpt, got[some], v[some], dtype, f"{shape} {dtype} first {first}: {plan}")


@pytest.mark.parametrize("first", [0, 100, 1000, 30000])
@pytest.mark.parametrize("shape", [(3, 1 << 20), (2, 300007), (100, 65539)], ids=lambda v: "x".join(map(str, v)))
@pytest.mark.parametrize("dtype", ["f32", "f16", "bf16", "f64"])
def test_layernorm_of_shared_rows_with_a_far_first_element(hpt, dev, shape, dtype, first):
    x = np.random.default_rng(4).standard_normal(shape)
    x[:, 0] += first
    a, dt, values = _stored(hpt, x, dtype)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
    plan = hpt.normalize_plan(t, 0, 1)
    assert plan.startswith("rowsplit"), plan
    got = t.layernorm([shape[1]], None, None, 1e-5).numpy()
    if dtype == "bf16":
        got = hpt.bf16_bits_to_f32(got)
    # (f64: the thread that holds the first element sums up to 32 elements around it)
    _check_layernorm(hpt, got, values, dtype, f"{shape} {dtype} first {first}: {plan}", f64_units=128)


@pytest.mark.parametrize("offset,step", [(0, 8), (1000, 8), (-1000, 8), (16000, 8), (-16000, 8)])
@pytest.mark.parametrize("shape", [(200, 1001), (200, 1000), (2000, 4099)], ids=lambda v: "x".join(map(str, v)))
def test_f16_log_softmax_of_transposed_rows_with_a_large_offset(hpt, dev, shape, offset, step):
    """One element `step` above the others, all far from zero: the result there is close to zero and shows every error of
    the logarithm of the sum. Allowed: half a unit of the last f16 place, and 1e-6 for the sum and its logarithm in f32."""
    x = np.full(shape, offset, np.float32)
    x[7] += step
    x[11::3] -= step
    a = x.astype(np.float16)
    assert np.array_equal(a.astype(np.float32), x)  # (the values are f16 numbers)
    t = hpt.Tensor.from_numpy(a).to_hip(dev).permute([1, 0])
    plan = hpt.normalize_plan(t, 1)
    assert plan.startswith("transposed-tile"), plan
    got = t.log_softmax(1).numpy().astype(np.float64)
    v = x.T.astype(np.float64)
    d = v - v.max(1, keepdims=True)
    want = d - np.log(np.exp(d).sum(1, keepdims=True))
    assert_close(got, want, 2.0 ** -11, 1e-6, f"{shape} offset {offset}: {plan}")
