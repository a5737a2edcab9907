"""Softmax over an axis of up to 1024 elements that is not the last: which inputs the kernel of whole vectors in 512 or 1024 threads takes and which stay
with the register columns or three launches (plans alone, no device), and the latter's results where the rule changed."""
import numpy as np
import pytest

from conftest import assert_close
from util import F32_ATOL, F32_RTOL, HALF_RTOL, half_atol


def _tall(plan):
    return plan.startswith("col-reg") and (" tpr=32 " in plan or " tpr=64 " in plan)


@pytest.mark.parametrize("dtype,shape,tall", [
    # four bytes, up to 256: whole segments up to one round of workgroups, a part of the second round, inner rows of a few vectors
    ("f32", (500, 256, 64), True), ("f32", (520, 256, 64), False), ("f32", (16, 222, 2244), False), ("f32", (24, 222, 2244), True), ("f32", (8181, 208, 12), False),
    ("f32", (8181, 208, 20), True), ("f32", (1024, 381, 14), False),
    # two bytes, 257 ... 512
    ("f16", (4200, 311, 16), False), ("f16", (4200, 311, 40), True), ("f16", (4200, 311, 10), True), ("f16", (489, 353, 11), False), ("f16", (5810, 323, 17), True),
    ("bf16", (22, 455, 3392), False), ("f16", (18, 259, 2816), True), ("f16", (15, 415, 2624), False), ("f16", (966, 544, 35), True), ("bf16", (8, 455, 3392), True), ("f16", (18, 410, 180), False),
    ("f16", (180, 410, 180), True),
    # two bytes, beyond 512
    ("f16", (19, 596, 3821), False), ("f16", (20, 1000, 801), True), ("f16", (90, 600, 517), True), ("f16", (40, 777, 1001), False), ("f16", (12, 600, 2051), True),
    ("f16", (12, 777, 2051), False), ("bf16", (1, 600, 801), False), ("f16", (536, 896, 180), False), ("f16", (700, 896, 180), True), ("f16", (98, 1000, 400), False), ("f16", (80, 1000, 400), True),
    ("f16", (140, 1000, 400), True), ("f16", (190, 1000, 400), False), ("f16", (3, 600, 10000), True), ("f16", (4, 600, 10000), False)])
def test_where_the_form_is_taken(hpt, dtype, shape, tall):
    plan = hpt.normalize_plan(hpt.Tensor.from_raw(1 << 40, list(shape), getattr(hpt, dtype)), 1)
    assert _tall(plan) == tall, plan


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,shape", [("f32", (520, 256, 64)), ("f32", (700, 208, 12)), ("f16", (900, 311, 16)), ("bf16", (900, 342, 27)), ("f16", (900, 353, 11)), ("bf16", (300, 290, 10)), ("f16", (18, 410, 180)),
                                         ("f16", (5, 700, 3821)), ("f16", (5, 596, 3821)), ("bf16", (90, 600, 517)), ("bf16", (270, 640, 200))])
def test_results_of_the_others(hpt, dev, dtype, shape):
    rng = np.random.default_rng(shape[2])
    x = (rng.standard_normal(shape, dtype=np.float32) * 3)
    x[:, 3, 0] = 30
    a, dt = (hpt.f32_to_bf16_bits(x), hpt.bf16) if dtype == "bf16" else (x.astype({"f32": np.float32, "f16": np.float16}[dtype]), None)
    back = hpt.bf16_bits_to_f32 if dtype == "bf16" else (lambda v: v)
    t = hpt.Tensor.from_numpy(a, dt).to_hip(dev)
    plan = hpt.normalize_plan(t, 1)
    v = back(a).astype(np.float64)
    d = v - v.max(1, keepdims=True)
    e = np.exp(d)
    for log in (False, True):
        got = back((t.log_softmax(1) if log else t.softmax(1)).numpy())
        want = d - np.log(e.sum(1, keepdims=True)) if log else e / e.sum(1, keepdims=True)
        if dtype == "f32":
            assert_close(got, want, F32_RTOL, F32_ATOL, plan)
        else:
            assert_close(got, want, HALF_RTOL, max(half_atol(want, 8 if dtype == "bf16" else 11), 6e-8), plan)
