"""Plans at the limits of what a launch may be, asked of the planner alone: no device memory is touched."""
import pytest


# a workgroup of 64 or 128 threads per [cols, L] slab, 2^32 work-items per launch at most; beyond, the plan of before
@pytest.mark.parametrize("dtype,slabs,cols,width,beyond", [
    ("bf16", 1 << 26, 97, 2, "col-group-tile"), ("f32", 1 << 26, 64, 3, "col-group-tile"), ("f32", 1 << 25, 401, 3, "col rows")])
def test_slab_softmax_within_one_launch(hpt, dtype, slabs, cols, width, beyond):
    def plan(n):
        return hpt.normalize_plan(hpt.Tensor.from_raw(1 << 40, [n, cols, width], getattr(hpt, dtype)), 1)
    assert plan(slabs - 1).startswith("col-slab"), plan(slabs - 1)
    assert plan(slabs).startswith(beyond), plan(slabs)
