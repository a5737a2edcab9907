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


# transposed views off the vector grid, stored [columns, rows]: where one group of lanes per row, register tiles and three passes
# meet - matrices of few elements were put through three launches
@pytest.mark.parametrize("dtype,cols,rows,softmax,layernorm", [
    ("f32", 64, 49, "transposed-tile-unaligned", "transposed-tile-unaligned"),
    ("f64", 32, 17, "transposed-tile-unaligned", "transposed-tile-unaligned"),
    ("f16", 300, 369, "transposed-tile-unaligned", "transposed-tile-unaligned"), ("f16", 300, 367, "generic", "generic"),
    ("bf16", 100, 120, "transposed-tile-unaligned", "transposed-tile-unaligned"), ("f16", 256, 90, "transposed-tile-unaligned", "transposed-tile-unaligned"),
    ("f16", 257, 90, "generic", "generic"), ("f32", 4096, 33, "transposed-tile-unaligned", "transposed-tile-unaligned"),
    ("f32", 4097, 33, "generic", "generic"), ("f32", 4608, 127, "generic", "transposed-unaligned"),
    ("f32", 6657, 127, "transposed-unaligned", "transposed-unaligned"), ("f32", 4097, 129, "transposed-unaligned", "transposed-unaligned"),
    ("f16", 6911, 127, "generic", "generic"), ("f16", 6912, 127, "generic", "transposed-unaligned"),
    ("bf16", 9984, 127, "transposed-unaligned", "transposed-unaligned"), ("f64", 4097, 33, "transposed-unaligned", "transposed-unaligned")])
def test_small_transposed_plans(hpt, dtype, cols, rows, softmax, layernorm):
    t = hpt.Tensor.from_raw(1 << 40, [cols, rows], getattr(hpt, dtype)).permute([1, 0])
    assert hpt.normalize_plan(t, 1).split()[0] == softmax
    assert hpt.normalize_plan(t, 0, 1).split()[0] == layernorm


# every second element of two-byte rows off the vector grid: few rows stay with single elements, which have more threads
@pytest.mark.parametrize("rows,stored,softmax,layernorm", [
    (340, 1763, "rowreg", "rowreg"), (850, 1763, "rowreg-step2", "rowreg"), (2268, 1763, "rowreg-step2", "rowreg-step2"), (389, 3853, "rowreg-step2", "rowreg"),
    (1038, 3853, "rowreg-step2", "rowreg-step2"), (50, 9001, "rowreg-step2", "rowreg-step2")])
def test_every_second_element_of_few_rows(hpt, rows, stored, softmax, layernorm):
    t = hpt.Tensor.from_raw(1 << 40, [rows, stored], hpt.f16)[:, ::2]
    assert (hpt.normalize_plan(t, 1).split()[0], hpt.normalize_plan(t, 0, 1).split()[0]) == (softmax, layernorm)
