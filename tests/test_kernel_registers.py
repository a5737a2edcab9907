"""Registers of the layernorm row kernels and of tall softmax columns, as the compiler reports them: a compute unit holds as many wavefronts as fit its registers, so a
change that costs a kernel a few of them costs time although every result stays the same. Compiled here for gfx950, nothing is launched."""
import re
import subprocess
from pathlib import Path

import pytest

# (kernel, most vector registers, most of them spilled): 512 of each of a compute unit's lanes, given out in eights, so 96 leave room for
# five wavefronts on each of its four SIMDs, 80 for six, 64 for eight, 128 for four
LIMITS = [
    # f16 [16384, 4096]: four vectors per thread, gamma / beta in LDS
    ("row_reg_kernel<NORM_LAYERNORM, f16_t, 8, 4, 1, false, false, 1, 1>", 96, 0),
    # f16 rows of three vectors per thread, x + residual as well
    ("row_reg_kernel<NORM_ADD_LAYERNORM, f16_t, 8, 3, 1, false, false, 1, 1>", 96, 0),
    # f32 [3276, 10240], [2730, 12288]: five and six vectors, the next row loaded ahead ([2730, 12288] 63 us with 14 spilled, 49 with 8)
    ("row_reg_kernel<NORM_LAYERNORM, float, 4, 5, 1, false, true, 0, 1>", 128, 0),
    ("row_reg_kernel<NORM_LAYERNORM, float, 4, 6, 1, false, true, 0, 1>", 128, 8),
    # f64 [1059, 5632]
    ("row_reg_kernel<NORM_LAYERNORM, double, 2, 6, 1, false, true, 0, 1>", 128, 20),
    # f32 [1024, 32768]: eight vectors, gamma / beta from L2
    ("row_reg_kernel<NORM_LAYERNORM, float, 4, 8, 1, false, true, 2, 1>", 120, 0),
    # every second element: f32 and f16
    ("row_reg_kernel<NORM_LAYERNORM, float, 4, 4, 2, false, false, 0, 1>", 80, 0),
    ("row_reg_kernel<NORM_LAYERNORM, f16_t, 8, 2, 2, false, false, 0, 1>", 64, 0),
    # f32 [8192, 4096]
    ("row_reg_kernel<NORM_LAYERNORM, float, 4, 4, 1, false, false, 0, 1>", 104, 0),
]

COLUMNS = [
    # softmax over an axis in the middle, f32 [512, 512, 512] and unaligned [476, 475, 53], log_softmax: held to 64 registers, so that two workgroups of 1024
    # threads share a compute unit
    ("col_tall_kernel<NORM_SOFTMAX, float, 1024, 16, 8, false, false>", 64, 0),
    ("col_tall_kernel<NORM_SOFTMAX, float, 1024, 32, 8, true, true>", 64, 0),
    ("col_tall_kernel<NORM_LOGSOFTMAX, float, 1024, 16, 8, true, false>", 64, 3),
    ("col_tall_kernel<NORM_LOGSOFTMAX, float, 1024, 32, 8, true, true>", 64, 3),
]


@pytest.fixture(scope="module")
def report(tmp_path_factory):
    from hpt_amd import build
    if not Path(build.HIPCC).exists():
        pytest.skip("needs hipcc")
    src = tmp_path_factory.mktemp("registers") / "kernels.hip"
    src.write_text('#include "transpose_norm.hpp"\nnamespace hpt {\n' + "".join(f"template __global__ void {k}(const {'ColRegArgs' if k.startswith('col') else 'NormArgs'});\n" for k, _, _ in LIMITS + COLUMNS) + "}\n")
    flags = [f for f in build.FLAGS if not f.startswith("--offload-compress")]
    r = subprocess.run([build.HIPCC, *flags, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-c", str(src), "-o", "/dev/null"],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    found = {}
    for line in r.stderr.splitlines():
        m = re.search(r"remark:\s+(Function Name|VGPRs|VGPRs Spill): (\S+)", line)
        if m and m[1] == "Function Name":
            kernel = found.setdefault(m[2], {})
        elif m:
            kernel[m[1]] = int(m[2])
    return found


def _mangled(kernel: str) -> str:
    """The part of a kernel's mangled name that its template arguments make up."""
    name, args = re.match(r"(\w+)<(.*)>", kernel).groups()
    codes = {"NORM_SOFTMAX": "Li0E", "NORM_LOGSOFTMAX": "Li1E", "NORM_LAYERNORM": "Li2E", "NORM_ADD_LAYERNORM": "Li3E", "f16_t": "DF16_", "float": "f", "double": "d", "false": "Lb0E", "true": "Lb1E"}
    return name + "I" + "".join(codes.get(a, f"Li{a}E") for a in args.split(", "))


@pytest.mark.parametrize("kernel,registers,spilled", LIMITS)
def test_layernorm_rows_keep_their_wavefronts(report, kernel, registers, spilled):
    match = [v for k, v in report.items() if _mangled(kernel) in k]
    assert len(match) == 1, f"{kernel}: {sorted(report)}"
    assert match[0]["VGPRs"] <= registers and match[0]["VGPRs Spill"] <= spilled, f"{kernel}: {match[0]}"


@pytest.mark.parametrize("kernel,registers,spilled", COLUMNS)
def test_tall_columns_keep_two_workgroups(report, kernel, registers, spilled):
    test_layernorm_rows_keep_their_wavefronts(report, kernel, registers, spilled)
