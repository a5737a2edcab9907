"""Every plan of the register row kernels has a kernel: tests/cpp/row_forms.cpp holds what the planner (hpt_amd/csrc/layout.cpp) gives to rows on and
off the vector grid against the numbers of vectors per thread that the launcher is compiled for. Pure host code: no GPU, no HIP runtime."""
import pathlib
import shutil
import subprocess

import pytest

ROOT = pathlib.Path(__file__).resolve().parents[1]


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_row_plan_has_a_kernel(tmp_path):
    exe = tmp_path / "row_forms"
    cmd = ["g++", "-std=c++17", "-O2", f"-I{ROOT / 'include'}", f"-I{ROOT / 'hpt_amd' / 'csrc'}", "-I/opt/rocm/include",
           "-D__HIP_PLATFORM_AMD__", "-x", "c++", str(ROOT / "hpt_amd" / "csrc" / "layout.cpp"),
           str(ROOT / "tests" / "cpp" / "row_forms.cpp"), "-o", str(exe)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout[-6000:]
