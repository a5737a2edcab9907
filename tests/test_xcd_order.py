"""The order in which workgroups are dealt to the XCDs is a permutation, whatever the launch's size and the run's length, and neighbours land on one XCD: the
function itself, compiled for the host."""
import re
import subprocess
from pathlib import Path

import pytest

PROGRAM = r"""
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <vector>
#define __device__
#define __forceinline__ inline
using std::min;
@ORDER@
int main(int, char** v) {
    const int run = atoi(v[1]);
    for (unsigned n : {1u, 2u, 7u, 8u, 9u, 15u, 16u, 17u, 63u, 64u, 65u, 100u, 255u, 256u, 257u, 511u, 512u, 513u, 1000u, 2047u, 2048u, 2049u, 4097u, 65535u, 100003u, 3000001u}) {
        std::vector<unsigned> at(n, ~0u);
        for (unsigned i = 0; i < n; ++i) {
            const unsigned w = xcd_order(i, n, run);
            if (w >= n || at[w] != ~0u) return printf("run 2^%d of %u: %u -> %u\n", run, n, i, w), 1;
            at[w] = i & 7;  // the XCD of part w
        }
        unsigned changes = 0;  // where neighbouring parts are on different XCDs
        for (unsigned w = 1; w < n; ++w) changes += at[w] != at[w - 1];
        const unsigned long long group = 8ull << run, most = 8 * (n / group) + 8;
        if (changes > most) return printf("run 2^%d of %u: %u changes, %llu at most\n", run, n, changes, most), 1;
    }
    return 0;
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    import os
    header = (Path(__file__).resolve().parent.parent / "hpt_amd" / "csrc" / "device_utils.hpp").read_text()
    found = re.search(r"^__device__ __forceinline__ unsigned xcd_order\(.*?^}\n", header, re.M | re.S)
    assert found, "xcd_order is not in device_utils.hpp"
    d = tmp_path_factory.mktemp("xcd")
    (d / "order.cpp").write_text(PROGRAM.replace("@ORDER@", found[0]))
    r = subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", str(d / "order.cpp"), "-o", str(d / "order")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    return d / "order"


# single workgroups, pairs, eight and 32 in a row, eight equal shares of the launch
@pytest.mark.parametrize("run_log2", [0, 1, 3, 5, 28])
def test_a_permutation_in_runs(program, run_log2):
    r = subprocess.run([str(program), str(run_log2)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
