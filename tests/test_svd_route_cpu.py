"""Which solver takes a small sector of a bond SVD (svd_rule.h, jacobi_takes and jacobi_slower_alone)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include "%s"
int main(int, char** argv) {
    const long nr = atol(argv[1]), nc = atol(argv[2]);
    const double cutoff = atof(argv[3]);
    printf("%%d %%d", (int)kv::jacobi_takes(nr, nc, cutoff), (int)kv::jacobi_slower_alone(nr, nc, cutoff));
}
"""


@pytest.fixture(scope="module")
def route(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("route")
    src, exe = str(d / "m.cpp"), str(d / "m")
    with open(src, "w") as f:
        f.write(MAIN % os.path.join(ROOT, "kylin-v_amd", "csrc", "holstein", "svd_rule.h"))
    subprocess.run([gxx, "-std=c++17", "-O1", "-o", exe, src], check=True)

    def run(nr, nc, cutoff):
        out = subprocess.run([exe, str(nr), str(nc), str(cutoff)], check=True, capture_output=True, text=True)
        return tuple(map(int, out.stdout.split()))

    return run


# (rows, columns, cutoff) -> taken at all, left to rocSOLVER where it is the only such sector
CASES = [
    # every value kept: any size up to the kernel's limits, long wide sectors and columns not
    ((1, 1, -1.0), (1, 0)), ((64, 64, -1.0), (1, 0)), ((65, 65, -1.0), (0, 0)), ((4161, 63, -1.0), (1, 0)),
    ((63, 4162, -1.0), (0, 0)), ((6144, 1, -1.0), (1, 0)), ((6145, 1, -1.0), (1, 1)), ((16384, 1, -1.0), (1, 1)),
    ((16385, 1, -1.0), (0, 1)), ((131072, 2, -1.0), (1, 0)), ((32768, 8, -1.0), (1, 0)),
    ((16, 6144, -1.0), (1, 0)), ((16, 6145, -1.0), (1, 1)), ((8, 16385, -1.0), (0, 1)),
    # truncating: from a longer side of 128
    ((127, 60, 0.0), (0, 0)), ((128, 60, 0.0), (1, 0)), ((2, 128, 1e-10), (1, 0)), ((262144, 1, 1e-10), (1, 0)),
    ((16, 6145, 1e-10), (1, 0)), ((63, 4161, 0.0), (1, 0)), ((8192, 31, 0.0), (1, 0)),
]


@pytest.mark.parametrize("sector,want", CASES)
def test_route_of_a_small_sector(route, sector, want):
    assert route(*sector) == want
