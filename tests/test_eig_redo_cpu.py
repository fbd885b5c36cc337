"""Which matrices of a batched eigensolve the second solver redoes (svd_rule.h, eig_redos)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

MAIN = r"""
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "%s"
// argv: status of each matrix ("-": the solver writes none), then sums of squares
int main(int argc, char** argv) {
    std::vector<int> info;
    std::vector<double> sq;
    const int n = (argc - 1) / 2;
    for (int i = 0; i < n; ++i)
        if (strcmp(argv[1 + i], "-")) info.push_back(atoi(argv[1 + i]));
    for (int i = 0; i < n; ++i) sq.push_back(strtod(argv[1 + n + i], nullptr));
    for (int b : kv::eig_redos(info, sq)) printf("%%d ", b);
}
"""


@pytest.fixture(scope="module")
def redos(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("redo")
    src, exe = str(d / "m.cpp"), str(d / "m")
    with open(src, "w") as f:
        f.write(MAIN % os.path.join(ROOT, "kylin-v_amd", "csrc", "holstein", "svd_rule.h"))
    subprocess.run([gxx, "-std=c++17", "-O1", "-o", exe, src], check=True)

    def run(info, sumsq):
        out = subprocess.run([exe, *map(str, info), *map(str, sumsq)], check=True, capture_output=True, text=True)
        return [int(x) for x in out.stdout.split()]

    return run


@pytest.mark.parametrize("info,sumsq,want", [
    # no status: only what is not finite, whatever the others' state
    ("---", (3.0, "nan", 5.0), [1]), ("--", ("inf", "nan"), [0, 1]), ("--", (1.0, 2.0), []),
    # a status as well
    ((0, 2, 0), (3.0, 4.0, 5.0), [1]), ((0, 0, 1), ("nan", 4.0, 5.0), [0, 2]), ((0,), (0.0,), []),
])
def test_redo_list(redos, info, sumsq, want):
    assert redos(info, sumsq) == want
