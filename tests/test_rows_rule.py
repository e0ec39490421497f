"""Which of two ways a solve takes (rocsolver_amd/csrc/rows_rule.hpp).

The header has no HIP in it: the host compiler builds it, and the rule is
checked at points on both sides of its lines where both kernels were timed.
Beyond 8 right-hand sides the tiles always win.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rocsolver_amd", "csrc")

PROGRAM = r"""
#include "rows_rule.hpp"
#include <cstdio>
int main()
{
    char type, op;
    int n, bc, nrhs;
    while(scanf(" %c %c %d %d %d", &type, &op, &n, &bc, &nrhs) == 5)
    {
        bool rows;
        if(n > 512)
        {
            const int tiles = (n + 127) / 128;
            puts((type == 'd' ? rsa::trsm_many<double>(op == 'T', tiles, nrhs, bc)
                              : rsa::trsm_many<float>(op == 'T', tiles, nrhs, bc))
                     ? "many" : "step");
            continue;
        }
        if(op == 'C')
            rows = type == 'd' ? rsa::potrs_by_rows<double>(n, nrhs, bc)
                               : rsa::potrs_by_rows<float>(n, nrhs, bc);
        else
            rows = type == 'd' ? rsa::getrs_by_rows<double>(op == 'T', n, nrhs, bc)
                               : rsa::getrs_by_rows<float>(op == 'T', n, nrhs, bc);
        puts(rows ? "rows" : "tiles");
    }
}
"""

# type, op (N, T: getrs; C: potrs), order, systems, right-hand sides, the faster kernel
MEASURED = [
    # getrs
    ("d", "N", 65, 512, 1, "rows"), ("d", "N", 96, 512, 1, "tiles"),
    ("d", "N", 65, 2048, 1, "rows"), ("d", "N", 128, 8192, 4, "rows"),
    ("d", "N", 256, 1024, 4, "rows"), ("d", "N", 304, 2904, 8, "rows"),
    ("d", "N", 96, 512, 4, "tiles"), ("d", "N", 512, 64, 1, "tiles"),
    ("d", "N", 128, 8192, 8, "tiles"), ("d", "T", 97, 8192, 4, "rows"),
    ("d", "T", 129, 1024, 1, "rows"), ("d", "T", 128, 8192, 4, "tiles"),
    ("d", "T", 256, 4096, 1, "tiles"), ("s", "N", 65, 512, 1, "rows"),
    ("s", "N", 128, 8192, 4, "rows"), ("s", "N", 304, 640, 4, "rows"),
    ("s", "N", 304, 768, 8, "rows"), ("s", "N", 304, 1024, 4, "tiles"),
    ("s", "N", 304, 1280, 4, "rows"), ("s", "N", 512, 512, 1, "tiles"),
    ("s", "T", 65, 8192, 1, "rows"), ("s", "T", 83, 8192, 4, "rows"),
    ("s", "T", 96, 8192, 4, "tiles"), ("s", "T", 512, 1024, 1, "tiles"),
    # blocked getrs: updates in launches of their own, or with the solves step by step
    ("d", "T", 513, 300, 100, "many"), ("d", "T", 800, 64, 600, "many"),
    ("d", "N", 513, 150, 33, "many"), ("s", "T", 800, 64, 600, "many"),
    ("s", "N", 600, 150, 40, "many"), ("d", "N", 513, 1, 2000, "step"),
    ("d", "N", 2500, 4, 64, "step"), ("s", "N", 2500, 1, 2000, "step"),
    ("s", "N", 600, 300, 1, "step"), ("s", "N", 600, 300, 17, "many"),
    ("s", "T", 1100, 64, 1, "step"), ("s", "T", 1100, 64, 17, "many"),
    ("d", "T", 1024, 64, 8, "step"), ("d", "T", 600, 150, 8, "many"), ("d", "N", 2000, 1, 1, "step"),
    # potrs
    ("d", "C", 1, 65536, 1, "rows"), ("d", "C", 8, 4096, 4, "rows"),
    ("d", "C", 32, 2048, 1, "rows"), ("d", "C", 64, 4096, 1, "rows"),
    ("d", "C", 129, 4096, 4, "rows"), ("d", "C", 257, 1280, 4, "rows"),
    ("d", "C", 32, 1024, 1, "tiles"), ("d", "C", 64, 4096, 4, "tiles"),
    ("d", "C", 512, 1024, 4, "tiles"), ("d", "C", 16, 16384, 8, "tiles"),
    ("s", "C", 1, 65536, 1, "rows"), ("s", "C", 8, 4096, 4, "rows"),
    ("s", "C", 33, 4096, 4, "rows"), ("s", "C", 65, 3072, 4, "rows"),
    ("s", "C", 129, 3072, 1, "rows"), ("s", "C", 64, 1536, 4, "tiles"),
    ("s", "C", 96, 1024, 1, "tiles"), ("s", "C", 128, 2048, 4, "tiles"),
]


def test_rule_at_measured_points(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    src, exe = str(tmp_path / "rule.cpp"), str(tmp_path / "rule")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", f"-I{CSRC}", src, "-o", exe], check=True)
    points = list(MEASURED)
    for t, op, n, bc, _, _ in MEASURED:  # more than 8 right-hand sides
        points += [(t, op, n, bc, r, "tiles") for r in (9, 16, 100) if n <= 512]
    # no batch is large enough where rows never win
    points += [("d", "T", 512, 2 ** 31 - 1, 1, "tiles"), ("s", "C", 512, 2 ** 31 - 1, 1, "tiles")]
    text = "\n".join(" ".join(map(str, p[:5])) for p in points)
    r = subprocess.run([exe], input=text, capture_output=True, text=True, check=True)
    got = r.stdout.split()
    assert len(got) == len(points)
    wrong = [(p, g) for p, g in zip(points, got) if p[5] != g]
    assert not wrong, wrong
