"""Splitting of batches over launches (rocsolver_amd/csrc/launch_split.hpp).

A launch takes fewer than 2^32 work-items in one grid dimension (a larger grid
can wrap around without an error).  The header has no HIP in it: it is compiled with the host compiler
and its parts are checked at the edges of that limit for every workgroup size
in use -- each below it, all of them together the whole batch, every group of
every system once.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "rocsolver_amd", "csrc")

PROGRAM = r"""
#include "launch_split.hpp"
#include <cstdio>
#include <cstdlib>
int main(int, char** v)
{
    long n = 0;
    return rsa::launch_split(atoll(v[1]), atoll(v[2]), atoi(v[3]), atoi(v[4]),
                             [&](int64_t s0, int64_t ns, int64_t g0, int64_t ng) {
                                 printf("%lld %lld %lld %lld\n", (long long)s0, (long long)ns,
                                        (long long)g0, (long long)ng);
                                 return ++n == atol(v[5]) ? 7 : 0;
                             });
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("no host compiler")
    d = tmp_path_factory.mktemp("split")
    src, exe = str(d / "split.cpp"), str(d / "split")
    with open(src, "w") as f:
        f.write(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-Wall", "-Werror", f"-I{CSRC}", src, "-o", exe], check=True)
    return exe


def parts(program, systems, groups, threads, unit, stop=0):
    r = subprocess.run([program, *map(str, (systems, groups, threads, unit, stop))],
                       capture_output=True, text=True)
    return r.returncode, [tuple(map(int, l.split())) for l in r.stdout.splitlines()]


@pytest.mark.parametrize("threads", [64, 128, 256, 512])
@pytest.mark.parametrize("unit", [1, 8])
@pytest.mark.parametrize("groups", [1, 2, 17, 32, 1 << 17, (1 << 25) - 1])
def test_parts(program, threads, unit, groups):
    cap = (2 ** 32 - 1) // threads
    edge = max(1, cap // groups)
    for systems in {1, 7, 8, 9, edge - 1, edge, edge + 1, edge + 9, 3 * edge + 5}:
        if not 1 <= systems < 2 ** 31:
            continue
        rc, got = parts(program, systems, groups, threads, unit)
        assert rc == 0
        covered, at = 0, {}
        for s0, ns, g0, ng in got:
            assert s0 % unit == 0 and ns > 0 and ng > 0
            assert -(-ns // unit) * unit * ng * threads < 2 ** 32
            # the groups of one range of systems follow each other without a gap
            assert g0 == at.get((s0, ns), 0)
            at[(s0, ns)] = g0 + ng
            covered += ns * ng
        assert covered == systems * groups
        assert all(g == groups for g in at.values())
        ranges = sorted(at)
        assert ranges[0][0] == 0 and sum(n for _, n in ranges) == systems
        assert all(a + n == b for (a, n), (b, _) in zip(ranges, ranges[1:]))
        # one launch where one is enough
        if -(-systems // unit) * unit * groups * threads < 2 ** 32:
            assert len(got) == 1


def test_empty_and_error(program):
    assert parts(program, 0, 5, 64, 8) == (0, [])
    assert parts(program, 5, 0, 64, 8) == (0, [])
    rc, got = parts(program, 3 << 24, 1, 256, 1, stop=2)  # the second launch fails
    assert rc == 7 and len(got) == 2
