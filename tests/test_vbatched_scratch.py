"""Register budget of the variable-size gesv kernel (vbatched.hpp).

The kernel's small-matrix packs and its large-matrix body share one register
file.  Lane numbers of the packs formed at kernel entry stay live through the
large body, which then spills them and reloads them in every step of a small
matrix: 124 bytes of scratch a lane made batches of orders up to 64 6 to 12 %
slower than 16 bytes did.  FP64 gesv, the widest instantiation, is compiled to
gfx950 assembly (device only) and its scratch read from the kernel descriptor.
"""
import os
import re
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_vbatched_dgesv_scratch(tmp_path):
    from rocsolver_amd import build
    src = os.path.join(build.CSRC, "vbatched_gesv_double.hip")
    out = str(tmp_path / "gesv.s")
    flags = [f for f in build.COMMON if f != "-fPIC"]
    r = subprocess.run([HIPCC, *flags, "--cuda-device-only", "-S", src, "-o", out],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    with open(out) as f:
        sizes = [int(x) for x in re.findall(r"\.private_segment_fixed_size:\s*(\d+)", f.read())]
    assert sizes and max(sizes) <= 16, sizes
