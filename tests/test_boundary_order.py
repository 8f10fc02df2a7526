"""The two sides of an axis that the ghost fill takes in one launch: the
copies' lines run on the host in several orders (the end's side first,
shuffled) must give what one side after the other gives, face for face
(tests/host/boundary_order.hip).  Random arrays: the face below the first cell
differs from the last face, also where the axis is periodic."""
import os
import subprocess

import pytest

from conftest import ROOT

HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
def test_both_sides_in_any_order(tmp_path):
    exe = str(tmp_path / "boundary_order")
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "-O1", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-I" + os.path.join(ROOT, "pluto_amd", "csrc"),
                    os.path.join(ROOT, "tests", "host", "boundary_order.hip"), "-o", exe],
                   check=True, capture_output=True, text=True)
    p = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert p.returncode == 0, p.stdout[-3000:] + p.stderr[-2000:]
