"""The site groups of the stencils by planes and the list of constrained links
with two staple sums, on the CPU: every group and every such link exactly once
(tests/cpp/plane_map_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_groups_and_pairs_are_listed_once(tmp_path):
    exe = tmp_path / "plane_map_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O2", "-std=c++17", "-x", "hip",
                    os.path.join(HERE, "cpp", "plane_map_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert len([ln for ln in r.stdout.splitlines() if ln.startswith("ok ")]) == 10
