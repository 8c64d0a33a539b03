"""The LDS-tiled top kernel on the CPU, over the grid it is launched on: the
blocks past the lattice neither load nor store (tests/cpp/top_tile_bounds_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_blocks_past_the_lattice_do_nothing(tmp_path):
    exe = tmp_path / "top_tile_bounds_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O1", "-std=c++20", "-x", "hip",
                    os.path.join(HERE, "cpp", "top_tile_bounds_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert len([ln for ln in r.stdout.splitlines() if ln.startswith("ok ")]) == 4
