"""The walks that deal site blocks to the XCDs, on the CPU: every block once
(tests/cpp/walk_map_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_every_block_once(tmp_path):
    exe = tmp_path / "walk_map_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O2", "-std=c++17", "-x", "hip",
                    os.path.join(HERE, "cpp", "walk_map_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split("\n")[:-1] == ["ok run_block", "ok wloop_block", "ok tile_map"]
