"""The block maps of batched stencil launches, on the CPU: every site block of
every chain exactly once, and no XCD with more of them than its share
(tests/cpp/batch_map_check.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="hipcc not on PATH")
def test_every_block_of_every_chain_once(tmp_path):
    exe = tmp_path / "batch_map_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "--offload-host-only", "-O2", "-std=c++17", "-x", "hip",
                    os.path.join(HERE, "cpp", "batch_map_check.cpp"), "-o", str(exe)],
                   check=True, capture_output=True, timeout=600)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert len([ln for ln in r.stdout.splitlines() if ln.startswith("ok ")]) == 7
