"""Field transfers on the CPU, over a stand-in for the HIP runtime
(tests/cpp/transfer_check.cpp): every site moved once, whatever device the
calling thread is on; errors that earlier calls left behind not taken for the
transfer's own; at most 32 MiB of pinned slots."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    if shutil.which("hipcc") is None:
        pytest.skip("hipcc not on PATH")
    out = tmp_path_factory.mktemp("transfer") / "transfer_check"
    subprocess.run(["hipcc", "--offload-arch=gfx950", "-O1", "-std=c++17", "-x", "hip",
                    os.path.join(HERE, "cpp", "transfer_check.cpp"), "-o", str(out)],
                   check=True, capture_output=True, timeout=600)
    return str(out)


@pytest.mark.parametrize("check", ["device", "error", "bound"])
def test_transfers(exe, check):
    r = subprocess.run([exe, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout == f"ok {check}\n"
