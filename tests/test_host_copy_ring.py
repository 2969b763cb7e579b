"""The pinned ring of the host copies, on the CPU: host_copy.hip's host code linked with
a device whose queue runs only when it is waited for (host_copy_check.cpp), so that a
slot written before its last copy has run shows as wrong data."""
import subprocess
from pathlib import Path

import pytest

from oct_amd import build

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = tmp_path_factory.mktemp("host_copy") / "check"
    # The host half alone: the device code's symbol stays unresolved and unused.
    cmd = [build._hipcc(), "--offload-host-only", f"--offload-arch={build.ARCH}", "-O1", "-std=c++17", "-x", "hip",
           "-no-hip-rt", "-Wl,--unresolved-symbols=ignore-all", f"-I{build.REPO_DIR / 'include'}",
           str(HERE / "host_copy_check.cpp"), str(build.CSRC_DIR / "host_copy.hip"), "-o", str(out), "-pthread"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    return out


@pytest.mark.parametrize("mode", ["uploads", "mixed", "errors"])
def test_no_slot_is_written_before_its_copy_has_run(check, mode):
    proc = subprocess.run([str(check), mode], capture_output=True, text=True, timeout=100)
    assert proc.returncode == 0, proc.stdout + proc.stderr
