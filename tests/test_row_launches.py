"""The grids of the row kernels for very many rows, on the CPU: reduction.hip's host code
linked with recorded launches (row_launch_check.cpp)."""
import subprocess
from pathlib import Path

import pytest

from oct_amd import build

HERE = Path(__file__).resolve().parent


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    out = tmp_path_factory.mktemp("row_launches") / "check"
    # The host half alone: the device code's symbol stays unresolved and unused.
    cmd = [build._hipcc(), "--offload-host-only", f"--offload-arch={build.ARCH}", "-O1", "-std=c++17", "-x", "hip",
           "-no-hip-rt", "-Wl,--unresolved-symbols=ignore-all", f"-I{build.REPO_DIR / 'include'}",
           str(HERE / "row_launch_check.cpp"), str(build.CSRC_DIR / "reduction.hip"), "-o", str(out), "-pthread"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    return out


# one, four and sixteen waves per row: 2^26, 2^24 and 2^22 rows are 2^32 threads
@pytest.mark.parametrize("rows,width", [(1, 64), (1000, 3840), ((1 << 24) - 1, 2048), (1 << 24, 1025), (1 << 24, 4096),
                                        ((1 << 22) - 1, 8192), (1 << 22, 4100), (5 << 21, 5000), (1 << 26, 256)])
def test_every_row_is_launched(check, rows, width):
    proc = subprocess.run([str(check), str(rows), str(width)], capture_output=True, text=True, timeout=60)
    assert proc.returncode == 0, proc.stdout + proc.stderr
