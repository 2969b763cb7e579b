"""Launches that the host code chooses, recorded on the CPU (recorded_launches.h): the grids
of the row kernels for very many rows, and the kernel of the decoder layer's GeGLU product."""
import subprocess
from pathlib import Path

import pytest

from oct_amd import build

HERE = Path(__file__).resolve().parent


def compiled(out, check, *sources):
    # The host half alone: the device code's symbol stays unresolved and unused.
    cmd = [build._hipcc(), "--offload-host-only", f"--offload-arch={build.ARCH}", "-O1", "-std=c++17", "-x", "hip",
           "-no-hip-rt", "-Wl,--unresolved-symbols=ignore-all", f"-I{build.REPO_DIR / 'include'}",
           str(HERE / check), *(str(build.CSRC_DIR / s) for s in sources), "-o", str(out), "-pthread"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    assert proc.returncode == 0, proc.stdout + proc.stderr
    return out


@pytest.fixture(scope="module")
def rows_check(tmp_path_factory):
    return compiled(tmp_path_factory.mktemp("row_launches") / "check", "row_launch_check.cpp", "reduction.hip")


@pytest.fixture(scope="module")
def geglu_check(tmp_path_factory):
    return compiled(tmp_path_factory.mktemp("geglu_launches") / "check", "geglu_launch_check.cpp", "sgemm_f32.hip",
                    "sgemm_rows.hip")


# one, four and sixteen waves per row: 2^26, 2^24 and 2^22 rows are 2^32 threads
@pytest.mark.parametrize("rows,width", [(1, 64), (1000, 3840), ((1 << 24) - 1, 2048), (1 << 24, 1025), (1 << 24, 4096),
                                        ((1 << 22) - 1, 8192), (1 << 22, 4100), (5 << 21, 5000), (1 << 26, 256)])
def test_every_row_is_launched(rows_check, rows, width):
    proc = subprocess.run([str(rows_check), str(rows), str(width)], capture_output=True, text=True, timeout=60)
    assert proc.returncode == 0, proc.stdout + proc.stderr


# up to 48 rows: the few-rows kernel, or the 64-row tile where it measured faster (a layer of
# 48 tokens, 2048 x 2 * 81920: 555 us and 539; of 16: 448 and 497) and can run
@pytest.mark.parametrize("rows,columns,k,kernel", [
    (1, 16384, 2048, "rows"), (48, 16384, 2048, "rows"), (48, 4096, 1024, "rows"), (16, 81920, 2048, "rows"),
    (48, 81920, 2048, "tiles"), (48, 81890, 2048, "rows"), (48, 81920, 2040, "rows"), (49, 16384, 2048, "tiles"),
    (200, 16384, 2040, "none")])
def test_geglu_kernel_of_a_shape(geglu_check, rows, columns, k, kernel):
    proc = subprocess.run([str(geglu_check), str(rows), str(columns), str(k)], capture_output=True, text=True,
                          timeout=60)
    assert proc.returncode == 0 and proc.stdout.split() == [kernel], proc.stdout + proc.stderr
