"""The rounding error of the FP32 plans that replaced the 64x64 direct-to-LDS tiles on
unaligned operands, on row counts that 128 divides badly and on few rows: no larger than
theirs on the same product (zero-padded for them; both against the binary64 product, the
2-norm over 10^4 to 4 10^6 outputs, whose ratio varies by a few per cent)."""
import numpy as np
import pytest

import oracle
from oct_amd import prometheus as p

pytestmark = pytest.mark.gpu


def _error(got, exact):
    return np.linalg.norm(got - exact) / np.linalg.norm(exact)


@pytest.mark.parametrize("m,n,k,tile,slices", [
    # staged tiles on unaligned rows, unsliced and sliced
    (1565, 2224, 101, 5, 1), (349, 380, 2966, 6, 12), (1951, 149, 1307, 5, 6),
    # the 64x128 direct-to-LDS tile
    (2446, 2112, 512, 5, 1),
    # few rows
    (1, 2816, 1024, 5, 16), (6, 9344, 512, 5, 6), (15, 2048, 1536, 5, 12)])
def test_error_is_no_larger_than_the_64x64_tiles(gpu_runtime, m, n, k, tile, slices):
    rt = gpu_runtime
    a, b = oracle.uniform(m + k, (m, k)), oracle.uniform(n, (k, n))
    exact = a.astype(np.float64) @ b.astype(np.float64)
    out, _ = rt.sgemm(m, n, k, a, b)
    k4, n4 = (k + 3) // 4 * 4, (n + 3) // 4 * 4
    held = [rt.upload_new(np.pad(a, ((0, 0), (0, k4 - k)))), rt.upload_new(np.pad(b, ((0, k4 - k), (0, n4 - n)))),
            rt.alloc(m * n4 * 4)]
    assert rt.sgemm_device_variant(*held, m, n4, k4, tile, slices)[0] == p.PROM_OK
    rt.synchronize()
    tiles = rt.download(np.empty((m, n4), np.float32), held[2])[:, :n]
    for ptr in held:
        rt.free(ptr)
    got, theirs = _error(np.asarray(out).reshape(m, n), exact), _error(tiles, exact)
    print(f"{m}x{n}x{k}: {got:.3e}, the 64x64 tiles {theirs:.3e}", flush=True)
    assert got <= 1.08 * theirs
