"""FP32 products whose rows are not 16-byte aligned or whose K is not whole tiles: the
register-staged kernels' loads at any alignment, the direct-to-LDS tiles' K tail, the
few-rows tail of a taller product, and the sum of K slices with a ragged last column."""
import ctypes

import numpy as np
import pytest

import oracle
from oct_amd import prometheus as p

# (m, n, k): K tails 4, 8 and 12 on 128-row tiles; unaligned rows of A alone, of B
# alone, of both; one column past a 4-wide group; one row past a tile; K below a tile
SHAPES = [(256, 256, 20), (640, 640, 1032), (384, 2304, 124), (129, 128, 516), (4097, 1001, 130), (176, 3000, 513),
          (2000, 100, 101), (1000, 101, 72), (128, 129, 1027), (561, 1833, 1475), (65, 66, 3), (3261, 340, 2070)]


def _check(rt, m, n, k, run):
    a, b = oracle.uniform(m + k, (m, k)), oracle.uniform(n, (k, n))
    # what lies past the operands must not reach the result, nor the result what lies
    # past it: NaN on either side of all three, which are 4-byte aligned only
    gap = 513
    at_a, at_b, at_c = gap, 2 * gap + m * k, 3 * gap + m * k + k * n
    host = np.full(at_c + m * n + gap, np.nan, np.float32)
    host[at_a:at_a + m * k], host[at_b:at_b + k * n] = a.ravel(), b.ravel()
    held = rt.alloc(host.nbytes)
    rt.upload(held, host)
    run(held + 4 * at_a, held + 4 * at_b, held + 4 * at_c)
    rt.synchronize()
    out = rt.download(np.empty_like(host), held)
    rt.free(held)
    got = out[at_c:at_c + m * n].reshape(m, n)
    assert np.isnan(out[at_b + k * n:at_c]).all() and np.isnan(out[at_c + m * n:]).all()
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    # each product and each of its additions rounds once, in any order
    bound = (k + 16) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_ragged_products(gpu_runtime, m, n, k):
    rt = gpu_runtime

    def run(a, b, c):
        rt.sgemm_device(a, b, c, m, n, k)

    _check(rt, m, n, k, run)


@pytest.mark.gpu
@pytest.mark.parametrize("tile", [0, 1, 2])
@pytest.mark.parametrize("slices", [1, 3])
@pytest.mark.parametrize("m,n,k", [(129, 257, 401), (64, 130, 258)])
def test_staged_tiles_at_any_alignment(gpu_runtime, tile, slices, m, n, k):
    rt = gpu_runtime

    def run(a, b, c):
        assert rt.sgemm_device_variant(a, b, c, m, n, k, tile, slices)[0] == p.PROM_OK

    _check(rt, m, n, k, run)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [2, 3, 4, 5, 6, 7, 103, 1025, 1027])
def test_sums_of_slices_for_any_column_count(gpu_runtime, n):
    """The slices' sum takes four columns per thread, the last ones together with columns that
    another thread stores, and one per thread below four; 130 rows of 13 slices."""
    rt = gpu_runtime
    m, k = 130, 1040

    def run(a, b, c):
        assert rt.sgemm_device_variant(a, b, c, m, n, k, 2, 13)[0] == p.PROM_OK

    _check(rt, m, n, k, run)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k", [(256, 256, 20), (640, 640, 1032), (384, 2304, 124), (129, 128, 516),
                                   (2944, 2816, 60)])
def test_k_tail_of_aligned_operands(gpu_runtime, m, n, k):
    a, b = oracle.uniform(m, (m, k)), oracle.uniform(n, (k, n))
    out, _ = gpu_runtime.sgemm(m, n, k, a, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (k + 16) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(np.asarray(out).reshape(m, n) - a64 @ b64) <= bound)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_ragged_plans_fit_their_report(m, n, k):
    info = p.PrometheusSgemmPlanInfo()
    info.struct_size = ctypes.sizeof(info)
    assert p.shared_library().prometheus_reactor_sgemm_plan(m, n, k, ctypes.byref(info)) == p.PROM_OK
    assert info.launches == 2 * info.repacked + sum(2 if s > 1 else 1 for s in info.k_slices[:info.products])
    assert info.head_rows == m or (info.products == 2 and info.head_rows % 128 == 0 and m - info.head_rows < 128)
    kk = (k + 3) // 4 * 4 if info.repacked else k
    for i in range(info.products):
        assert info.k_slices[i] == 1 or info.k_slice_len[i] * info.k_slices[i] >= kk - 16 * info.k_slices[i]


@pytest.mark.parametrize("m,n,k", [(14050, 976, 6828), (2109, 1518, 3169), (5722, 4096, 1581), (168, 11520, 6074),
                                   (3496, 4276, 11340), (620, 2527, 3414), (8192, 4784, 8200)])
def test_ragged_plans_stay_within_the_noalloc_scratch(m, n, k):
    """Tall products with K tails and unaligned rows that have a plan within the
    allocation-free entry's scratch take one."""
    info = p.PrometheusSgemmPlanInfo()
    info.struct_size = ctypes.sizeof(info)
    assert p.shared_library().prometheus_reactor_sgemm_plan(m, n, k, ctypes.byref(info)) == p.PROM_OK
    assert info.scratch_bytes <= p.SGEMM_NOALLOC_SCRATCH_BYTES
