"""Host-pointer calls of every copy size: one piece by the copy kernel (up to 512 KiB,
any byte tail), chunks by kernel and by DMA, and many calls through the same pinned
slots, each with data of its own.  The result must be the device-pointer entry's."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def on_device(rt, a, b):
    m, k = a.shape
    n = b.shape[1]
    ptrs = [rt.upload_new(a), rt.upload_new(b), rt.alloc(m * n * 4)]
    rt.sgemm_device(*ptrs, m, n, k)
    rt.synchronize()
    out = rt.download(np.empty((m, n), np.float32), ptrs[2])
    for ptr in ptrs:
        rt.free(ptr)
    return out


# operand bytes beside 16, 512 KiB (362 * 362 * 4 = 524176, 363 * 361 * 4 = 524172, 512 * 256 * 4 = 512 KiB),
# 1 MiB, 2 MiB and several chunks
@pytest.mark.parametrize("m,n,k", [(1, 1, 1), (1, 3, 5), (3, 5, 7), (127, 129, 131), (362, 362, 362), (363, 361, 363),
                                   (512, 513, 256), (512, 512, 512), (700, 749, 751), (1000, 1300, 530)])
def test_sizes(gpu_runtime, m, n, k):
    a, b = oracle.uniform(m, (m, k)), oracle.uniform(n + 1, (k, n))
    out, _ = gpu_runtime.sgemm(m, n, k, a, b)
    np.testing.assert_array_equal(np.asarray(out).reshape(m, n), on_device(gpu_runtime, a, b))


def test_slots_are_reused_with_fresh_data(gpu_runtime):
    shapes = [(64, 64, 64), (200, 210, 220), (513, 300, 400), (16, 700, 900)]
    for i in range(60):
        m, n, k = shapes[i % len(shapes)]
        a = np.full((m, k), np.float32(i + 1))
        b = np.full((k, n), np.float32(1 + i % 3))
        out, _ = gpu_runtime.sgemm(m, n, k, a, b)
        assert np.all(np.asarray(out) == np.float32((i + 1) * (1 + i % 3) * k))


def test_batch_uploads_run_ahead_of_the_device(gpu_runtime):
    """A batch queues its uploads, products and downloads without a wait between them: operands
    of 1 to 8 MiB, which leave a slot in the middle, and 20 MiB, which come round the ring."""
    shapes = [(75, 975, 2048), (320, 64, 4096), (16, 1280, 4096), (300, 300, 1000), (64, 2000, 975)]
    problems = []
    for i in range(48):
        m, n, k = shapes[i % len(shapes)]
        problems.append((np.full((m, k), np.float32(i + 1)), np.full((k, n), np.float32(1 + i % 3))))
    rc, status, outs = gpu_runtime.sgemm_batch(problems)
    assert rc == 0, status
    for i, (out, (a, _)) in enumerate(zip(outs, problems)):
        # every partial sum is a whole number below 2^24: exact in any order
        assert np.all(out == np.float32((i + 1) * (1 + i % 3) * a.shape[1])), i
