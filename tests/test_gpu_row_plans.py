"""Row reductions and RMSNorm at the edges of their plans: one wave, four or sixteen
waves per row, rows over several workgroups; widths beside each boundary, rows at
any 4-byte address, infinities and NaN.

Sums and the oracle accumulate in binary64, so an output carries a few fp32
roundings of its own (exp, reciprocal, products): 8 ulps covers them.
"""
import threading
import time

import numpy as np
import pytest

import oracle
from oct_amd import prometheus as p

pytestmark = pytest.mark.gpu

WIDTHS = [1, 3, 4, 255, 256, 257, 1023, 1024, 1025, 2047, 2049, 4096, 4097, 8191, 8192, 8193, 16384, 16385, 32767,
          32768, 32769, 65536, 70001]


class Device:
    """fp32 arrays on the device, `shift` floats past an aligned address."""

    def __init__(self, rt, shift):
        self.rt, self.shift, self.held = rt, shift, []

    def new(self, count):
        self.held.append(self.rt.alloc((count + self.shift) * 4))
        return self.held[-1] + 4 * self.shift

    def put(self, x):
        ptr = self.new(x.size)
        self.rt.upload(ptr, np.ascontiguousarray(x, np.float32))
        return ptr

    def get(self, ptr, shape):
        self.rt.synchronize()
        return self.rt.download(np.empty(shape, np.float32), ptr)

    def free(self):
        for ptr in self.held:
            self.rt.free(ptr)


def reduce_on_device(rt, x, op, shift=0):
    d = Device(rt, shift)
    rows, width = x.shape
    shape = (rows, width) if op == p.OP_SOFTMAX else (rows,)
    out = d.new(int(np.prod(shape)))
    rt.reduction_device(d.put(x), out, rows, width, op)
    got = d.get(out, shape)
    d.free()
    return got


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("width", WIDTHS)
def test_rows_against_binary64(gpu_runtime, width, shift):
    rows = 40 if width in (16385, 32768) else 5  # more than 32 rows stay whole up to 32768
    x = oracle.normal(width, (rows, width), 0.0, 3.0)
    x64 = x.astype(np.float64)
    assert np.array_equal(reduce_on_device(gpu_runtime, x, p.OP_MAX, shift), x.max(axis=1))
    s = reduce_on_device(gpu_runtime, x, p.OP_SUM, shift)
    assert np.all(np.abs(s - x64.sum(axis=1)) <= 2.0 ** -23 * np.abs(x64).sum(axis=1))
    e = np.exp(x64 - x64.max(axis=1, keepdims=True))
    ref = e / e.sum(axis=1, keepdims=True)
    y = reduce_on_device(gpu_runtime, x, p.OP_SOFTMAX, shift)
    # (x - max) log2 e is rounded before the short rows' exp2: |x - max| ulps more
    spread = np.abs(x64 - x64.max(axis=1, keepdims=True))
    assert np.all(np.abs(y - ref) <= (8 + 2 * spread) * 2.0 ** -24 * ref + 1e-37)


@pytest.mark.parametrize("pad", [0, 5])
@pytest.mark.parametrize("width", [w for w in WIDTHS if w > 1])
def test_rmsnorm_against_binary64(gpu_runtime, width, pad):
    rows = 40 if width in (16385, 32768) else 5
    full = oracle.normal(width + 1, (rows, width + pad))
    x64, w = full[:, :width].astype(np.float64), oracle.normal(width + 2, (width,), 1.0, 0.1)
    d = Device(gpu_runtime, 0)
    out, inv = d.new(rows * width), d.new(rows)
    gpu_runtime.rmsnorm_device(d.put(full), d.put(w), out, inv, rows, width, width + pad, 1e-6)
    y, i = d.get(out, (rows, width)), d.get(inv, (rows,))
    d.free()
    ref = 1.0 / np.sqrt(np.mean(x64 * x64, axis=1) + 1e-6)
    assert np.all(np.abs(i - ref) <= 8 * 2.0 ** -24 * ref)
    want = x64 * ref[:, None] * w
    assert np.all(np.abs(y - want) <= 8 * 2.0 ** -24 * np.abs(want) + 1e-37)


@pytest.mark.parametrize("width", [300, 3001, 9000, 40000])
def test_infinities_and_nan(gpu_runtime, width):
    """A NaN counts for a maximum only as the row's first value; a stretch of negative
    infinities (a masked part of a row) adds nothing; a row of nothing else is NaN."""
    x = oracle.normal(9, (6, width))
    x[0, width // 2:] = -np.inf
    x[1, :-1] = -np.inf
    x[2, 7] = np.nan
    x[3, 0] = np.nan
    x[4, width - 2] = np.inf
    x[5] = -np.inf
    m = reduce_on_device(gpu_runtime, x, p.OP_MAX)
    assert m[0] == x[0].max() and m[1] == x[1, -1] and m[2] == np.nanmax(x[2]) and np.isnan(m[3])
    assert m[4] == np.inf and m[5] == -np.inf
    y = reduce_on_device(gpu_runtime, x, p.OP_SOFTMAX)
    e = np.exp(x[0].astype(np.float64) - x[0].max())
    assert np.allclose(y[0], e / e.sum(), rtol=4e-6, atol=0)
    assert np.all(y[1, :-1] == 0) and y[1, -1] == 1
    assert np.all(np.isnan(y[2:6]))
    s = reduce_on_device(gpu_runtime, x, p.OP_SUM)
    assert s[0] == -np.inf and s[1] == -np.inf and np.isnan(s[2]) and np.isnan(s[3])
    assert s[4] == np.inf and s[5] == -np.inf


@pytest.mark.parametrize("op", [p.OP_SUM, p.OP_SOFTMAX])
def test_more_parts_than_the_buffer_holds(gpu_runtime, op):
    """26220 rows of 5 parts each go in blocks of 2^17 // 5 = 26214 rows."""
    rt, rows, width = gpu_runtime, 26220, 32769
    picks = [0, 26213, 26214, 26219]
    d = Device(rt, 0)
    src = d.new(rows * width)
    dst = d.new(rows * width if op == p.OP_SOFTMAX else rows)
    x = oracle.normal(5, (len(picks), width))
    for i, row in enumerate(picks):
        rt.upload(src + 4 * row * width, x[i])
    rt.reduction_device(src, dst, rows, width, op)
    for i, row in enumerate(picks):
        v = x[i].astype(np.float64)
        if op == p.OP_SUM:
            want, got, ulps = np.array([v.sum()]), d.get(dst + 4 * row, (1,)), 8.0
        else:
            # x - max and its product with log2 e round once each, and the power takes
            # both errors, |x - max| half ulps each, as relative ones
            e = np.exp(v - v.max())
            want, got, ulps = e / e.sum(), d.get(dst + 4 * row * width, (width,)), 8 + 2 * np.abs(v - v.max())
        assert np.all(np.abs(got - want) <= ulps * 2.0 ** -24 * np.abs(want) + 1e-37), row
    d.free()


@pytest.mark.parametrize("op,rows,width", [(p.OP_SUM, 64, 4096), ("rmsnorm", 64, 2048), (p.OP_SOFTMAX, 8, 65536)])
def test_device_reductions_do_not_wait_for_a_host_call(gpu_runtime, op, rows, width):
    """A device-pointer reduction is queued at once while another thread's host-pointer
    product (6 ms, its copies included) holds the runtime's buffers."""
    rt = gpu_runtime
    n = 4096
    a = np.ones((n, n), np.float32)
    x, w = rt.upload_new(np.ones((rows, width), np.float32)), rt.upload_new(np.ones(width, np.float32))
    out = rt.alloc(rows * width * 4)

    def reduce():
        if op == "rmsnorm":
            rt.rmsnorm_device(x, w, out, None, rows, width, width, 1e-6)
        else:
            rt.reduction_device(x, out, rows, width, op)

    windows = []

    def products():
        for _ in range(3):
            t0 = time.perf_counter()
            rt.sgemm(n, n, n, a, a)
            windows.append((t0, time.perf_counter()))

    try:
        reduce()
        rt.sgemm(n, n, n, a, a)
        thread = threading.Thread(target=products)
        thread.start()
        calls = []
        while thread.is_alive() and len(calls) < 3000:
            t0 = time.perf_counter()
            reduce()
            calls.append((t0, time.perf_counter()))
            time.sleep(2e-4)
        thread.join()
        rt.synchronize()
    finally:
        for ptr in (x, w, out):
            rt.free(ptr)
    inside = sum(any(t0 < c0 and c1 < t1 for t0, t1 in windows) for c0, c1 in calls)
    # one that waits for the product returns with it: at most the first and last of each
    assert inside >= 12, (inside, len(calls), [t1 - t0 for t0, t1 in windows])
