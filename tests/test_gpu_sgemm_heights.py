"""The 64x128 tile of the fp32 SGEMM, the GeGLU product's tile heights and the GEMV's
row tails, at their edges, against binary64 (bound as in test_gpu_sgemm_rows.py)."""
import numpy as np
import pytest

import oracle
from oct_amd import prometheus as p

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1056, 2816, 512), (1088, 1000, 256), (321, 4096, 2048), (832, 3980, 1952)])
def test_tall_products(gpu_runtime, m, n, k):
    a, b = oracle.uniform(m, (m, k)), oracle.uniform(n, (k, n))
    out, _ = gpu_runtime.sgemm(m, n, k, a, b)
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (k + 16) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(np.asarray(out).reshape(m, n) - a64 @ b64) <= bound)


@pytest.mark.parametrize("m,k,shift", [(1, 1, 0), (5, 3, 1), (9, 255, 1), (130, 257, 0), (64, 1026, 1), (33, 4099, 0),
                                       (7, 8191, 1), (1000, 62, 0)])
def test_gemv_row_tails(gpu_runtime, m, k, shift):
    rt = gpu_runtime
    a, x = oracle.uniform(m, (m, k)), oracle.uniform(k, (k,))
    held = [rt.alloc((c + shift) * 4) for c in (m * k, k, m)]
    da, dx, dy = (ptr + 4 * shift for ptr in held)
    rt.upload(da, a)
    rt.upload(dx, x)
    rt.sgemm_device(da, dx, dy, m, 1, k)
    rt.synchronize()
    y = rt.download(np.empty(m, np.float32), dy)
    for ptr in held:
        rt.free(ptr)
    a64, x64 = a.astype(np.float64), x.astype(np.float64)
    assert np.all(np.abs(y - a64 @ x64) <= (k + 16) * 2.0 ** -24 * (np.abs(a64) @ np.abs(x64)))


@pytest.mark.parametrize("tokens", [49, 64, 65, 128, 129, 160, 192, 193, 300])
def test_geglu_tile_heights(gpu_runtime, tokens):
    from oracle import blocks

    x, w = blocks.make_decoder_layer(4, tokens, 512, 2, 128, 1024)
    rc, res, out = gpu_runtime.decoder_layer_f32(x, w, 2, 128)
    assert rc == p.PROM_OK, (res.stage, res.detail_code)
    assert oracle.normwise_rel_err(out, blocks.decoder_layer_f32(x, w, 2, 128)) <= 1e-5
