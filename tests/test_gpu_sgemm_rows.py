"""The fp32 SGEMM of few rows (sgemm_rows.hip) at its edges: every row-block count,
column tails, K tails, K slices, operands at any 4-byte address.

The oracle is the binary64 product; an output sums k fp32 products in some order,
so |err| <= (k + 16) 2^-24 sum |a b| (16 more roundings for the waves' and slices' sums).
"""
import numpy as np
import pytest

import oracle
from oct_amd import prometheus as p

pytestmark = pytest.mark.gpu

SHAPES = [(m, n, k) for m in (1, 15, 16, 17, 32, 33, 48) for n, k in ((64, 16), (333, 250), (2048, 1536))] + [
    (1, 2, 1), (2, 3, 5), (7, 129, 17), (16, 31, 1000), (31, 100, 4099), (48, 16, 8192), (3, 20000, 40),
    (15, 2048, 16384), (33, 1001, 1003), (49, 256, 512)]


def check(got, a, b):
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (a.shape[1] + 16) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_few_rows_against_oracle(gpu_runtime, m, n, k):
    a, b = oracle.uniform(m + n, (m, k)), oracle.uniform(n + k + 7, (k, n))
    out, _ = gpu_runtime.sgemm(m, n, k, a, b)
    check(np.asarray(out).reshape(m, n), a, b)


@pytest.mark.parametrize("m,n,k", [(5, 200, 37), (16, 1536, 257), (40, 129, 2050)])
def test_few_rows_unaligned_and_infinite_row(gpu_runtime, m, n, k):
    """Operands one float past an aligned address; a row of A that is not finite stays
    in its own output row although the next rows' K tails lie beside it."""
    rt = gpu_runtime
    a, b = oracle.uniform(1, (m, k)), np.abs(oracle.uniform(2, (k, n))) + np.float32(0.5)
    a[m // 2] = np.inf
    held = [rt.alloc((x.size + 1) * 4) for x in (a, b)] + [rt.alloc((m * n + 1) * 4)]
    da, db, dc = (ptr + 4 for ptr in held)
    rt.upload(da, a)
    rt.upload(db, b)
    rt.sgemm_device(da, db, dc, m, n, k)
    rt.synchronize()
    got = rt.download(np.empty((m, n), np.float32), dc)
    for ptr in held:
        rt.free(ptr)
    assert np.all(np.isposinf(got[m // 2]))
    keep = np.arange(m) != m // 2
    check(got[keep], a[keep], b)


@pytest.mark.parametrize("tokens,ffn", [(1, 96), (16, 200), (17, 1000), (48, 512)])
def test_decoder_layer_of_few_tokens(gpu_runtime, tokens, ffn):
    """The layer whose products, the gate|up one with GeGLU among them, are of few rows."""
    from oracle import blocks

    x, w = blocks.make_decoder_layer(3, tokens, 256, 2, 64, ffn)
    rc, res, out = gpu_runtime.decoder_layer_f32(x, w, 2, 64, position_offset=5)
    assert rc == p.PROM_OK, (res.stage, res.detail_code)
    ref = blocks.decoder_layer_f32(x, w, 2, 64, position_offset=5)
    assert oracle.normwise_rel_err(out, ref) <= 1e-5
