"""The bf16 GEMM's macro tiles, K slices and padded copies, at their edges.

The oracle is numpy's binary64 product of the bf16 operands, widened exactly.
Every product of two bf16 values is exact in fp32, so an output differs from it
only by the fp32 sums: at most k roundings of partial sums no larger than
sum |a b|, in any order (MFMA, K slices): |err| <= k 2^-24 sum |a b|.
"""
import numpy as np
import pytest

import oracle
from oct_amd import prometheus as p

pytestmark = pytest.mark.gpu

SHAPES = [
    (1, 8, 8), (1, 128, 64), (31, 129, 72), (32, 128, 56), (33, 136, 64), (63, 64, 200), (65, 72, 1096),
    (96, 4096, 4096),    # K slices of a 32- or 64-row tile
    (129, 1000, 640), (193, 520, 264), (257, 3840, 1288), (300, 2056, 8),
    (700, 640, 2048), (1056, 3840, 512), (1500, 2000, 192), (2049, 1032, 328),
    # rows that are not 16-byte aligned: copies of A, of B, of both
    (200, 512, 333), (130, 333, 512), (257, 1001, 777), (64, 999, 2001), (5, 7, 9),
]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_bf16_tiles_against_oracle(gpu_runtime, m, n, k):
    a = oracle.to_bf16(oracle.uniform(m + k, (m, k)))
    b = oracle.to_bf16(oracle.uniform(n + k + 1, (k, n)))
    got = np.asarray(gpu_runtime.gemm_bf16(m, n, k, a, b)).reshape(m, n).astype(np.float64)
    a64, b64 = (oracle.from_bf16(x).astype(np.float64) for x in (a, b))
    bound = k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)


@pytest.mark.parametrize("m,n,k", [(40, 256, 72), (150, 384, 1160), (1056, 512, 328)])
def test_bf16_tail_of_k_reads_no_other_row(gpu_runtime, m, n, k):
    """A row of infinities stays in its own output row: the chunks of A past k, which
    lie in the next row, are not multiplied with the zero rows of B past k."""
    a = oracle.to_bf16(oracle.uniform(3, (m, k)))
    b = oracle.to_bf16(np.abs(oracle.uniform(4, (k, n))) + np.float32(0.5))
    a[m // 2] = oracle.to_bf16(np.full(k, np.inf, np.float32))
    got = np.asarray(gpu_runtime.gemm_bf16(m, n, k, a, b)).reshape(m, n)
    assert np.all(np.isposinf(got[m // 2]))
    assert np.all(np.isfinite(np.delete(got, m // 2, axis=0)))


@pytest.mark.parametrize("tokens,ffn", [(33, 200), (130, 1032), (600, 2048)])
def test_dit_block_swiglu_tiles(gpu_runtime, tokens, ffn):
    """Blocks whose W1|W3 product runs on the tiles, ffn not a multiple of the tile's columns."""
    from oracle import blocks

    heads = 4
    x, cond, w = blocks.make_dit_block(5, tokens, heads * 128, ffn, 32)
    coords = blocks.joint_coordinates(1, tokens, 0)
    rc, res, out = gpu_runtime.dit_block_bf16(x, coords, cond, w, heads=heads)
    assert rc == p.PROM_OK, (res.stage, res.detail_code)
    ref = blocks.dit_block_bf16(x, coords, cond, w, heads)
    # the block bar of test_gpu_blocks.py
    assert oracle.normwise_rel_err(out, ref) <= 2e-2
