"""The bf16 GEMM's kernels, K slices and padded copies, at their edges: the plan's own
choice (32x128, 64x64 and 64x128 tiles at these sizes) and every kernel by number.

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


# macro tiles (rows, columns) and K tiles in flight (stages - 1) of kernels 0-8
TILES = [(32, 128, 3), (64, 64, 4), (64, 128, 2), (64, 256, 3), (128, 128, 3), (192, 128, 3), (128, 256, 2),
         (192, 256, 1), (256, 256, 1)]
SWIGLU_TILES = [2, 3, 4, 6, 7, 8, p.GEMM_BF16_FIVE_STAGE]


def run_variant(rt, a, b, tile, slices=1, swiglu=False):
    m, k = a.shape
    n = b.shape[1] // 2 if swiglu else b.shape[1]
    dtype = np.uint16 if swiglu else np.float32
    gap = 64  # what lies beside the output is not written
    host = np.full(m * n + 2 * gap, 7, dtype)
    held = [rt.upload_new(a), rt.upload_new(b), rt.upload_new(host)]
    rc, status = rt.gemm_bf16_device_variant(held[0], held[1], held[2] + gap * host.itemsize, m, n, k, tile, slices,
                                             p.GEMM_BF16_SWIGLU if swiglu else 0)
    assert rc == p.PROM_OK, status
    rt.synchronize()
    out = rt.download(np.empty_like(host), held[2])
    for ptr in held:
        rt.free(ptr)
    assert np.all(out[:gap] == 7) and np.all(out[-gap:] == 7)
    return out[gap:-gap].reshape(m, n)


def operands(m, n, k):
    a = oracle.to_bf16(oracle.uniform(m + k, (m, k)))
    b = oracle.to_bf16(oracle.uniform(n + k + 1, (k, n)))
    return a, b, oracle.from_bf16(a).astype(np.float64), oracle.from_bf16(b).astype(np.float64)


def edge_shapes(rows, columns, flight):
    return [(1, 8, 8), (rows - 1, columns + 8, 64), (rows + 1, columns - 8, 64 * flight + 8),
            (2 * rows + 33, 2 * columns + 40, 64 * (flight + 1)), (rows, columns, 64 * (2 * flight + 3) + 56)]


@pytest.mark.parametrize("slices", [1, 3])
@pytest.mark.parametrize("tile", range(9))
def test_every_tile_at_its_edges(gpu_runtime, tile, slices):
    """One row and column past and short of a tile, K tails, fewer K tiles than the ring has
    stages, as many, and more; slices of unequal K (at least one K tile each)."""
    for m, n, k in edge_shapes(*TILES[tile]):
        if (k + 63) // 64 < slices:
            continue
        a, b, a64, b64 = operands(m, n, k)
        got = run_variant(gpu_runtime, a, b, tile, slices).astype(np.float64)
        bound = (k + slices) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
        assert np.all(np.abs(got - a64 @ b64) <= bound), (m, n, k)


@pytest.mark.parametrize("tile", range(9))
def test_every_tile_keeps_an_infinite_row_to_itself(gpu_runtime, tile):
    rows, columns, flight = TILES[tile]
    for k in (72, 64 * (flight + 2) + 8):
        m, n = rows + 5, columns + 8
        a = oracle.to_bf16(oracle.uniform(3, (m, k)))
        b = oracle.to_bf16(np.abs(oracle.uniform(4, (k, n))) + np.float32(0.5))
        a[m // 2] = oracle.to_bf16(np.full(k, np.inf, np.float32))
        got = run_variant(gpu_runtime, a, b, tile)
        assert np.all(np.isposinf(got[m // 2]))
        assert np.all(np.isfinite(np.delete(got, m // 2, axis=0)))


@pytest.mark.parametrize("m,n,k", [(1, 8, 32), (255, 264, 64), (257, 248, 96), (300, 520, 160), (513, 1032, 224),
                                   (256, 256, 992)])
def test_five_stage_kernel_at_its_edges(gpu_runtime, m, n, k):
    """Ragged rows and columns; K of an odd number of K tiles of 32, fewer than five, and more."""
    a, b, a64, b64 = operands(m, n, k)
    got = run_variant(gpu_runtime, a, b, p.GEMM_BF16_FIVE_STAGE).astype(np.float64)
    bound = k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert np.all(np.abs(got - a64 @ b64) <= bound)


@pytest.mark.parametrize("tile", SWIGLU_TILES)
def test_swiglu_form_of_every_tile(gpu_runtime, tile):
    five = tile == p.GEMM_BF16_FIVE_STAGE
    rows, columns, flight = (256, 256, 4) if five else TILES[tile]
    shapes = ([(255, 128, 32), (257, 256, 96), (300, 384, 224)] if five else
              [(m, n // 2 // 8 * 8, k) for m, n, k in edge_shapes(rows, columns, flight) if n >= 16])
    for m, f, k in shapes:
        a, b, a64, b64 = operands(m, 2 * f, k)
        got = oracle.from_bf16(run_variant(gpu_runtime, a, b, tile, swiglu=True)).astype(np.float64)
        gate, up = a64 @ b64[:, :f], a64 @ b64[:, f:]
        size = k * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
        silu = gate / (1.0 + np.exp(-gate))
        # the sums' errors through |silu'| <= 1.1, the exponential and reciprocal (2^-20), one rounding to
        # bf16 (8 significant bits: half of the spacing 2^-7 at 1)
        bound = 1.1 * size[:, :f] * np.abs(up) + np.abs(silu) * size[:, f:] + size[:, :f] * size[:, f:]
        bound += (2.0 ** -8 + 2.0 ** -20) * (np.abs(silu * up) + bound) + 1e-38
        assert np.all(np.abs(got - silu * up) <= bound), (m, f, k)


def test_variants_that_cannot_run_are_refused(gpu_runtime):
    rt = gpu_runtime
    ptr = rt.alloc(1 << 20)
    for m, n, k, tile, slices, flags in [(64, 64, 60, 1, 1, 0), (64, 60, 64, 1, 1, 0), (64, 64, 64, 1, 2, 0),
                                         (64, 64, 64, 11, 1, 0), (64, 64, 64, 1, 17, 0), (64, 64, 48, 9, 1, 0),
                                         (64, 64, 64, 9, 2, 0), (64, 64, 64, 1, 1, p.GEMM_BF16_SWIGLU),
                                         (64, 64, 64, 9, 1, p.GEMM_BF16_SWIGLU), (64, 64, 64, 10, 1, p.GEMM_BF16_SWIGLU),
                                         (64, 64, 128, 2, 2, p.GEMM_BF16_SWIGLU)]:
        rc, status = rt.gemm_bf16_device_variant(ptr, ptr + (1 << 18), ptr + (1 << 19), m, n, k, tile, slices, flags)
        assert rc == p.PROM_ERROR and (status.stage, status.detail) == (p.STAGE_INIT, p.DETAIL_INVALID_ARGUMENT)
    rt.free(ptr)
