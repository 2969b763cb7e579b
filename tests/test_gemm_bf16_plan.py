"""The bf16 GEMM's choice of kernel, on the CPU through the plan query (a pure function of
the shape).  Every kernel and its sliced form is reached by a shape of ordinary use, and the
shapes that GPU tests name a kernel for run on it."""
import pytest

from oct_amd import prometheus as p

FIVE_STAGE = p.GEMM_BF16_FIVE_STAGE


@pytest.mark.parametrize("shape,tile,sliced,padded", [
    ((32, 256, 256), 0, False, False), ((32, 256, 1152), 0, True, False), ((35, 262, 1227), 0, True, True),
    ((32, 256, 384), 1, False, False), ((47, 256, 2176), 1, True, False), ((37, 335, 287), 1, False, True),
    ((103, 8320, 384), 2, False, False), ((36, 1536, 8064), 2, True, False),
    ((166, 11008, 896), 3, False, False), ((70, 2816, 10112), 3, True, False),
    ((582, 3456, 512), 4, False, False), ((450, 768, 8576), 4, True, False),
    ((337, 11392, 256), 5, False, False), ((142, 3712, 5504), 5, True, False),
    ((585, 9216, 256), 6, False, False), ((202, 9344, 2688), 6, True, False),
    ((1480, 5504, 256), 7, False, False), ((907, 4352, 6400), 7, True, False),
    ((1030, 11264, 256), 8, False, False), ((476, 8320, 4096), 8, True, False),
    ((1541, 8320, 256), FIVE_STAGE, False, False), ((4096, 4096, 4096), FIVE_STAGE, False, False),
    ((5, 7, 9), p.GEMM_BF16_STAGED, False, False),
    # the FFN down projection of a 1056-token block
    ((1056, 3840, 10240), 3, False, False),
    # the ragged shapes of test_gpu_gemm.py
    ((4224, 2056, 72), 7, False, False), ((600, 8200, 136), 6, False, False), ((1024, 4096, 8), 2, False, False),
    ((1100, 16400, 96), 7, False, False), ((2560, 3584, 8224), 5, False, False)])
def test_kernel_of_a_shape(shape, tile, sliced, padded):
    plan = p.gemm_bf16_plan(*shape)
    assert plan is not None and (plan[0], plan[1] > 1, plan[2]) == (tile, sliced, padded), plan


@pytest.mark.parametrize("shape,tile", [((1, 64, 128), 2), ((1, 12216, 1024), 3), ((67, 8888, 512), 4),
                                        ((67, 17424, 128), 6), ((269, 13912, 128), 7), ((198, 16784, 128), 8),
                                        ((488, 14848, 256), FIVE_STAGE), ((1696, 10240, 3840), FIVE_STAGE)])
def test_swiglu_kernel_of_a_shape(shape, tile):
    assert p.gemm_bf16_plan(*shape, p.GEMM_BF16_SWIGLU) == (tile, 1, False)


def test_shapes_without_a_plan():
    assert p.gemm_bf16_plan(64, 60, 64, p.GEMM_BF16_SWIGLU) is None  # columns not a multiple of 8
    assert p.gemm_bf16_plan(0, 64, 64) is None and p.gemm_bf16_plan(70000, 70000, 1) is None


@pytest.mark.parametrize("tokens,qkv,out,up,down", [(1696, 6, 6, FIVE_STAGE, 6),
                                                    (2208, FIVE_STAGE, 5, FIVE_STAGE, 5),
                                                    (4224, FIVE_STAGE, FIVE_STAGE, FIVE_STAGE, FIVE_STAGE)])
def test_operand_layouts_of_the_dit_block(tokens, qkv, out, up, down):
    """The products of the 3840-wide block: those on the five-stage kernel read K-blocked operands."""
    width, ffn, blocked = 3840, 10240, p.GEMM_BF16_BLOCKED_A
    assert p.gemm_bf16_plan(tokens, 3 * width, width, blocked)[0] == qkv
    assert p.gemm_bf16_plan(tokens, width, width, blocked)[0] == out
    assert p.gemm_bf16_plan(tokens, ffn, width, p.GEMM_BF16_SWIGLU)[0] == up
    assert p.gemm_bf16_plan(tokens, width, ffn, blocked)[0] == down
