"""The rule that chooses the general entry point's kernel (csrc/fa2_general_rule.h), on the CPU."""
import itertools

import pytest

from general_rule import DIMS, DIMS_SMALL, SPLIT, STAGED, kernel


def test_the_kernels_and_their_sizes():
    assert kernel(4, 12, 2, 1000, 1000, 64) == DIMS
    assert kernel(1, 12, 2, 1000, 1000, 64) == DIMS_SMALL
    assert kernel(4, 12, 2, 1000, 1000, 256) == DIMS
    assert kernel(32, 12, 2, 64, 64, 64) == kernel(16, 12, 2, 1000, 1000, 16) == STAGED
    assert kernel(1, 12, 2, 200, 200, 64) == kernel(1, 12, 2, 1000, 1000, 256) == SPLIT
    # few queries over many keys: up to a 16-row tile per CU, each has one to itself on the split kernel
    for d in (32, 64):
        assert kernel(1, 12, 2, 300, 8000, d) == kernel(4, 12, 2, 64, 8000, d) == SPLIT
        assert kernel(64, 12, 2, 1, 500, d) == kernel(64, 12, 2, 15, 500, d) == SPLIT
        assert kernel(1, 12, 2, 400, 2000, d) == DIMS_SMALL
    assert kernel(4, 12, 2, 1000, 1000, 64, 128) == STAGED
    for d, dv, T in itertools.product((16, 32, 64, 128, 256), (16, 32, 64, 128, 256), (1, 64, 4096)):
        assert kernel(16, 12, 2, T, T, d, dv, bits16=False) == SPLIT


@pytest.mark.parametrize("d", [32, 64, 256])
@pytest.mark.parametrize("B,T", [(1, 1000), (4, 1000), (16, 300)])
def test_scales_and_strides_the_prefill_kernel_cannot_take(d, B, T):
    usual = kernel(B, 12, 2, T, T, d)
    for scale in (0.0, -0.125, float("nan"), float("inf")):
        assert kernel(B, 12, 2, T, T, d, scale=scale) in (SPLIT, STAGED)
    for st in ((0, d), (d, d - 8), (1 << 23, d), (d, 1 << 23)):
        assert kernel(B, 12, 2, T, T, d, strides=st) in (SPLIT, STAGED)
    assert kernel(B, 12, 2, T, T, d, strides=((1 << 23) - 8, 4 * d)) == usual
    assert kernel(B, 12, 2, T, 0, d) in (SPLIT, STAGED)


@pytest.mark.parametrize("d,threads,rows", [(32, 512, 128), (64, 512, 128), (256, 256, 128)])
def test_launches_of_one_dimension_stay_below_2_32_threads(d, threads, rows):
    """HIP refuses a dimension of 2^32 threads; the staged kernel's three-dimensional grid takes as many
    work-groups as a call may have (65,535 x 65,535 heads)."""
    most = 2 ** 32 // threads            # work-groups
    heads = -(-most // 65535)            # of 65,535 rows: just too many
    for kv_heads in (1, heads):
        assert kernel(65535, heads, kv_heads, rows, rows, d) == STAGED
        assert kernel(32768, heads, kv_heads, 2 * rows + 1, rows, d) == STAGED
        assert kernel(65535, heads - 2, 1 if kv_heads == 1 else heads - 2, rows, rows, d) == DIMS
    assert kernel(65535, heads - 2, 1, rows, rows, d, xcd_log2=0) == DIMS
