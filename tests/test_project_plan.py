"""The tiles of products of bf16 weights, as vkl_project_plan tells them (the host functions that the launchers follow; no GPU)."""
import ctypes as C

import pytest

from vkllama_amd import stack


def plan(*a, **k):
    p = stack.project_plan(*a, **k)
    return p.tile_rows, p.ksplit


def test_arguments_are_checked():
    p, f = stack.ProjectPlan(), stack.lib().vkl_project_plan
    good = (stack.BF16, 4, 8, 64, stack.F32, 0)
    assert f(*good, C.byref(p)) == 0 and f(*good, None) == 1
    for i, bad in ((0, 5), (1, 0), (2, 0), (2, -8), (3, 0), (3, 65), (4, 7), (5, -1), (5, 4)):
        assert f(*(bad if j == i else v for j, v in enumerate(good)), C.byref(p)) == 1, (i, bad)


def test_short_rows_of_32_bits_take_no_planes():
    p = stack.project_plan(stack.F32, 5, 128, 128)
    assert (p.tile_rows, p.planes) == (0, 1)
    p = stack.project_plan(stack.F32, 5, 2048, 2048)
    assert (p.tile_rows, p.planes) == (64, 3)


# A last row of 256-row tiles with few rows is cheap: tiles of 192 rows took 3 to 7 % longer, by themselves and beside the plans before
# them.  More of them, and rows that fill 256, keep what was measured as faster.
@pytest.mark.parametrize("M,N,K,rows,parts", [(513, 7680, 5120, 256, 1), (555, 7680, 5120, 256, 1), (576, 7680, 5120, 256, 1), (2074, 2048, 7552, 256, 1),
                                              (577, 7680, 5120, 192, 1), (700, 7680, 5120, 192, 1), (1049, 4096, 4096, 192, 1), (1049, 5120, 5120, 192, 1),
                                              (2200, 2048, 7552, 192, 1)])
def test_few_rows_in_the_last_tile(M, N, K, rows, parts):
    assert plan(stack.BF16, M, N, K, stack.F32 if N < 6000 else stack.BF16) == (rows, parts)


# parts that are no power of two: 128, 192 and 256 rows, none below 144 rows of x
@pytest.mark.parametrize("M,N,K,rows,parts", [(300, 2056, 7552, 128, 5), (600, 2048, 5504, 128, 3), (366, 3072, 11264, 192, 5), (528, 2048, 7552, 192, 5),
                                              (1025, 2048, 5504, 256, 3), (1100, 4096, 15104, 256, 3), (143, 4096, 11008, None, None)])
def test_parts_that_are_no_power_of_two(M, N, K, rows, parts):
    got = plan(stack.BF16, M, N, K)
    assert got == (rows, parts) if rows else got[1] in (1, 2, 4, 8, 16)
