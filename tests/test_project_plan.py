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
