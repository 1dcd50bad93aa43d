"""Calls of few rows that go back and forth between two kernels: those that one of them was timed ahead on by more than 3 % go to it."""
from __future__ import annotations

import ctypes

import pytest

from vllm_amd import _lib


@pytest.mark.parametrize("m,k,n", [(2, 7040, 2560), (4, 3968, 2880), (4, 6784, 2944), (4, 3968, 2240), (2, 7552, 3456), (4, 7680, 3008)])
def test_long_streams_of_single_tiles_stay_with_the_decode_kernel(m, k, n):
    """4-bit codes in groups of 128 rows, 2 .. 4 rows: 5.0 .. 5.6 us on the decode kernel, 4 .. 13 % more on the one with operands in registers."""
    plan = (ctypes.c_double * 7)()
    _lib.check(_lib.load().vaq_w4a16_regs_plan(m, n, k, 1, 0, plan))
    assert plan[0] == 1 and plan[6] == 0, list(plan)


@pytest.mark.parametrize("m,k,n", [(4, 2048, 2048), (3, 2688, 4096), (4, 5120, 5120), (4, 9216, 4416), (2, 3584, 18944), (4, 3456, 2368), (3, 7680, 704), (4, 5504, 2560)])
def test_and_others_do_not(m, k, n):
    plan = (ctypes.c_double * 7)()
    _lib.check(_lib.load().vaq_w4a16_regs_plan(m, n, k, 1, 0, plan))
    assert plan[6] == 1, list(plan)


@pytest.mark.parametrize("m,k,n,here", [(22, 2976, 10240, 0), (30, 2064, 7104, 0), (17, 2016, 9088, 0), (20, 2608, 7808, 0), (26, 2688, 12544, 1), (32, 4096, 4096, 1), (24, 8192, 8192, 1), (32, 2048, 2048, 1),
                                        (30, 3328, 6144, 1)])
def test_fp8_weights_of_17_to_32_rows(m, k, n, here):
    """The kernel for some dozen rows against the stream kernel: 8.4, 5.8, 6.2 and 7.0 us there, 4 .. 14 % more here."""
    plan = (ctypes.c_double * 5)()
    _lib.check(_lib.load().vaq_fp8_regs_plan(m, n, k, plan))
    assert plan[4] == here, list(plan)
