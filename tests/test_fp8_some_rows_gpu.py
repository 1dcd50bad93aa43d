"""The FP8 kernel for some dozen rows, against exact sums: every launch shape, remainders of rows, columns and K, and the calls that go to it."""
from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(m, n, k, seed, device, gap=0):
    """Small integers as e4m3 (every product and sum exact), rows `gap` bytes further apart than K with NaN codes between them."""
    g = torch.Generator().manual_seed(seed)
    a, w = torch.randint(-2, 3, (m, k), generator=g).float(), torch.randint(-1, 2, (n, k), generator=g).float()
    views = []
    for x in (a, w):
        wide = torch.full((x.shape[0], k + gap), 0x7f, dtype=torch.uint8, device=device).view(torch.float8_e4m3fn)
        wide[:, :k] = x.to(torch.float8_e4m3fn).to(device)
        views.append(wide[:, :k])
    return views[0], views[1].t(), a @ w.t()


def _run(a, b, device, dtype=torch.float16, sa=None, sb=None, bias=None):
    import vllm_amd._custom_ops as ops
    m, n = a.shape[0], b.shape[1]
    return ops.cutlass_scaled_mm(a, b, torch.ones(m, 1, device=device) if sa is None else sa, torch.ones(n, 1, device=device) if sb is None else sb, dtype, bias)


@pytest.mark.parametrize("mb", [1, 2, 3, 4])
@pytest.mark.parametrize("j", [1, 2, 3, 4])
def test_every_launch_shape_exact(device, mb, j):
    """From a K of one chunk (most wavefronts without a step) to several turns of the ring with any part of a step at the end; one row, ragged last blocks of rows and of
    n-tiles, several blocks of rows.  (Shapes that do not fit LDS are not built: such a switch changes nothing.)"""
    from vllm_amd import _tuning
    for k in (16, 128, 240, 256, 384, 896, 1024, 1040, 1152, 2048, 2176, 3056, 5248):
        m, n = 1 + (k * 7 + mb * 37) % 200, 16 * (1 + (k // 128 * 5 + j * 11) % 37)
        a, b, want = _case(m, n, k, k + mb, device, gap=64 if k % 256 else 0)
        with _tuning.override(exp=[0] * 11 + [j | mb << 4]):
            assert torch.equal(_run(a, b, device).cpu().float(), want), (m, n, k)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("per_row,per_col,bias", [(True, True, True), (False, False, False), (True, False, True), (False, True, False)])
def test_scales_and_bias_as_the_tile_kernel(device, dtype, per_row, per_col, bias):
    """Exact sums: the scales, the bias and the roundings between them decide every bit, and are those of the tile kernel."""
    from vllm_amd import _tuning
    g = torch.Generator().manual_seed(5)
    m, n, k = 61, 208, 640
    a, b, _ = _case(m, n, k, 3, device)
    sa, sb = torch.rand(m if per_row else 1, 1, generator=g).to(device), torch.rand(n if per_col else 1, 1, generator=g).to(device)
    bb = torch.randn(n, generator=g).to(dtype).to(device) if bias else None
    with _tuning.override(fp8_path=2):
        want = _run(a, b, device, dtype, sa, sb, bb)
    with _tuning.override(exp=[0] * 11 + [3 | 2 << 4]):
        assert torch.equal(_run(a, b, device, dtype, sa, sb, bb), want)


@pytest.mark.parametrize("mb,j", [(1, 4), (2, 2), (2, 3), (2, 4), (3, 2), (3, 3), (4, 1), (4, 2), (4, 3)])
@pytest.mark.parametrize("bias", [False, True])
def test_one_scale_and_one_step_exact(device, mb, j, bias):
    """One scale for every row and one for every column, so that all results of a wavefront may share their loads, at K where all wavefronts or the last one with work take
    a single step: nothing but the wait for the activations stands between the requests and the reads."""
    from vllm_amd import _tuning
    for k in (16, 784, 1024, 1280, 1792, 2560, 3328):
        m, n = 16 * mb - 3, 16 * (3 * j + 1)
        a, b, want = _case(m, n, k, k + j, device)
        bb = torch.full((n,), 2.0, dtype=torch.float16, device=device) if bias else None
        half = torch.full((1, 1), 0.5, device=device)
        with _tuning.override(exp=[0] * 11 + [j | mb << 4]):
            assert torch.equal(_run(a, b, device, sa=half, sb=half, bias=bb).cpu().float(), want / 4 + (2 if bias else 0)), (m, n, k)


@pytest.mark.parametrize("m,n,k", [(16, 4096, 14336), (17, 1024, 1024), (32, 4096, 4096), (33, 2048, 2048), (64, 1280, 2560), (64, 4096, 4096), (100, 1024, 4096), (128, 2048, 2048),
                                   (200, 1024, 1024), (256, 1024, 4096), (33, 4224, 2256), (48, 1024, 1040), (64, 1344, 3904), (100, 1200, 2320)])
def test_as_chosen_exact(device, m, n, k):
    from vllm_amd import _lib
    plan = (ctypes.c_double * 5)()
    _lib.check(_lib.load().vaq_fp8_regs_plan(m, n, k, plan))
    assert plan[4] == 1
    a, b, want = _case(m, n, k, k, device)
    assert torch.equal(_run(a, b, device).cpu().float(), want)


def test_infinite_results_and_nan_codes_stay_in_their_rows_and_columns(device):
    """A NaN code among the activations or the weights makes its row or column NaN and nothing else; behind K it does nothing (the gap's codes are NaN)."""
    from vllm_amd import _tuning
    for k in (512, 720):
        a, b, want = _case(37, 96, k, 7, device, gap=48)
        a.view(torch.uint8)[5, k - 1] = 0x7f
        b.t().view(torch.uint8)[17, 0] = 0xff
        with _tuning.override(exp=[0] * 11 + [2 | 2 << 4]):
            out = _run(a, b, device).cpu().float()
        bad = torch.zeros(37, 96, dtype=torch.bool)
        bad[5], bad[:, 17] = True, True
        assert torch.equal(out.isnan(), bad) and torch.equal(out[~bad], want[~bad])
