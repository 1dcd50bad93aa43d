"""Per-token quantisation of few long rows, several workgroups to a row: the bits of the kernel with one, which takes the same rows among more."""
from __future__ import annotations

import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _quant(x, out, out_stride, scales, ub):
    from vllm_amd import _lib
    tag = {torch.float16: _lib.VAQ_F16, torch.bfloat16: _lib.VAQ_BF16, torch.float32: _lib.VAQ_F32}[x.dtype]
    ptr = lambda t: None if t is None else ctypes.c_void_p(t.data_ptr())
    _lib.check(_lib.load().vaq_fp8_quant_per_token(ptr(x), tag, x.stride(0), ptr(out), out_stride, ptr(scales), ptr(ub), x.shape[0], x.shape[1],
                                                   ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,hidden", [(9, 8192), (16, 14336), (64, 16384), (33, 8200), (64, 11000), (8, 8192), (65, 8192), (12, 8184), (12, 16392)])
@pytest.mark.parametrize("bound", [False, True])
def test_rows_as_among_more_rows(device, dtype, rows, hidden, bound):
    g = torch.Generator().manual_seed(rows + hidden)
    x = torch.randn(320, hidden, generator=g).to(dtype).to(device)
    x[3, hidden - 1], x[5, 7], x[7] = float("inf"), float("nan"), 0.0
    ub = torch.tensor([0.9], device=device) if bound else None
    want, many = torch.zeros(320, hidden, dtype=torch.uint8, device=device), torch.zeros(320, device=device)
    _quant(x, want, hidden, many, ub)      # 320 rows: one workgroup each
    got, few = torch.full((rows, hidden + 16), 0xaa, dtype=torch.uint8, device=device), torch.zeros(rows, device=device)
    _quant(x[:rows], got, hidden + 16, few, ub)
    assert torch.equal(got[:, :hidden], want[:rows]) and torch.equal(few, many[:rows]) and bool((got[:, hidden:] == 0xaa).all())


def test_codes_over_the_rows_they_are_made_from(device):
    x = torch.randn(16, 14336, generator=torch.Generator().manual_seed(1)).to(torch.bfloat16).to(device)
    want, s0, s1 = torch.zeros(16, 14336, dtype=torch.uint8, device=device), torch.zeros(16, device=device), torch.zeros(16, device=device)
    _quant(x, want, 14336, s0, None)
    _quant(x, x.view(torch.uint8), 2 * 14336, s1, None)
    assert torch.equal(x.view(torch.uint8)[:, :14336], want) and torch.equal(s0, s1)
