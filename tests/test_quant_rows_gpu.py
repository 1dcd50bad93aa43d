"""Rows of the FP8 quantisers and fused norms: every lane's and wavefront's part in the row reductions, and the longest rows that
are held in registers."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle import fp8 as f

pytestmark = pytest.mark.gpu


def _same(got, want):
    return all(np.array_equal(g.cpu().view(torch.uint8).numpy(), w.view(torch.uint8).numpy()) for g, w in zip(got, want))


# (the last three: a wavefront, 256 and 512 threads to a row)
@pytest.mark.parametrize("tokens,hidden", [(256, 2048), (512, 4096), (64, 512), (1024, 1024), (1024, 4096), (640, 5120)])
def test_row_maximum_in_every_place(device, tokens, hidden):
    """The row's largest magnitude sits in another chunk of 8 in every row; dyadic inputs, so that the sum of squares of the norm
    is exact in any order."""
    import vllm_amd._custom_ops as ops
    torch.manual_seed(hidden)
    x = (torch.randint(-4, 5, (tokens, hidden)) / 4).to(torch.bfloat16)
    rows = torch.arange(tokens)
    x[rows, (rows * 8 + rows % 8) % hidden] = torch.where(rows % 2 == 0, 3.0, -3.0).to(torch.bfloat16)
    assert _same(ops.scaled_fp8_quant(x.to(device), use_per_token_if_dynamic=True), f.ref_dynamic_per_token_quant(x))
    w = torch.ones(hidden, dtype=torch.bfloat16)
    got_q, got_s = ops.rms_norm_dynamic_per_token_quant(x.to(device), w.to(device), 0.0, ops.FP8_DTYPE)
    # bound: the row's root mean square is off by two roundings at most (division, rsqrt: 2^-23 relative each), which can move a
    # norm to its neighbour of 2^-8 relative
    y = x.float() / x.float().pow(2).mean(1, keepdim=True).sqrt()
    top = y.abs().amax(1, keepdim=True)
    assert torch.allclose(got_s.cpu() * 448, top, rtol=2 ** -8 * 1.01, atol=0)
    assert torch.allclose(got_q.cpu().float() * got_s.cpu(), y, rtol=0, atol=float(top.max()) * (2 ** -4 + 2 ** -7))


@pytest.mark.parametrize("hidden", [16384, 16392, 20480, 24584, 32768, 32776])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_long_rows_bit_exact(device, hidden, dtype):
    import vllm_amd._custom_ops as ops
    x = torch.randn(5, hidden, generator=torch.Generator().manual_seed(hidden)).to(dtype)
    x[1, -1] = 17.0
    assert _same(ops.scaled_fp8_quant(x.to(device), use_per_token_if_dynamic=True), f.ref_dynamic_per_token_quant(x))
    assert _same(ops.scaled_fp8_quant(x.to(device)), f.ref_dynamic_per_tensor_quant(x))
    scale = torch.tensor([0.01])
    assert _same(ops.scaled_fp8_quant(x.to(device), scale.to(device))[:1], [f.ref_static_quant(x, scale)])
