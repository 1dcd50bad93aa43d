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


@pytest.mark.parametrize("tokens,d", [(1, 8), (3, 24), (1, 6144), (2, 3080), (2, 6144), (1, 12296), (517, 1000), (292, 14336), (293, 14336), (2341, 14336)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_silu_chunks_equal_single_elements(device, tokens, d, dtype):
    """Chunks of 8 against the element-wise kernel of the same arithmetic (an output that is not 8-byte aligned): one chunk, a last
    workgroup in part, both workgroup sizes beside the lines between them (768, 1536 and 524288 chunks), and a thread's second chunk."""
    import vllm_amd._custom_ops as ops
    x = torch.randn(tokens, 2 * d, device=device, dtype=dtype, generator=torch.Generator(device=device).manual_seed(d))
    scale = torch.full((1,), 4 / 448, device=device)
    buf = torch.zeros(tokens * d + 8, dtype=torch.uint8, device=device)
    odd = buf[1:1 + tokens * d].view(ops.FP8_DTYPE).view(tokens, d)
    out = torch.empty(tokens, d, dtype=ops.FP8_DTYPE, device=device)
    ops.silu_and_mul_quant(odd, x, scale)
    ops.silu_and_mul_quant(out, x, scale)
    assert torch.equal(out.view(torch.uint8), odd.view(torch.uint8))


@pytest.mark.parametrize("shape", [(1, 1), (1, 7), (3, 8), (1, 2047), (5, 411), (2, 3076), (3, 4096), (3, 4099), (333, 3001), (2, 1050633), (1, 33554441)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_per_tensor_runs_equal_rows(device, shape, dtype):
    """Rows without gaps go as one run of vectors: single elements, remainders behind the last vector, one and several rounds of the
    grid.  The same rows behind a gap take a workgroup each: codes and scales are the same bits, the first shapes the oracle's too;
    the largest magnitude is the last element."""
    import vllm_amd._custom_ops as ops
    rows, hidden = shape
    x = torch.randn(rows, hidden, device=device, generator=torch.Generator(device=device).manual_seed(hidden)).to(dtype)
    x[-1, -1] = -21.5
    gap = torch.zeros(rows + 1, hidden + 8, dtype=dtype, device=device)[:rows, 8:]
    gap.copy_(x)
    scale = torch.full((1,), 0.01, device=device)
    for given in (scale, None):
        got, want = (ops.scaled_fp8_quant(v, given) for v in (x, gap))
        assert torch.equal(got[0].view(torch.uint8), want[0].view(torch.uint8)) and torch.equal(got[1], want[1])
        if x.numel() < 1 << 20:
            ref = f.ref_static_quant(x.cpu(), scale.cpu()) if given is not None else f.ref_dynamic_per_tensor_quant(x.cpu())
            assert _same(got[:1], [ref[0] if isinstance(ref, tuple) else ref])


@pytest.mark.parametrize("rows,hidden,gap", [(3, 1061, 0), (300, 2047, 0), (1030, 2049, 0), (1030, 5119, 0), (7, 4097, 1), (5, 16385, 0), (4, 32767, 0),
                                             (4, 4096, 3), (1030, 2048, 5), (1, 1000, 3), (6, 40000, 0)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
def test_rows_by_single_elements_bit_exact(device, rows, hidden, gap, dtype):
    """Lengths, row strides and addresses that rule vectors out, on each size of workgroup that takes such rows."""
    import vllm_amd._custom_ops as ops
    x = torch.randn(rows, hidden + gap, generator=torch.Generator().manual_seed(hidden)).to(dtype)[:, gap:]
    x[-1, -1] = 23.0
    view = torch.zeros(rows, hidden + gap, dtype=dtype, device=device)[:, gap:]
    view.copy_(x)
    assert _same(ops.scaled_fp8_quant(view, use_per_token_if_dynamic=True), f.ref_dynamic_per_token_quant(x.contiguous()))
