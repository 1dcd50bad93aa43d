"""The W4A16 kernel of 256 x 256 tiles (w4a16_tile256_kernel.h) in every weight format, forced, against the CPU oracle."""
from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import w4a16 as o
from tests.helpers import W4A16Layer, check_gemm_close

pytestmark = pytest.mark.gpu

TILE = 48

# (K, N, M): one quantisation group; even and odd numbers of them, whole turns of the weight ring and a remainder; strips that end inside a tile, in the first and in
# the last tile column; rows that end inside a block of 16, inside a tile and with one
SHAPES = [(128, 64, 257), (256, 192, 256), (384, 320, 255), (640, 576, 300), (1408, 256, 513)]


def _forced(layer, a, split, bias=None):
    from vllm_amd import _tuning
    with _tuning.override(prefill_tile=TILE + 1, prefill_split=split):
        return layer(a) if bias is None else layer(a, bias)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group_size,asym", [(4, 128, False), (4, 128, True), (4, -1, False), (4, -1, True), (4, 64, False), (4, 64, True), (4, 32, False), (4, 32, True),
                                                  (8, 128, False), (8, -1, False), (8, 64, False), (8, 32, False)])
def test_tile256(device, bits, group_size, asym, dtype):
    """Gaussian activations against the oracle, whole and in parts of K; one-hot activations return rn16((q - z) * s) bit for bit: every word is
    dequantised with its own sub-group's scale, every k-octet meets its activation chunk, nothing is added twice."""
    for k, n, m in SHAPES:
        case = o.make_w4a16_case(k, n, group_size, asym=asym, dtype=dtype, seed=k + n, num_bits=bits)
        layer = W4A16Layer(case, device, dtype)
        w = o.case_w_ref(case)
        a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dtype)
        rows = [(37 * i + 32 * (i % 4) + m) % k for i in range(m)]
        hot = torch.zeros(m, k, dtype=dtype)
        hot[torch.arange(m), torch.tensor(rows)] = 1
        ref = o.gemm_ref(a, w)
        a, hot = a.to(device), hot.to(device)
        for split in (1, 2, 3):
            what = f"g={group_size} bits={bits} k={k} n={n} m={m} split {split}"
            assert torch.equal(_forced(layer, hot, split).cpu(), w[rows]), what
            out = _forced(layer, a, split)
            check_gemm_close(out, ref, what)
            assert torch.equal(out, _forced(layer, a, split)), f"{what}: not deterministic"
        assert bool((layer.workspace == 0).all()), "workspace counters not restored to zero"


@pytest.mark.parametrize("bits,group_size", [(4, 32), (8, 128)])
def test_tile256_bias_strided_rows_and_unaligned_output(device, bits, group_size):
    """Bias, padded activation rows with NaN between them and an output that is 8-byte aligned only, through the C ABI."""
    from vllm_amd import _lib
    lib = _lib.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)
    for k, n, m in ((640, 320, 270), (384, 64, 33)):
        case = o.make_w4a16_case(k, n, group_size, asym=False, seed=n, num_bits=bits)
        layer = W4A16Layer(case, device)
        a = torch.full((m, k + 24), float("nan"), dtype=torch.bfloat16, device=device)[:, :k]
        a.copy_(torch.randn(m, k, generator=torch.Generator().manual_seed(k)).to(torch.bfloat16))
        bias = torch.randn(n, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16).to(device)
        ref = o.gemm_ref(a.cpu(), o.case_w_ref(case)) + bias.cpu().double()
        tmp, counters = torch.empty(3 << 20, device=device), torch.zeros(4096, dtype=torch.int32, device=device)
        for split in (1, 2):
            tuning = _lib.VaqTuning()
            tuning.prefill_tile, tuning.prefill_split = TILE + 1, split
            buf = torch.zeros(m * n + 8, dtype=torch.bfloat16, device=device)
            _lib.check(lib.vaq_w4a16_gemm_tuned(
                a.data_ptr(), a.stride(0), layer.w.data_ptr(), layer.scales.data_ptr(), None, None, bias.data_ptr(), buf.data_ptr() + 8, tmp.data_ptr(),
                tmp.numel() * 4, None, counters.data_ptr(), counters.numel(), m, n, k, group_size, _lib.VAQ_BF16,
                _lib.VAQ_WTYPE_U8B128 if bits == 8 else _lib.VAQ_WTYPE_U4B8, 2, stream, ctypes.byref(tuning)))
            torch.cuda.synchronize()
            check_gemm_close(buf[4:4 + m * n].view(m, n), ref, f"split {split} k={k} n={n} m={m}")
            assert bool((buf[:4] == 0).all()) and bool((buf[4 + m * n:] == 0).all()), "stores outside the output"
        assert bool((counters == 0).all())
