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


def _tile256(layer, a, split, bias=None, out=None, tail=False):
    """Through the C ABI on the tile path, which a call of 17 .. 256 rows by the plain entry point may leave for a decode kernel.  `split`: parts of K, of every tile or (`tail`) of
    those of the last round only.  The scratch that the call is refused without says that the plan is the one that was asked for."""
    from vllm_amd import _lib
    lib, (m, k), n = _lib.load(), a.shape, layer.n
    tuning, sizes = _lib.VaqTuning(), [ctypes.c_size_t() for _ in range(3)]
    tuning.prefill_tile = TILE + 1
    if tail:
        tuning.exp[6] = split
    else:
        tuning.prefill_split = split
    _lib.check(lib.vaq_w4a16_gemm_workspace_tuned(m, n, k, 0, 0, *map(ctypes.byref, sizes), ctypes.byref(tuning)))
    tiles = -(-m // 256) * -(-n // 256)
    parts = min(split, k // 128) * tiles if not tail else split * (tiles % lib.vaq_num_cus(a.device.index or 0))
    split_bytes = parts * 256 * 256 * 4 if min(split, k // 128) > 1 else 0
    assert sizes[0].value >= split_bytes
    tmp = torch.empty(max(split_bytes, 16) // 4, device=a.device)
    out = torch.empty(m, n, dtype=a.dtype, device=a.device) if out is None else out
    wtype = {"uint4": _lib.VAQ_WTYPE_U4, "uint4b8": _lib.VAQ_WTYPE_U4B8, "uint8b128": _lib.VAQ_WTYPE_U8B128}[str(layer.wtype)]

    def call(nbytes):
        return lib.vaq_w4a16_gemm_tuned(
            a.data_ptr(), a.stride(0), layer.w.data_ptr(), layer.scales.data_ptr(), layer.zp.data_ptr() if layer.zp.numel() else None, None,
            None if bias is None else bias.data_ptr(), out.data_ptr(), tmp.data_ptr(), nbytes, None, layer.workspace.data_ptr(),
            layer.workspace.numel(), m, n, k, layer.g, _lib.VAQ_BF16 if a.dtype == torch.bfloat16 else _lib.VAQ_F16, wtype, 2,
            torch.cuda.current_stream(a.device).cuda_stream, ctypes.byref(tuning))
    if split_bytes and not tail:
        assert call(split_bytes - 16) == _lib.VAQ_ERR_INVALID_ARG
    _lib.check(call(split_bytes))
    return out


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
            assert torch.equal(_tile256(layer, hot, split).cpu(), w[rows]), what
            out = _tile256(layer, a, split)
            check_gemm_close(out, ref, what)
            assert torch.equal(out, _tile256(layer, a, split)), f"{what}: not deterministic"
        assert bool((layer.workspace == 0).all()), "workspace counters not restored to zero"


@pytest.mark.parametrize("bits,group_size", [(4, 32), (8, 128)])
def test_tile256_bias_strided_rows_and_unaligned_output(device, bits, group_size):
    """Bias, padded activation rows with NaN between them and an output that is 8-byte aligned only, through the C ABI."""
    for k, n, m in ((640, 320, 270), (384, 64, 33)):
        case = o.make_w4a16_case(k, n, group_size, asym=False, seed=n, num_bits=bits)
        layer = W4A16Layer(case, device)
        a = torch.full((m, k + 24), float("nan"), dtype=torch.bfloat16, device=device)[:, :k]
        a.copy_(torch.randn(m, k, generator=torch.Generator().manual_seed(k)).to(torch.bfloat16))
        bias = torch.randn(n, generator=torch.Generator().manual_seed(5)).to(torch.bfloat16).to(device)
        ref = o.gemm_ref(a.cpu(), o.case_w_ref(case)) + bias.cpu().double()
        for split in (1, 2):
            buf = torch.zeros(m * n + 8, dtype=torch.bfloat16, device=device)
            _tile256(layer, a, split, bias, out=buf[4:])
            check_gemm_close(buf[4:4 + m * n].view(m, n), ref, f"split {split} k={k} n={n} m={m}")
            assert bool((buf[:4] == 0).all()) and bool((buf[4 + m * n:] == 0).all()), "stores outside the output"
        assert bool((layer.workspace == 0).all())


@pytest.mark.parametrize("bits,group_size,asym,dtype", [(4, 128, False, torch.bfloat16), (4, 64, False, torch.bfloat16), (4, 64, True, torch.float16),
                                                        (4, 32, True, torch.float16), (8, 128, False, torch.float16), (8, 64, False, torch.bfloat16),
                                                        (8, 32, False, torch.bfloat16)])
def test_tile256_last_round_split(device, bits, group_size, asym, dtype):
    """Only the tiles of a half-empty last round in parts of K, beside whole ones: parts that begin inside K at another scale row, ragged rows, exact from one-hot rows."""
    from vllm_amd import _lib
    cus = _lib.load().vaq_num_cus(torch.device(device).index or 0)
    k, n, m = 2048, 3328, 21 * 256 - 5
    tiles = ((m + 255) // 256) * (n // 256)
    if not (tiles > cus and 0 < tiles % cus <= cus // 3):
        pytest.skip(f"{tiles} tiles on {cus} compute units leave no last round of a third and less")
    case = o.make_w4a16_case(k, n, group_size, asym=asym, dtype=dtype, seed=9, num_bits=bits)
    layer, w = W4A16Layer(case, device, dtype), o.case_w_ref(case)
    rows = [(37 * i + 32 * (i % 4) + m) % k for i in range(m)]
    hot = torch.zeros(m, k, dtype=dtype)
    hot[torch.arange(m), torch.tensor(rows)] = 1
    hot, a = hot.to(device), torch.randn(m, k, generator=torch.Generator().manual_seed(3)).to(dtype).to(device)
    whole = _tile256(layer, a, 1)
    for split in (2, 3):
        assert torch.equal(_tile256(layer, hot, split, tail=True).cpu(), w[rows]), f"{split} parts"
        out = _tile256(layer, a, split, tail=True)
        check_gemm_close(out[-300:], o.gemm_ref(a[-300:].cpu(), w), f"rows of the split tiles, {split} parts")
        same = (out == whole).all(dim=1)
        assert bool(same[:256].all()) and not bool(same.all()), f"{split} parts"
        assert bool((layer.workspace == 0).all()), "workspace counters not restored to zero"
