"""The W4A16 tile kernels with weights dequantised in registers (w4a16_strip_kernel.h, and w4a16_tile256_kernel.h: 48), every shape forced, against the CPU oracle."""
from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import w4a16 as o
from tests.helpers import W4A16Layer, check_gemm_close

pytestmark = pytest.mark.gpu

EVERY_FORMAT = (41, 42, 43, 44, 46, 48, 51, 52)
PLAIN_ONLY = (66,)      # 4-bit codes in groups of 128 rows / channelwise

# (K, N, M): one quantisation group; fewer groups than a workgroup takes side by side, and a remainder of them; one to several turns
# of the weight ring and each remainder of it; a last strip and a last tile row that are mostly empty
SHAPES = [(128, 64, 65), (384, 192, 97), (640, 320, 257), (1408, 448, 130), (2688, 128, 96)]


def _acts(m, k, dtype=torch.bfloat16, seed=0):
    return torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).to(dtype)


def _forced(layer, a, tile, split, bias=None):
    from vllm_amd import _tuning
    with _tuning.override(prefill_tile=tile + 1, prefill_split=split, exp=[0, 0, 1]):
        return layer(a) if bias is None else layer(a, bias)


def _one_hot(m, k, dtype):
    rows = [(37 * i + 32 * (i % 4) + m) % k for i in range(m)]
    a = torch.zeros(m, k, dtype=dtype)
    a[torch.arange(m), torch.tensor(rows)] = 1
    return a, rows


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group_size,asym", [(4, 128, False), (4, 128, True), (4, -1, False), (4, 64, True), (4, 32, True), (4, 32, False),
                                                  (8, 128, False), (8, -1, False), (8, 64, False), (8, 32, False)])
def test_strip_tiles(device, bits, group_size, asym, dtype):
    """Gaussian activations against the oracle, whole and in parts of K; one-hot activations return rn16((q - z) * s) bit for
    bit: every k-octet lands in the slot its activation chunk is read for, every column in its lane, nothing is added twice."""
    for k, n, m in SHAPES:
        case = o.make_w4a16_case(k, n, group_size, asym=asym, dtype=dtype, seed=k + n, num_bits=bits)
        layer = W4A16Layer(case, device, dtype)
        w = o.case_w_ref(case)
        a = _acts(m, k, dtype, seed=m)
        ref = o.gemm_ref(a, w)
        hot, rows = _one_hot(m, k, dtype)
        a, hot = a.to(device), hot.to(device)
        for tile in EVERY_FORMAT + (PLAIN_ONLY if bits == 4 and group_size in (128, -1) else ()):
            what = f"tile {tile} g={group_size} bits={bits} k={k} n={n} m={m}"
            for split in (1, 2, 3):
                assert torch.equal(_forced(layer, hot, tile, split).cpu(), w[rows]), f"{what} split {split}"
                out = _forced(layer, a, tile, split)
                check_gemm_close(out, ref, f"{what} split {split}")
                assert torch.equal(out, _forced(layer, a, tile, split)), f"{what} split {split}: not deterministic"
        assert bool((layer.workspace == 0).all()), "workspace counters not restored to zero"


def test_strip_tiles_infinities_stay_in_their_rows(device):
    """Infinite and NaN activations: the rows of the other tile kernel.  Requests past K, past M and for K groups past the end
    bring zeros that no result may meet (0 * inf)."""
    for k, n, m in ((384, 192, 97), (1408, 448, 130)):
        layer = W4A16Layer(o.make_w4a16_case(k, n, 128, asym=True, seed=k), device)
        a = _acts(m, k, seed=m).to(device)
        a[0, 0], a[3, k - 1], a[m - 1, k // 2], a[5, 7] = float("inf"), float("-inf"), float("inf"), float("nan")
        want = _forced(layer, a, 12, 1)
        assert not bool(torch.isfinite(want[[0, 3, 5, m - 1]]).any())
        for tile in EVERY_FORMAT + PLAIN_ONLY:
            for split in (1, 2):
                out = _forced(layer, a, tile, split)
                special = ~torch.isfinite(want)
                assert torch.equal(torch.isfinite(out), ~special), f"tile {tile} split {split}"
                assert torch.equal(torch.nan_to_num(out[special], 1, 2, 3), torch.nan_to_num(want[special], 1, 2, 3)), f"tile {tile} split {split}"


def test_strip_tiles_bias_strided_rows_and_unaligned_output(device):
    """Bias, padded activation rows and an output that is 8-byte aligned only (stored in 8-byte pieces), through the C ABI."""
    from vllm_amd import _lib
    lib = _lib.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)
    for k, n, m in ((640, 320, 70), (1408, 64, 33), (256, 128, 17)):
        case = o.make_w4a16_case(k, n, 128, asym=False, seed=n)
        layer = W4A16Layer(case, device)
        a = torch.randn(m, k + 24, generator=torch.Generator().manual_seed(k)).to(torch.bfloat16).to(device)[:, :k]
        bias = _acts(1, n, seed=5)[0].to(device)
        ref = o.gemm_ref(a.cpu(), o.case_w_ref(case)) + bias.cpu().double()
        tmp = torch.empty(3 * 1024 * 1024, device=device)
        counters = torch.zeros(4096, dtype=torch.int32, device=device)
        for tile in EVERY_FORMAT + PLAIN_ONLY:
            for split in (1, 2):
                tuning = _lib.VaqTuning()
                tuning.prefill_tile, tuning.prefill_split = tile + 1, split
                sizes = [ctypes.c_size_t() for _ in range(3)]
                _lib.check(lib.vaq_w4a16_gemm_workspace_tuned(m, n, k, 0, 0, *map(ctypes.byref, sizes), ctypes.byref(tuning)))
                assert sizes[0].value <= tmp.numel() * 4 and sizes[2].value <= counters.numel()
                buf = torch.zeros(m * n + 8, dtype=torch.bfloat16, device=device)
                _lib.check(lib.vaq_w4a16_gemm_tuned(
                    a.data_ptr(), a.stride(0), layer.w.data_ptr(), layer.scales.data_ptr(), None, None, bias.data_ptr(), buf.data_ptr() + 8,
                    tmp.data_ptr(), tmp.numel() * 4, None, counters.data_ptr(), counters.numel(), m, n, k, 128, _lib.VAQ_BF16,
                    _lib.VAQ_WTYPE_U4B8, 2, stream, ctypes.byref(tuning)))
                torch.cuda.synchronize()
                check_gemm_close(buf[4:4 + m * n].view(m, n), ref, f"tile {tile} split {split} k={k} n={n} m={m}")
                assert bool((buf[:4] == 0).all()) and bool((buf[4 + m * n:] == 0).all()), "stores outside the output"
        assert bool((counters == 0).all())


def test_strip_tiles_rows_almost_4_gib_apart(device):
    """Activations whose last row ends with its storage, just below the 4 GiB that 32-bit offsets reach; everything between the rows is
    NaN, so that no result takes anything from there."""
    k, n, m, pitch = 1408, 320, 127, 1 << 24
    assert (m * pitch * 2) < 1 << 32 < ((m + 1) * pitch * 2) + 1
    base = torch.full((m, pitch), float("nan"), dtype=torch.bfloat16, device=device)
    a = base[:, pitch - k:]
    a.copy_(_acts(m, k, seed=4))
    for bits, group_size in ((4, 128), (8, 64)):
        case = o.make_w4a16_case(k, n, group_size, asym=bits == 4, seed=n, num_bits=bits)
        layer = W4A16Layer(case, device)
        want = [_forced(layer, a.contiguous(), tile, 2) for tile in EVERY_FORMAT]
        check_gemm_close(want[0], o.gemm_ref(a.cpu(), o.case_w_ref(case)), f"bits={bits}")
        for tile, ref in zip(EVERY_FORMAT, want):
            assert torch.equal(_forced(layer, a, tile, 2), ref), f"tile {tile} bits={bits}"


def test_strip_tiles_of_last_round_split(device):
    """256 x 256 tiles with only the tiles of a half-empty last round in parts of K: ragged rows, exact from one-hot rows."""
    from vllm_amd import _lib, _tuning
    cus = _lib.load().vaq_num_cus(torch.device(device).index or 0)
    k, n, m = 2048, 3328, 21 * 256 - 5
    tiles = ((m + 255) // 256) * (n // 256)
    if not (tiles > cus and 0 < tiles % cus <= cus // 2):
        pytest.skip(f"{tiles} tiles on {cus} compute units leave no half-empty last round")
    case = o.make_w4a16_case(k, n, 128, asym=True, seed=9)
    layer = W4A16Layer(case, device)
    w = o.case_w_ref(case)
    hot, rows = _one_hot(m, k, torch.bfloat16)
    a = _acts(m, k, seed=3).to(device)
    exp = [0] * 7
    exp[6] = 2
    with _tuning.override(prefill_tile=49, exp=exp):
        assert torch.equal(layer(hot.to(device)).cpu(), w[rows])
        split = layer(a)
    with _tuning.override(prefill_tile=49, prefill_split=1):
        whole = layer(a)
    check_gemm_close(split[-300:], o.gemm_ref(a[-300:].cpu(), w), "rows of the split tiles")
    same = (split == whole).all(dim=1)
    assert bool(same[:256].all()) and not bool(same.all())
    assert bool((layer.workspace == 0).all()), "workspace counters not restored to zero"
