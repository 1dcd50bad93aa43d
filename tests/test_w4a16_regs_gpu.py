"""The W4A16 kernel with activations in registers (w4a16_regs_kernel.h), every launch shape of it forced, against the CPU oracle."""
from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import w4a16 as o
from tests.helpers import W4A16Layer, check_gemm_close

pytestmark = pytest.mark.gpu


def _shapes(bits, group_size=128):
    """(n-tiles, m-blocks, wavefronts) of a workgroup."""
    return [(j, mb, nw) for mb in (1, 2, 3) for nw, js in ((8, range(1, 5)), (4, range(3, 9 if bits == 4 else 7))) for j in js
            if (bits, group_size, j, mb, nw) != (8, 32, 4, 3, 8)]


def _forced(shape, split):
    from vllm_amd import _tuning
    j, mb, nw = shape
    return _tuning.override(exp=[0] * 8 + [j | mb << 4 | nw << 8 | split << 12])


def _acts(m, k, dtype=torch.bfloat16, seed=0):
    return torch.randn(m, k, generator=torch.Generator().manual_seed(seed)).to(dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group_size,asym", [(4, 128, False), (4, 128, True), (4, -1, False), (4, 64, True), (4, 64, False), (4, 32, True),
                                                  (4, 32, False), (8, 128, False), (8, -1, False), (8, 64, False), (8, 32, False)])
def test_every_launch_shape(device, bits, group_size, asym, dtype):
    """Gaussian activations against the oracle, whole and in parts of K; one-hot activations return rn16((q - z) * s) bit for bit.  (K, N, M): fewer k-tiles than
    wavefronts, one to three turns of the weight ring with each remainder, a last range of n-tiles that is mostly empty, rows below, at and past a block."""
    for k, n, m in ((128, 64, 1), (1536, 192, 4), (640, 320, 17), (1152, 192, 32), (2688, 448, 49), (3072, 128, 100)):
        case = o.make_w4a16_case(k, n, group_size, asym=asym, dtype=dtype, seed=k + n, num_bits=bits)
        layer = W4A16Layer(case, device, dtype)
        w = o.case_w_ref(case)
        a = _acts(m, k, dtype, seed=m)
        ref = o.gemm_ref(a, w)
        rows = [(37 * i + 32 * (i % 4) + m) % k for i in range(m)]
        hot = torch.zeros(m, k, dtype=dtype)
        hot[torch.arange(m), torch.tensor(rows)] = 1
        a, hot = a.to(device), hot.to(device)
        for shape in _shapes(bits, group_size):
            for split in (1, 2, 3):
                if split > 1 and k // 128 // split < shape[2]:
                    continue
                what = f"shape {shape} split {split} g={group_size} bits={bits} k={k} n={n} m={m}"
                with _forced(shape, split):
                    assert torch.equal(layer(hot).cpu(), w[rows]), what
                    out = layer(a)
                    check_gemm_close(out, ref, what)
                    assert torch.equal(out, layer(a)), f"{what}: not deterministic"
        assert bool((layer.workspace == 0).all()), "workspace counters not restored to zero"


def test_special_values_stay_in_their_rows(device):
    """Infinite and NaN activations make their own rows' results non-finite and leave the others alone: what a wavefront requests past its
    last k-tile, and the rows that stand in for those past M, meet no result."""
    for k, n, m in ((640, 320, 21), (2688, 192, 40), (1152, 64, 4)):
        layer = W4A16Layer(o.make_w4a16_case(k, n, 128, asym=True, seed=k), device)
        a = _acts(m, k, seed=m).to(device)
        special = [0, 2] if m < 6 else [0, 3, 5, m - 1]
        for row, value in zip(special, (float("inf"), float("nan"), float("-inf"), float("inf"))):
            a[row, (row * 131) % k] = value
        plain = [i for i in range(m) if i not in special]
        for shape in _shapes(4):
            for split in (1, 2):
                if k // 128 // split < shape[2] and split > 1:
                    continue
                with _forced(shape, split):
                    got, clean = layer(a), layer(torch.nan_to_num(a, 0, 0, 0))
                assert torch.equal(got[plain], clean[plain]) and not bool(torch.isfinite(got[special]).any()), f"{shape} {split}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("bits,group_size,asym", [(4, 128, False), (4, -1, True), (4, 64, True), (4, 32, False), (8, 128, False), (8, 32, False)])
def test_infinite_and_huge_activations_are_those_of_the_weights(device, bits, group_size, asym, dtype):
    """inf * w has the sign of w, and is NaN where w = 0; bf16 activations close to the largest number give finite results where the products with
    the weights are finite (codes with their bias of 128 and more would overflow in fp32).  The other rows keep their bits."""
    for k, n, m in ((640, 320, 21), (2688, 192, 40), (1152, 64, 4), (1536, 192, 100)):
        case = o.make_w4a16_case(k, n, group_size, asym=asym, dtype=dtype, seed=k, num_bits=bits)
        layer, w = W4A16Layer(case, device, dtype), o.case_w_ref(case).double()
        a = _acts(m, k, dtype, seed=m)
        clean = a.clone()
        special, at = ([0, 2] if m < 6 else [0, 3, 5, m - 1]), [(131 * i + 7) % k for i in range(m)]
        for row, value in zip(special, (float("inf"), 2.0 ** 126 if dtype == torch.bfloat16 else 4096.0, float("-inf"), float("inf"))):
            a[row, at[row]] = value
        a, clean = a.to(device), clean.to(device)
        plain = [i for i in range(m) if i not in special]
        for shape in _shapes(bits, group_size)[::3]:
            for split in (1, 2):
                if split > 1 and k // 128 // split < shape[2]:
                    continue
                what = f"{shape} {split} g={group_size} bits={bits} m={m}"
                with _forced(shape, split):
                    got, want = layer(a).cpu(), layer(clean).cpu()
                assert torch.equal(got[plain], want[plain]), what
                for row in special:
                    ref = a[row].cpu().double() @ w
                    if bool(torch.isfinite(a[row]).all()):      # one rounding to 16 bits of the result, fp32 sums of up to k terms beside it
                        assert bool(((got[row].double() - ref).abs() <= ref.abs() * 2.0 ** -8 + ref.abs().max() * k * 2.0 ** -24).all()), what
                    else:
                        assert torch.equal(torch.nan_to_num(got[row].double(), 0.25, 1, -1), torch.nan_to_num(ref, 0.25, 1, -1)), what


def test_bias_strided_rows_and_unaligned_output(device):
    """Bias, padded activation rows (NaN between them) and an output that is 8-byte aligned only, through the C ABI; scratch that is too small for the parts
    of K sends the call to another kernel instead of failing."""
    from vllm_amd import _lib
    lib = _lib.load()
    stream = ctypes.c_void_p(torch.cuda.current_stream(device).cuda_stream)
    for k, n, m in ((640, 320, 19), (2048, 64, 33), (2176, 128, 5)):
        case = o.make_w4a16_case(k, n, 128, asym=False, seed=n)
        layer = W4A16Layer(case, device)
        a = torch.full((m, k + 24), float("nan"), dtype=torch.bfloat16, device=device)[:, :k]
        a.copy_(_acts(m, k, seed=k))
        bias = _acts(1, n, seed=5)[0].to(device)
        ref = o.gemm_ref(a.cpu(), o.case_w_ref(case)) + bias.cpu().double()
        tmp = torch.empty(1024 * 1024, device=device)
        counters = torch.zeros(4096, dtype=torch.int32, device=device)
        for shape in _shapes(4):
            for split in (1, 2):
                if split > 1 and k // 128 // split < shape[2]:
                    continue
                tuning = _lib.VaqTuning()
                tuning.exp[8] = shape[0] | shape[1] << 4 | shape[2] << 8 | split << 12
                sizes = [ctypes.c_size_t() for _ in range(3)]
                _lib.check(lib.vaq_w4a16_gemm_workspace_tuned(m, n, k, 0, 0, *map(ctypes.byref, sizes), ctypes.byref(tuning)))
                assert sizes[0].value <= tmp.numel() * 4 and sizes[2].value <= counters.numel()
                for given in (tmp.numel() * 4, 512):
                    buf = torch.zeros(m * n + 8, dtype=torch.bfloat16, device=device)
                    _lib.check(lib.vaq_w4a16_gemm_tuned(
                        a.data_ptr(), a.stride(0), layer.w.data_ptr(), layer.scales.data_ptr(), None, None, bias.data_ptr(), buf.data_ptr() + 8,
                        tmp.data_ptr(), given, None, counters.data_ptr(), counters.numel(), m, n, k, 128, _lib.VAQ_BF16,
                        _lib.VAQ_WTYPE_U4B8, 0, stream, ctypes.byref(tuning)))
                    torch.cuda.synchronize()
                    check_gemm_close(buf[4:4 + m * n].view(m, n), ref, f"shape {shape} split {split} k={k} n={n} m={m}")
                    assert bool((buf[:4] == 0).all()) and bool((buf[4 + m * n:] == 0).all()), "stores outside the output"
        assert bool((counters == 0).all())
