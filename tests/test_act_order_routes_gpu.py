"""act_order on the kernels that run on columns permuted ahead of them, and on those that gather: same numbers either way."""
from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import w4a16 as o
from tests.helpers import W4A16Layer

pytestmark = pytest.mark.gpu


def _layer(k, n, g, bits, asym, device):
    """Scales of one power of two, activations of small integers: every product and every sum in float32 is exact, so each route has to give the
    same bits."""
    case = o.make_w4a16_case(k, n, g, asym=asym, act_order=True, seed=k + n, **({"num_bits": 8} if bits == 8 else {}))
    case["scales"] = torch.full_like(case["scales"], 2.0 ** -8)
    return W4A16Layer(case, device, torch.float16)


def _x(m, k, device, stride=0):
    wide = torch.full((m, k + stride), float("nan"), dtype=torch.float16, device=device)
    wide[:, :k] = torch.randint(-2, 3, (m, k), generator=torch.Generator().manual_seed(m * k)).to(torch.float16).to(device)
    return wide[:, :k]


def _sorted_call(layer, x):
    empty = torch.empty(0, dtype=torch.int32, device=x.device)
    return layer.ops.gptq_marlin_gemm(x[:, layer.sort_idx.long()].contiguous(), None, layer.w, None, layer.scales, None, layer.zp, empty, empty,
                                      layer.workspace, layer.wtype, x.shape[0], layer.n, layer.k, is_k_full=True, use_fp32_reduce=True)


@pytest.mark.parametrize("k,n,g,bits,asym", [(4096, 4096, 128, 4, False), (2048, 2112, 64, 4, True), (1664, 1152, 32, 4, False), (7040, 1024, 128, 4, True),
                                             (2560, 2560, 64, 8, False), (4992, 320, 128, 8, False), (1024, 9280, 128, 4, False), (256, 64, 128, 4, False)])
def test_permuted_ahead_equals_gathered_equals_sorted(device, k, n, g, bits, asym):
    from vllm_amd import _tuning
    layer = _layer(k, n, g, bits, asym, device)
    for m in (1, 2, 4, 5, 8, 16, 17, 31, 32, 33, 48, 64, 65, 128, 200, 256, 257):
        x = _x(m, k, device, 8 * (m % 2))
        out = layer(x)
        with _tuning.override(exp=[0] * 9 + [1]):
            gathered = layer(x)
        assert torch.equal(out, gathered) and torch.equal(out, _sorted_call(layer, x)), (m, k, n)
    assert bool((layer.workspace == 0).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("k,n,g,bits,asym", [(640, 3008, 64, 4, False), (1024, 1024, 128, 4, True), (1152, 2048, 32, 4, True), (512, 4160, 128, 8, False),
                                             (2048, 1024, 64, 8, False), (4096, 1088, 128, 4, False)])
def test_infinite_and_huge_activations_beyond_32_rows(device, k, n, g, bits, asym, dtype):
    """From 33 rows on (4-bit codes in groups of 128 rows: 65) an infinite activation gives infinities of the weights' signs (NaN where the weight is 0), and a bf16 one of 2^122
    (codes with their bias of 128 and more would overflow, the weights themselves stay below 2^5) finite results, as on the tile kernels: workgroups of 16 rows, which give NaN, take no such call.  The other rows keep their bits."""
    case = o.make_w4a16_case(k, n, g, asym=asym, act_order=True, dtype=dtype, seed=k + n, num_bits=bits)
    layer, w = W4A16Layer(case, device, dtype), o.case_w_ref(case).double()
    for m in (33, 48, 64, 65, 80, 96, 125, 128, 160, 200, 256)[3 if g == 128 and bits == 4 else 0:]:
        a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(dtype)
        clean, special, at = a.clone(), [0, 17, 30, m - 1], [(131 * i + 7) % k for i in range(m)]
        for row, value in zip(special, (float("inf"), 2.0 ** 122 if dtype == torch.bfloat16 else 4096.0, float("-inf"), float("inf"))):
            a[row, at[row]] = value
        got, want = layer(a.to(device)).cpu(), layer(clean.to(device)).cpu()
        plain = [i for i in range(m) if i not in special]
        assert torch.equal(got[plain], want[plain]), m
        for row in special:
            ref = a[row].double() @ w
            if bool(torch.isfinite(a[row]).all()):      # one rounding to 16 bits of a weight and one of the result, fp32 sums of up to k terms beside them
                assert bool(((got[row].double() - ref).abs() <= ref.abs() * 2.0 ** -7 + ref.abs().max() * k * 2.0 ** -24).all()), (m, row)
            else:
                assert torch.equal(torch.nan_to_num(got[row].double(), 0.25, 1, -1), torch.nan_to_num(ref, 0.25, 1, -1)), (m, row)


def _c_call(lib, _lib, layer, x, c_tmp, a_tmp, counters):
    out = torch.empty((x.shape[0], layer.n), dtype=x.dtype, device=x.device)
    ptr = lambda t: None if t is None or t.numel() == 0 else ctypes.c_void_p(t.data_ptr())
    rc = lib.vaq_w4a16_gemm(ptr(x), x.stride(0), ptr(layer.w), ptr(layer.scales), None, ptr(layer.sort_idx), None, ptr(out), ptr(c_tmp),
                            0 if c_tmp is None else c_tmp.numel() * 4, ptr(a_tmp), ptr(counters), 0 if counters is None else counters.numel(), x.shape[0],
                            layer.n, layer.k, layer.g, _lib.VAQ_F16, _lib.VAQ_WTYPE_U4B8, 0, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    return rc, out


@pytest.mark.parametrize("m,k,n", [(8, 4096, 4096), (16, 4096, 4096), (32, 4096, 4096), (8, 14336, 4096), (16, 14336, 4096), (32, 14336, 1024)])
def test_callers_without_room_for_permuted_columns(device, m, k, n):
    """Up to 32 rows the gather inside the kernel is left for a caller whose scratch has no room for the columns and what the call needs behind them, down to what
    that kernel itself needs; below both a call is refused and launches nothing.  What is written behind the scratch would show."""
    from vllm_amd import _lib
    lib = _lib.load()
    layer = _layer(k, n, 128, 4, False, device)
    x = _x(m, k, device)
    want = layer(x)
    sizes = [ctypes.c_size_t() for _ in range(3)]
    _lib.check(lib.vaq_w4a16_gemm_workspace_of_format(m, n, k, layer.g, _lib.VAQ_WTYPE_U4B8, 1, 0, *map(ctypes.byref, sizes)))
    asked, ints = sizes[0].value // 4, max(sizes[2].value, 1)
    assert sizes[0].value >= 2 * m * k and sizes[1].value == 0
    # float32s of scratch: of the kernel that gathers, by its parts of K, and with the columns ahead of them of what runs without act_order
    plan, regs = (ctypes.c_double * 6)(), (ctypes.c_double * 7)()
    _lib.check(lib.vaq_w4a16_decode_plan(m, n, k, 1, 0, 0, plan))
    _lib.check(lib.vaq_w4a16_regs_plan(m, n, k, 1, 0, regs))
    tile = lambda parts, blocks: int(parts) * (n // 16) * blocks * 256 if parts > 1 else 0
    columns, gathered = m * k // 2, tile(plan[3], (m + 15) // 16)
    regs_rows = -(-m // (16 * int(regs[1]))) * int(regs[1])
    permuted = columns + min(gathered, tile(regs[3], regs_rows) if regs[6] else gathered)
    need = min(gathered, permuted)
    assert need < asked
    counters = torch.zeros(ints, dtype=torch.int32, device=device)
    given = {asked, asked + 1, asked - 1, asked // 2, columns, columns + 4, columns - 1, permuted, permuted - 1, gathered, need + 1, need - 1, need // 2}
    for count in sorted(c for c in given if c >= 0):
        buf = torch.full((count + 64,), 7.0, dtype=torch.float32, device=device)
        rc, out = _c_call(lib, _lib, layer, x, buf[:count], None, counters)
        assert rc == (_lib.VAQ_OK if count >= need else _lib.VAQ_ERR_INVALID_ARG), (count, need, asked)
        assert bool((buf[count if rc == _lib.VAQ_OK else 0:] == 7.0).all()) and bool((counters == 0).all())
        assert rc != _lib.VAQ_OK or torch.equal(out, want), count
    rc, out = _c_call(lib, _lib, layer, x, None, None, counters)
    assert rc == (_lib.VAQ_ERR_INVALID_ARG if need else _lib.VAQ_OK) and (need or torch.equal(out, want))


def test_replayed_graph(device):
    layer = _layer(4096, 4096, 128, 4, False, device)
    x = _x(16, 4096, device)
    layer(x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = layer(x)
    for seed in range(4):
        x.copy_(torch.randint(-2, 3, x.shape, generator=torch.Generator().manual_seed(seed)).to(x.dtype))
        want = layer(x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want), seed
