"""8-bit codes as one operand of a product in the W4A16 kernel with activations in registers (w4a16_regs_kernel.h), against the CPU oracle and 64-bit sums."""
from __future__ import annotations

import pytest
import torch

from oracle import w4a16 as o
from tests.helpers import W4A16Layer

# (n-tiles, m-blocks, wavefronts): each number of m-blocks, the fewest and the most n-tiles
SHAPES = [(1, 1, 8), (4, 2, 8), (3, 1, 4), (6, 2, 4), (6, 3, 4), (1, 3, 8)]


def _forced(shape):
    from vllm_amd import _tuning
    j, mb, nw = shape
    return _tuning.override(exp=[0] * 8 + [j | mb << 4 | nw << 8 | 1 << 12])


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group_size", [128, -1, 64, 32])
def test_every_code_in_every_place(device, group_size, dtype):
    """Columns that run through all 256 codes, each starting elsewhere, times the rows of the identity: the weights bit for bit."""
    k, n = 256, 128
    case = o.make_w4a16_case(k, n, group_size, dtype=dtype, seed=3, num_bits=8)
    case["q"][:] = (torch.arange(k)[:, None] * 37 + torch.arange(n)[None] * 5).numpy() % 256
    case["qweight"] = o.gptq_pack(case["q"], 8)
    layer, w = W4A16Layer(case, device, dtype), o.case_w_ref(case)
    eye = torch.eye(k, dtype=dtype, device=device)
    for shape in SHAPES:
        for rows in (eye[:5], eye):
            with _forced(shape):
                assert torch.equal(layer(rows).cpu(), w[:len(rows)]), f"shape {shape}, {len(rows)} rows"


SUMS = ((256, 64, 20), (2688, 192, 50), (1152, 320, 1))      # (K, N, M)


def _sums(k, n, m, group_size, dtype):
    """A case with activations far from zero in the mean, so that a code's bias weighs most: the case, activations, codes, scales of every row, sums in 64 bits and how far
    from them a result may be.  One rounding of the result (half a unit of its last place: 2^-8 / 2^-11 of a number of 8 / 11 significant bits) and K rounded fp32 sums,
    none beyond the sum of the magnitudes of |a| (bias + code) s, whose errors of at most 2^-24 of it each, either way, add up like steps of a random walk: K^0.5
    of them, and as much again for the sums that take the bias out."""
    unit, bias = (2.0 ** -8, 0.0) if dtype == torch.bfloat16 else (2.0 ** -11, 1024.0)
    case = o.make_w4a16_case(k, n, group_size, dtype=dtype, seed=k, num_bits=8)
    a = (torch.randn(m, k, generator=torch.Generator().manual_seed(m)) + 3).to(dtype)
    q, s = torch.from_numpy(case["q"]).double(), case["scales"].double().repeat_interleave(group_size, 0)
    exact, most = a.double() @ ((q - 128) * s), a.double().abs() @ ((q + bias + 128) * s)
    return case, a, q, s, exact, unit * exact.abs() + 2 * k ** 0.5 * 2.0 ** -24 * most


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group_size", [128, 32])
def test_sums_against_64_bits(device, group_size, dtype):
    for k, n, m in SUMS:
        case, a, _, _, exact, bound = _sums(k, n, m, group_size, dtype)
        layer = W4A16Layer(case, device, dtype)
        for shape in SHAPES:
            with _forced(shape):
                err = (layer(a.to(device)).cpu().double() - exact).abs()
            assert bool((err <= bound).all()), f"shape {shape} k={k} n={n} m={m}: {(err / bound).max()}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("group_size", [128, 32])
def test_the_bound_of_the_sums_tells_mistakes(group_size, dtype):
    """In 64 bits, planted in the oracle: one row of K left out, and one group's sum that takes 1 too few out of its codes, pass the bound in most of the results."""
    for k, n, m in SUMS:
        _, a, q, s, exact, bound = _sums(k, n, m, group_size, dtype)
        assert bool(((exact.to(dtype).double() - exact).abs() <= bound).all())
        for row in (0, k // 2, k - 1):
            w = (q - 128) * s
            w[row] = 0
            beyond = ((a.double() @ w).to(dtype).double() - exact).abs() > bound
            assert beyond.double().mean() > 0.5, f"row {row} of {k} left out: {beyond.double().mean():.2f}"
        for g in (0, k // group_size - 1):
            z = torch.full((k, 1), 128.0, dtype=torch.double)
            z[g * group_size:(g + 1) * group_size] = 127
            beyond = ((a.double() @ ((q - z) * s)).to(dtype).double() - exact).abs() > bound
            assert beyond.double().mean() > 0.5, f"group {g}: {beyond.double().mean():.2f}"
