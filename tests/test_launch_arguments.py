"""Divisions that the kernels make by multiplication with a number from the host (tile_handover.h, w4a16_regs_kernel.h)."""
from __future__ import annotations

import os
import shutil
import subprocess

import numpy as np
import pytest

from vllm_amd.build import CSRC, HIPCC_FLAGS

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "launch_arguments_check.hip")


@pytest.fixture(scope="module")
def launch_check(tmp_path_factory):
    """The functions that the kernels find their work by, compiled for the host (native/launch_arguments_check.hip)."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    exe = str(tmp_path_factory.mktemp("launch") / "launch_arguments_check")
    subprocess.run([hipcc, "--offload-host-only", "-O1", "-std=c++17", "-w", "-I", str(CSRC), CHECK, "-o", exe], check=True)
    return exe


def test_every_workgroup_finds_its_work(launch_check):
    r = subprocess.run([launch_check], capture_output=True, text=True)
    assert r.returncode == 0 and "mismatches=0" in r.stdout, r.stdout


@pytest.mark.parametrize("mistake", [1, 2, 3, 4])
def test_and_the_check_can_fail(launch_check, mistake):
    """A wrong number for bands of tiles, for copies of a range, for blocks of rows, for parts of K."""
    r = subprocess.run([launch_check, str(mistake)], capture_output=True, text=True)
    assert r.returncode == 1 and "mismatches=" in r.stdout


@pytest.mark.parametrize("d", [1, 2, 3, 4, 5, 7, 8, 12, 96, 255, 256, 1000, 9504, 65535, 65536, 1 << 20, (1 << 31) - 1, 1 << 31])
def test_quotients_of_the_tile_order(d):
    """x / d = umulhi(x, 2^32 / d), plus one where the rest says so, for any 32-bit x."""
    rng = np.random.default_rng(d)
    q = rng.integers(0, (1 << 32) // d, 4000, dtype=np.uint64) * d
    x = np.concatenate([rng.integers(0, 1 << 32, 20000, dtype=np.uint64), q, q + (d - 1), q + (d > 1),
                        np.array([0, 1, d - 1, d, (1 << 32) - 1], dtype=np.uint64)])
    x = x[x < (1 << 32)]
    magic = np.uint64(0xFFFFFFFF if d <= 1 else (1 << 32) // d)
    got = (x * magic) >> np.uint64(32)
    got = np.where(x - got * np.uint64(d) >= d, got + np.uint64(1), got)
    np.testing.assert_array_equal(got, x // np.uint64(d))


def test_band_heights_use_the_same_numbers():
    assert [(1 << 32) // h for h in (4, 3, 2)] == [0x40000000, 0x55555555, 0x80000000]


def test_quotients_of_copies():
    """unit / copies by 2^32 / copies + 1 for up to 2^25 units, and a copy's number / blocks of rows in 12 bits."""
    x = np.concatenate([np.arange(1 << 16), np.arange((1 << 25) - (1 << 16), 1 << 25)]).astype(np.uint64)
    for copies in range(2, 129):
        got = (x * np.uint64((1 << 32) // copies + 1)) >> np.uint64(32)
        np.testing.assert_array_equal(got, x // np.uint64(copies))
    rest = np.arange(128)
    for blocks in range(1, 17):
        np.testing.assert_array_equal(rest * ((4096 + blocks - 1) // blocks) >> 12, rest // blocks)


def test_leading_arguments_are_asked_for_in_registers():
    assert "-amdgpu-kernarg-preload-count=16" in HIPCC_FLAGS


@pytest.mark.gpu
@pytest.mark.parametrize("k,gs,wks,wn", [(4096, 4, 8, 1), (4096, 4, 8, 2), (4096, 8, 4, 1), (4096, 16, 2, 7), (3584, 7, 4, 1), (3584, 14, 2, 3),
                                         (2048, 2, 4, 1), (4224, 4, 4, 2), (512, 1, 4, 1), (384, 1, 2, 1)])
@pytest.mark.parametrize("m", [1, 3, 5, 9, 15, 16, 21])
def test_activation_fill_of_every_shape(device, k, gs, wks, wn, m):
    """Workgroups whose wavefronts are a whole number of pieces of a row, of rows, or neither, slabs that end inside K and past it, and rows
    between the numbers that are staged: a row that is not there leaves the others alone."""
    import torch

    from oracle import w4a16 as o
    from tests.helpers import W4A16Layer, check_gemm_close
    from vllm_amd import _tuning
    n = 192
    case = o.make_w4a16_case(k, n, 128, asym=bool(m & 1), seed=k + m + gs)
    layer = W4A16Layer(case, device)
    a = torch.randn(m, k, generator=torch.Generator().manual_seed(m)).to(torch.bfloat16).to(device)
    with _tuning.override(decode_impl=1, decode2_gs=gs, decode2_wks=wks, decode2_wn=wn):
        check_gemm_close(layer(a), o.gemm_ref(a.cpu(), o.case_w_ref(case)), f"k={k} plan {gs}, {wks}, {wn} m={m}")
    assert bool((layer.workspace == 0).all())
