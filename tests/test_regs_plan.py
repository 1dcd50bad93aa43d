"""Plans of the W4A16 kernel with activations in registers: the price formula, the choices it makes over recorded timings, scratch."""
from __future__ import annotations

import ctypes
import importlib.util
import os
import random

import numpy as np
import pytest

from vllm_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def fit():
    spec = importlib.util.spec_from_file_location("plan_price_fit", os.path.join(ROOT, "profiles", "plan_prices", "fit.py"))
    module = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(module)
    return module


def _plan(m, n, k, sub, w8):
    """n-tiles, m-blocks, wavefronts, parts of K, predicted us, us of what takes it otherwise, 1 if this kernel takes it."""
    plan = (ctypes.c_double * 7)()
    _lib.check(_lib.load().vaq_w4a16_regs_plan(m, n, k, sub, w8, plan))
    return list(plan)


def test_price_formula_of_the_fit_is_the_one_of_the_library(fit):
    rng, rows, want = random.Random(3), [], []
    for _ in range(300):
        m, k, n = int(256 ** rng.random()), 128 * int(110 ** rng.random()), 64 * int(2 * 1000 ** rng.random())
        sub, w8 = rng.choice([1, 2, 4]), rng.choice([0, 1])
        j, mb, nw, sk, us, _, _ = _plan(m, n, k, sub, w8)
        rows.append([k, n, m, sub, w8, 0, 0, nw, j, mb, sk, 1.0])
        want.append(us)
    t = fit.Regs()
    t.load_rows(np.array(rows))
    assert np.allclose(t.prices(), want, rtol=1e-9)
    lib, plan = _lib.load(), (ctypes.c_double * 7)()
    for bad in ((0, 64, 128, 1), (8, 60, 128, 1), (8, 64, 100, 1), (8, 64, 128, 3), (300, 64, 128, 1)):
        assert lib.vaq_w4a16_regs_plan(*bad, 0, plan) == _lib.VAQ_ERR_INVALID_ARG


def test_choices_over_recorded_timings(fit):
    """Every format and number of rows: the cheapest plan is a fast one, and the calls that go to this kernel gain by it."""
    t = fit.Regs()
    t.load([os.path.join(ROOT, "profiles", "plan_prices", "w4_regs.csv.gz")])
    price = np.where(t.allowed(), t.prices(), np.inf)
    n = t.key.max() + 1
    best, cheapest, took = (np.full(n, np.inf) for _ in range(3))
    np.minimum.at(best, t.key, t.us)
    np.minimum.at(cheapest, t.key, price)
    at = price == cheapest[t.key]
    took[t.key[at]] = t.us[at]
    first = np.zeros(n, int)
    first[t.key] = np.arange(len(t.key))
    # calls that go to this kernel, where the library's plan was among those timed
    ratio = np.full(n, np.nan)
    for q, i in enumerate(first):
        j, mb, nw, sk, _, _, takes = _plan(int(t.m[i]), int(t.n[i]), int(t.k[i]), int(t.sub[i]), int(t.w8[i]))
        same = np.flatnonzero((t.key == q) & (t.j == j) & (t.mb == mb) & (t.nw == nw) & (t.sk == sk)) if takes else []
        if len(same):
            ratio[q] = t.us[same[0]] / t.other[q]
    for w8 in (0, 1):
        for sub in (1, 2, 4):
            here = (t.sub[first] == sub) & (t.w8[first] == w8)
            several = here & (np.bincount(t.key, minlength=n) > 1)      # (of some problems only the plan that the library chooses was timed)
            assert np.exp(np.log(took[several] / best[several]).mean()) < 1.025
            gain = ratio[here & np.isfinite(ratio)]
            assert len(gain) > 100 and np.exp(np.log(gain).mean()) < 0.9 and (gain > 1.03).mean() < 0.1 and (gain > 1.15).mean() < 0.01


def test_scratch_of_every_plan_fits_the_library_owned_one():
    """Parts of K: within the scratch of the entry point that owns it, the counters of a layer, and what the workspace query says."""
    from vllm_amd.layers.quantization.utils.marlin_utils import marlin_workspace_ints
    lib, rng, split = _lib.load(), random.Random(1), 0
    for _ in range(400):
        m, k, n = int(256 ** rng.random()), 128 * int(220 ** rng.random()), 64 * int(2 * 1000 ** rng.random())
        group, wtype = rng.choice([128, 64, 32]), rng.choice([_lib.VAQ_WTYPE_U4B8, _lib.VAQ_WTYPE_U8B128])
        if k * n >= 1 << 31:
            continue
        j, mb, nw, sk, _, _, takes = _plan(m, n, k, 128 // group, int(wtype == _lib.VAQ_WTYPE_U8B128))
        rb = -(-m // (16 * int(mb)))
        tmp, counters = (int(sk) * n * rb * int(mb) * 64, n // 16 * rb * int(mb)) if sk > 1 else (0, 0)
        assert tmp <= 16 << 20 and counters <= marlin_workspace_ints(n) and counters <= 65536
        if takes:
            sizes = [ctypes.c_size_t() for _ in range(3)]
            _lib.check(lib.vaq_w4a16_gemm_workspace_of_format(m, n, k, group, wtype, 0, 0, *map(ctypes.byref, sizes)))
            assert sizes[0].value >= tmp and sizes[2].value >= counters
            split += sk > 1
    assert split > 10


@pytest.mark.parametrize("k,m4,m16", [(512, 26.5, 27.2), (1024, 33.4, 34.0), (2048, 38.0, 39.4), (3072, 47.6, 50.3), (4096, 54.9, 59.0), (5120, 153.7, 155.2)])
def test_vocabulary_layers_are_weighed_against_the_kernel_that_runs(k, m4, m16):
    """N from 65536 on, 3 .. 16 rows: without this kernel the register-resident one runs (timed us at N = 128256, cold), not the LDS-staged one."""
    for m, us in ((4, m4), (16, m16)):
        *_, other, takes = _plan(m, 128256, k, 1, 0)
        assert abs(other / us - 1) < 0.25 and takes


@pytest.mark.parametrize("k,n,m,takes", [(4096, 4096, 16, 0), (4096, 3072, 16, 0), (2048, 10240, 16, 0), (2048, 4608, 32, 0), (11008, 3584, 1, 0), (13824, 3584, 2, 0),
                                         (4096, 6144, 4, 1), (4096, 6144, 16, 1), (5120, 5120, 1, 1), (5120, 5120, 16, 1), (4096, 4096, 24, 1), (4096, 28672, 32, 1)])
def test_layers_where_one_kernel_is_well_ahead(k, n, m, takes):
    """Timed 4 .. 11 % behind and 5 .. 25 % ahead of the decode kernel."""
    assert _plan(m, n, k, 1, 0)[-1] == takes


@pytest.mark.parametrize("k,n,m,sub,single", [(9344, 2304, 15, 1, False), (8192, 2304, 15, 1, True), (4736, 2304, 15, 1, True)])
def test_long_streams_of_one_n_tile_of_8_bit_codes(k, n, m, sub, single):
    """73 k-tiles on eight wavefronts, ten turns: 10.05 us with one n-tile and K whole, 8.8 with two and K in three parts, at prices 6 % apart."""
    assert (_plan(m, n, k, sub, 1)[0] == 1) == single


@pytest.mark.parametrize("k,n,m,sub", [(21760, 12096, 157, 1), (14592, 17920, 129, 2), (3456, 5888, 189, 2), (13056, 2880, 69, 2), (11648, 20160, 139, 2)])
def test_unrounded_weights_stay_where_they_were(k, n, m, sub):
    """Calls that the kernel with operands in registers took before there were 256 x 256 tiles: these round the weights to 16 bits."""
    assert _plan(m, n, k, sub, 0)[-1] == 1


def test_no_call_is_weighed_against_256_x_256_tiles():
    """Where those are the cheapest tiles, what this kernel is weighed against costs more than they do."""
    rng, tile, seen = random.Random(7), (ctypes.c_double * 4)(), 0
    for _ in range(3000):
        m, k, n = rng.randint(100, 256), 128 * int(16 * 14 ** rng.random()), 64 * int(64 * 30 ** rng.random())
        sub, w8 = rng.choice([1, 2, 4]), rng.choice([0, 1])
        if k * n >= 1 << 30:
            continue
        _lib.check(_lib.load().vaq_w4a16_tile_plan(m, n, k, sub, w8, 0, tile))
        if tile[0] == 48:
            # (4-bit codes in groups of 64 / 32: strips at the prices that the shares were set at, up to 0.4 % below their own)
            assert _plan(m, n, k, sub, w8)[5] > tile[3] * (0.99 if sub > 1 and not w8 else 1)
            seen += 1
    assert seen > 200
