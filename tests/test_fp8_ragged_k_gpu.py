"""FP8 GEMMs whose K ends inside a step of the tile kernels: the bytes behind K are a neighbouring row's, or nobody's."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _case(m, n, k, seed, device, off=0, behind=64):
    """Small integers as e4m3 (every product and sum exact), in rows that lie `off + behind` further apart than K with NaN codes around them."""
    g = torch.Generator().manual_seed(seed)
    a, w = torch.randint(-2, 3, (m, k), generator=g).float(), torch.randint(-1, 2, (n, k), generator=g).float()
    views = []
    for x in (a, w):
        wide = torch.full((x.shape[0], off + k + behind), 0x7f, dtype=torch.uint8, device=device).view(torch.float8_e4m3fn)
        wide[:, off:off + k] = x.to(torch.float8_e4m3fn).to(device)
        views.append(wide[:, off:off + k])
    return views[0], views[1].t(), a @ w.t()


def _run(a, b, device):
    import vllm_amd._custom_ops as ops
    m, n = a.shape[0], b.shape[1]
    return ops.cutlass_scaled_mm(a, b, torch.ones(m, 1, device=device), torch.ones(n, 1, device=device), torch.float16).cpu().float()


@pytest.mark.parametrize("cfg,depth", [(1, 5), (13, 4), (14, 5), (15, 5), (16, 5), (17, 3), (19, 3)])
@pytest.mark.parametrize("rest", [16, 48, 64, 80, 112])
def test_every_tile_shape_and_end_of_k_exact(device, cfg, depth, rest):
    """Every shape with every kind of last step, from a K below one step to past the second turn of the ring, whole and in parts."""
    from vllm_amd import _tuning
    for steps in (0, 1, 2, depth - 1, depth, 2 * depth + 1):
        k, split = 128 * steps + rest, 2 if steps == 2 * depth + 1 else 1
        m, n = 1 + (97 * steps + 31 * rest) % 600, 16 + (112 * steps + 16 * rest) % 560
        a, b, want = _case(m, n, k, cfg + rest, device)
        with _tuning.override(fp8_path=2, fp8_tile_cfg=cfg, fp8_split=split):
            assert torch.equal(_run(a, b, device), want), (cfg, m, n, k, split)
    import vllm_amd._custom_ops as ops
    assert all(bool((t == 0).all()) for t in ops._FP8_COUNTERS.values())


@pytest.mark.parametrize("cfg", [1, 13, 14, 15, 16, 17, 19])
def test_last_columns_of_their_storage_exact(device, cfg):
    """Operands that end with their storage: what a last step may ask for behind K does not exist."""
    from vllm_amd import _tuning
    for m, n, k, off in ((256, 384, 432, 64), (131, 400, 848, 48), (300, 272, 144, 16), (257, 96, 688, 512)):
        a, b, want = _case(m, n, k, cfg, device, off=off, behind=0)
        with _tuning.override(fp8_path=2, fp8_tile_cfg=cfg):
            assert torch.equal(_run(a, b, device), want), (cfg, m, n, k)


@pytest.mark.parametrize("m,n,k", [(33, 1024, 1040), (65, 4352, 4320), (100, 2048, 8400), (250, 1536, 1616), (877, 1472, 5728), (2100, 2112, 2512), (64, 960, 14320),
                                   (198, 5632, 1472), (40, 18368, 1248), (700, 512, 704), (1700, 1024, 5968), (48, 256, 16)])
def test_as_chosen_exact(device, m, n, k):
    """Plans as they are chosen (rotated starts, a tile row past M, K in parts), rows without gaps."""
    a, b, want = _case(m, n, k, k, device, behind=0)
    assert torch.equal(_run(a, b, device), want)


def test_operands_beyond_2_gib(device):
    """Rows so far apart that a place in the operand does not leave room for the offset of a chunk past K: K % 128 = 64 takes the tiles by slices
    of 64 bytes, other K the kernel that tests every load."""
    for k in (192, 208):
        m, n, pitch = 70, 64, 32 << 20
        g = torch.Generator().manual_seed(k)
        x, w = torch.randint(-2, 3, (m, k), generator=g).float(), torch.randint(-1, 2, (n, k), generator=g).float()
        wide = torch.empty(m * pitch, dtype=torch.uint8, device=device).view(torch.float8_e4m3fn).view(m, pitch)
        wide[:, :k] = x.to(torch.float8_e4m3fn).to(device)
        assert torch.equal(_run(wide[:, :k], w.to(torch.float8_e4m3fn).to(device).t(), device), x @ w.t()), k
        del wide


@pytest.mark.parametrize("rows_far", ["activations", "weights"])
def test_every_tile_shape_beyond_2_gib(device, rows_far):
    """K % 128 = 64 on operands of 2 .. 4 GiB: every shape by slices of 64 bytes (and the 256 x 256 tile), whole and in parts of K, as chosen too."""
    from vllm_amd import _tuning
    pitch = 48 << 20
    k, m, n = 192 + 128 * 4, *((70, 336) if rows_far == "activations" else (300, 80))
    g = torch.Generator().manual_seed(k + m)
    x, w = torch.randint(-2, 3, (m, k), generator=g).float(), torch.randint(-1, 2, (n, k), generator=g).float()
    want = x @ w.t()
    views = [t.to(torch.float8_e4m3fn).to(device) for t in (x, w)]
    far = 0 if rows_far == "activations" else 1
    wide = torch.empty(views[far].shape[0] * pitch, dtype=torch.uint8, device=device).view(torch.float8_e4m3fn).view(-1, pitch)
    wide[:, k:k + 128] = torch.full((1,), 0x7f, dtype=torch.uint8, device=device).view(torch.float8_e4m3fn)
    wide[:, :k] = views[far]
    views[far] = wide[:, :k]
    assert torch.equal(_run(views[0], views[1].t(), device), want)
    for cfg in (1, 3, 4, 5, 6, 7, 9, 13, 14, 15, 16, 17, 19):
        for split in (1, 2):
            with _tuning.override(fp8_path=2, fp8_tile_cfg=cfg, fp8_split=split):
                assert torch.equal(_run(views[0], views[1].t(), device), want), (cfg, split)
