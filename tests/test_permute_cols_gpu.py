"""Column permutation (act_order's gather of the activations): rows dealt out to workgroups."""
from __future__ import annotations

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 3, 4, 333, 1024, 1500, 2500])
@pytest.mark.parametrize("k", [8, 1032, 2048, 4096, 8200])
def test_permute_cols_rows_per_workgroup(device, m, k):
    """One, two and four rows to a workgroup, with a last workgroup that holds fewer; K below and beyond a workgroup's threads."""
    import vllm_amd._custom_ops as ops
    perm = torch.from_numpy(np.random.default_rng(k).permutation(k).astype(np.int32))
    a = torch.randn(m, k + 8, generator=torch.Generator().manual_seed(m)).to(torch.bfloat16)[:, :k]
    assert torch.equal(ops.permute_cols(a.to(device), perm.to(device)).cpu(), a[:, perm.long()])


@pytest.mark.parametrize("m,k", [(1024, 2056), (1025, 2056), (2049, 1536), (2049, 4088), (1025, 9088), (2049, 9088), (1281, 16376), (1300, 4104), (4100, 4104),
                                 (2500, 1528), (600, 65528)])
def test_permute_cols_threads_of_a_row(device, m, k):
    """One row to a workgroup of 256 or 512 threads, both sides of each line between them and of the lines to more rows."""
    import vllm_amd._custom_ops as ops
    perm = torch.from_numpy(np.random.default_rng(k).permutation(k).astype(np.int32)).to(device)
    a = torch.randn(m, k, device=device, generator=torch.Generator(device=device).manual_seed(m)).to(torch.bfloat16)
    assert torch.equal(ops.permute_cols(a, perm), a[:, perm.long()])
