"""The allocation-free grouped GEMM's capacity is the one that its message
names: a batch a little smaller runs, one a little larger is refused."""
import re

import pytest
import torch

import dgamd

pytestmark = pytest.mark.gpu


def test_capacity_is_the_one_named(dev):
    x = torch.ones(16, dtype=torch.float64, device=dev)
    out = torch.zeros((4000, 16), dtype=torch.float64, device=dev)
    descs = [dgamd.gemm_desc("N", "N", 4, 4, 4, 1.0, x, 4, x, 4, 0.0, c, 4) for c in out]
    with pytest.raises(dgamd.DGError) as e:
        dgamd.grouped_dgemm_noalloc_t(descs)
    assert e.value.status == dgamd.DG_ERR_WORKSPACE
    named = int(re.search(r"about (\d+) problems", str(e.value)).group(1))
    with pytest.raises(dgamd.DGError):
        dgamd.grouped_dgemm_noalloc_t(descs[: named + named // 100])
    torch.cuda.synchronize()
    assert not out.any()
    n = named - named // 100  # each table starts on a 256-byte boundary
    dgamd.grouped_dgemm_noalloc_t(descs[:n])
    torch.cuda.synchronize()
    assert torch.all(out[:n] == 4.0) and not out[n:].any()
