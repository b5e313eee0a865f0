"""Block-cyclic unpacking in row blocks of 16 to 32 that share lines, each XCD
on an eighth of the column: row block counts around multiples of eight, fewer
than eight, a short last block, and blocks at the ends of the rule.  Unpacking
moves, so every bit agrees with the CPU oracle, and nothing else is written."""
import numpy as np
import pytest
import torch

import dgamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mb", [15, 16, 17, 24, 31, 32, 33])
@pytest.mark.parametrize("blocks,short", [(1, 3), (1, 0), (3, 1), (8, 0), (8, 5), (9, 0), (63, 7), (65, 0)])
@pytest.mark.parametrize("P,Q,nb,pad,off", [(2, 2, 4, 1, 0), (3, 2, 5, 0, 1), (4, 1, 7, 5, 0)])
def test_unpack_row_blocks(dev, mb, blocks, short, P, Q, nb, pad, off):
    rows, cols = blocks * mb - short, 23
    ldg = rows + pad
    G = np.random.default_rng(rows + mb).standard_normal(ldg * cols)
    packed = torch.from_numpy(oracle.pack_block_cyclic(G, ldg, rows, cols, mb, nb, P, Q)).to(dev)
    buf = torch.full((ldg * cols + off + 3,), 7.0, dtype=torch.float64, device=dev)
    dgamd.unpack_block_cyclic_t(packed, mb, nb, P, Q, buf[off:off + ldg * cols], ldg, rows, cols)
    got = buf.cpu().numpy()
    assert np.all(got[:off] == 7.0) and np.all(got[off + ldg * cols:] == 7.0)
    got = got[off:off + ldg * cols].reshape(cols, ldg)
    assert np.array_equal(got[:, :rows], G.reshape(cols, ldg)[:, :rows]) and np.all(got[:, rows:] == 7.0)
