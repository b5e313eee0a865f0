"""Column runs that are whole 128-byte lines and runs that share lines, with
either buffer starting 0-3 elements past a line: pack and unpack are moves, so
every bit agrees with the CPU oracle and nothing else is written."""
import numpy as np
import pytest
import torch

import dgamd
import oracle

pytestmark = pytest.mark.gpu


def shifted(a, off, dev):
    """Device copy of `a` starting `off` elements past a line, 7.0 around it."""
    buf = torch.full((a.size + off + 4,), 7.0, dtype=torch.from_numpy(a[:0]).dtype, device=dev)
    view = buf[off:off + a.size]
    view.copy_(torch.from_numpy(a))
    return buf, view


@pytest.mark.parametrize("goff,poff", [(0, 0), (1, 0), (0, 1), (1, 1), (2, 2)])
@pytest.mark.parametrize("rows,cols,ldg,parts,mb,nb,P,Q", [
    (96, 7, 96, 2, 32, 3, 3, 2), (96, 7, 112, 6, 16, 2, 2, 3), (96, 7, 97, 3, 32, 3, 2, 2), (127, 9, 127, 1, 127, 4, 1, 2),
    (129, 5, 144, 2, 130, 5, 2, 1), (640, 5, 640, 5, 128, 1, 4, 2), (643, 5, 643, 5, 33, 2, 3, 2)])
def test_pack_unpack_runs(dev, rows, cols, ldg, parts, mb, nb, P, Q, goff, poff):
    rng = np.random.default_rng(rows * 7 + ldg + parts)
    G = rng.standard_normal(ldg * cols)
    ro, co = oracle.block_splits(rows, parts), oracle.block_splits(cols, 2)
    zero = np.zeros(rows * cols)
    for ref, pack, unpack in (
            (oracle.pack_block2d(G, ldg, rows, cols, ro, co),
             lambda g, p: dgamd.pack_block2d_t(g, ldg, rows, cols, ro, co, p),
             lambda p, g: dgamd.unpack_block2d_t(p, ro, co, g, ldg, rows, cols)),
            (oracle.pack_block_cyclic(G, ldg, rows, cols, mb, nb, P, Q),
             lambda g, p: dgamd.pack_block_cyclic_t(g, ldg, rows, cols, mb, nb, P, Q, p),
             lambda p, g: dgamd.unpack_block_cyclic_t(p, mb, nb, P, Q, g, ldg, rows, cols))):
        _, g = shifted(G, goff, dev)
        pbuf, p = shifted(zero, poff, dev)
        pack(g, p)
        got = pbuf.cpu().numpy()
        assert np.array_equal(got[poff:poff + rows * cols], ref)
        assert np.all(got[:poff] == 7.0) and np.all(got[poff + rows * cols:] == 7.0)
        gbuf, g2 = shifted(np.full(ldg * cols, 3.5), goff, dev)
        unpack(p, g2)
        got = gbuf.cpu().numpy()
        assert np.all(got[:goff] == 7.0) and np.all(got[goff + ldg * cols:] == 7.0)
        got = got[goff:goff + ldg * cols].reshape(cols, ldg)
        assert np.array_equal(got[:, :rows], G.reshape(cols, ldg)[:, :rows]) and np.all(got[:, rows:] == 3.5)


@pytest.mark.parametrize("soff,doff", [(0, 0), (1, 0), (3, 2), (0, 3)])
@pytest.mark.parametrize("rows,cols,lds,ldd", [(64, 5, 64, 96), (257, 4, 260, 257), (3, 6, 5, 4)])
def test_copy_block_f32_runs(dev, rows, cols, lds, ldd, soff, doff):
    src = np.random.default_rng(rows + soff).standard_normal(lds * cols).astype(np.float32)
    _, s = shifted(src, soff, dev)
    dbuf, d = shifted(np.full(ldd * cols, 2.5, np.float32), doff, dev)
    dgamd.copy_block_t(rows, cols, s, lds, d, ldd)
    got = dbuf.cpu().numpy()[doff:doff + ldd * cols].reshape(cols, ldd)
    assert np.array_equal(got[:, :rows], src.reshape(cols, lds)[:, :rows]) and np.all(got[:, rows:] == 2.5)
