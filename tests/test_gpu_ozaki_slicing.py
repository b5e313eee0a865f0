"""Slicing of both operands around its 32-row by 128-k tiles: sizes at the
tile edges, padded and odd leading dimensions, buffers 8 bytes past a 16-byte
boundary, lines contiguous and strided, against the CPU oracle bit for bit."""
import numpy as np
import pytest
import torch

import dgamd
import oracle

pytestmark = pytest.mark.gpu

KINDS = [(dgamd.DG_OZAKI_INT8, oracle.OZ_INT8_BITS), (dgamd.DG_OZAKI_BF16, oracle.OZ_BF16_BITS)]


@pytest.mark.parametrize("kind,bits", KINDS)
@pytest.mark.parametrize("opA,opB", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,s,pad,off", [(32, 64, 128, 8, 0, 0), (33, 31, 129, 10, 1, 1), (1, 65, 127, 16, 3, 0),
                                             (95, 1, 260, 3, 0, 1), (257, 290, 1, 4, 2, 1), (40, 70, 515, 12, 1, 0)])
def test_slices_bit_exact(dev, kind, bits, opA, opB, m, n, k, s, pad, off):
    rng = np.random.default_rng(m + 3 * n + k)

    def operand(rows, cols):
        a = np.ldexp(rng.uniform(-1, 1, (rows, cols)), rng.integers(-20, 21, (rows, cols)))
        buf = torch.full((off + (rows + pad) * cols,), float("nan"), dtype=torch.float64, device=dev)
        view = buf[off:]
        view.reshape(cols, rows + pad)[:, :rows].copy_(torch.from_numpy(np.ascontiguousarray(a.T)))
        return a, view

    a, A = operand(*((m, k) if opA == "N" else (k, m)))
    b, B = operand(*((k, n) if opB == "N" else (n, k)))
    c, C = operand(m, n)
    dgamd.ozaki_dgemm_t(opA, opB, m, n, k, 1.5, A, a.shape[0] + pad, B, b.shape[0] + pad, -0.5, C, m + pad, s, kind)
    got = C.cpu().numpy().reshape(n, m + pad)
    ref = oracle.ozaki_dgemm(np.ascontiguousarray(a if opA == "N" else a.T),
                             np.ascontiguousarray(b if opB == "N" else b.T), s, 1.5, -0.5, c, bits=bits)
    assert np.array_equal(got[:, :m].T.copy().view(np.uint64), np.ascontiguousarray(ref).view(np.uint64))
    assert np.all(np.isnan(got[:, m:]))
