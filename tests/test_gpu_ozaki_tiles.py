"""Large outputs run on 256 x 256 tiles, small ones on 128 x 128 tiles.  An
element depends on its row of op(A) and its column of op(B) alone, so a block
of a large product equals the product of the block's lines, bit for bit; one
block is also checked against the CPU oracle."""
import numpy as np
import pytest
import torch

import dgamd
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,s,k", [
    (dgamd.DG_OZAKI_INT8_CRT, 14, 1), (dgamd.DG_OZAKI_INT8_CRT, 14, 640), (dgamd.DG_OZAKI_INT8_CRT, 15, 769),
    (dgamd.DG_OZAKI_INT8, 8, 100), (dgamd.DG_OZAKI_INT8, 9, 641), (dgamd.DG_OZAKI_BF16, 11, 64),
    (dgamd.DG_OZAKI_BF16, 11, 500)])
def test_block_of_large_product(dev, kind, s, k):
    m, n = 2300, 2100
    rng = np.random.default_rng(k + s)
    a = np.ldexp(rng.uniform(-1, 1, (m, k)), rng.integers(-20, 21, (m, k)))
    b = np.ldexp(rng.uniform(-1, 1, (k, n)), rng.integers(-20, 21, (k, n)))
    A = torch.from_numpy(a).to(dev).t().contiguous()  # column-major m x k
    B = torch.from_numpy(b).to(dev).t().contiguous()
    C = torch.full((n, m), float("nan"), dtype=torch.float64, device=dev)
    dgamd.ozaki_dgemm_t("N", "N", m, n, k, 1.0, A.reshape(-1), m, B.reshape(-1), k, 0.0, C.reshape(-1), m, s, kind)
    for r0, c0, mm, nn in ((0, 0, 256, 256), (2043, 1844, 257, 256), (1000, 700, 60, 70)):
        D = torch.full((nn, mm), float("nan"), dtype=torch.float64, device=dev)
        Ab = A[:, r0:r0 + mm].contiguous()
        Bb = B[c0:c0 + nn].contiguous()
        dgamd.ozaki_dgemm_t("N", "N", mm, nn, k, 1.0, Ab.reshape(-1), mm, Bb.reshape(-1), k, 0.0, D.reshape(-1), mm, s,
                            kind)
        assert torch.equal(C[c0:c0 + nn, r0:r0 + mm], D)
    if kind != dgamd.DG_OZAKI_INT8_CRT:
        bits = oracle.OZ_BF16_BITS if kind == dgamd.DG_OZAKI_BF16 else oracle.OZ_INT8_BITS
        ref = oracle.ozaki_dgemm(np.ascontiguousarray(a[1000:1060]), np.ascontiguousarray(b[:, 700:770]), s, 1.0, 0.0,
                                 np.zeros((60, 70)), bits=bits)
        assert np.array_equal(D.t().cpu().numpy(), ref)
