"""FP32 products of short K (sgemm_short_kernel) at the sizes where it can go
wrong: every remainder of a 16-deep step, whole and partial tiles, one row,
one column, and a strip.  The results are within a rounding bound of the product
and the bits of sgemm_kernel, which a process with DG_GEMM_TILE=64x64 runs on
the same calls.  Operands end with their buffers, C is not read with beta = 0,
and nothing but C is written."""
import os
import subprocess
import sys

import numpy as np
import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "distributed-gemm-thesis_amd"))
import dgamd  # noqa: E402

pytestmark = pytest.mark.gpu

CALLS = [(oa, ob, m, n, k, pad, beta) for oa in "NT" for ob in "NT"
         for i, (m, n) in enumerate([(1, 1), (1, 70), (37, 129), (63, 64), (64, 64), (65, 3), (103, 200), (127, 66), (130, 61)])
         for j, k in enumerate([1, 2, 3, 15, 16, 17, 31, 32, 33, 48, 63])
         for pad, beta in [((0, 1, 4)[(i + j) % 3], (0.0, -0.5)[(i + j) % 2])]]
# cut into whole 128x128 tiles and strips of 8 rows and 4 columns: the strip of rows is short
CALLS += [(oa, ob, 48 * 128 + 8, 48 * 128 + 4, 32, 0, 1.0) for oa, ob in ("TN", "NN")]
STRIP = 8


def results(dev):
    out = []
    for i, (oa, ob, m, n, k, pad, beta) in enumerate(CALLS):
        if i % 50 == 0:
            print(oa, ob, m, n, k, pad, beta, flush=True)
        bufs = []
        for j, (r, c) in enumerate([(m, k) if oa == "N" else (k, m), (k, n) if ob == "N" else (n, k), (m, n)]):
            b = torch.full(((r + pad) * c,), float("nan"), dtype=torch.float32, device=dev)
            x = torch.empty(r * c, dtype=torch.float32, device=dev)
            dgamd.generate_t(3 * i + j + 1, dgamd.DG_DIST_UNIFORM_PM1, x)
            if j < 2 or beta:
                b.view(c, r + pad)[:, :r] = x.view(c, r)
            bufs.append((b if j == 2 else b[: (r + pad) * (c - 1) + r].clone(), r + pad, r, c))
        (A, lda, ra, ca), (B, ldb, rb, cb), (C, ldc, _, _) = bufs
        c0 = C.clone()
        dgamd.sgemm_t(oa, ob, m, n, k, 1.5, A, lda, B, ldb, beta, C, ldc)
        a, b = A.as_strided((ra, ca), (1, lda)), B.as_strided((rb, cb), (1, ldb))
        a, b = a if oa == "N" else a.t(), b if ob == "N" else b.t()
        c0, C = c0.view(n, ldc), C.view(n, ldc)
        if m > 1000:
            a, c0, C = a[m - STRIP:], c0[:, m - STRIP:], C[:, m - STRIP:].clone()
        out.append((a, b, c0, C))
    return out


def test_bits_and_bound(dev, tmp_path):
    got = results(dev)
    for (oa, ob, m, n, k, pad, beta), (A, B, c0, C) in zip(CALLS, got):
        a, b, before, c = [x.cpu().numpy() for x in (A, B, c0, C)]
        a, b, m = a.astype(np.float64), b.astype(np.float64), a.shape[0]
        assert np.isnan(c[:, m:]).all()
        old = beta * before[:, :m].T.astype(np.float64) if beta else np.zeros((m, n))
        bound = 2.0 ** -24 * (k + 2) * (1.5 * np.abs(a) @ np.abs(b) + np.abs(old))
        assert np.all(np.abs(c[:, :m].T - (1.5 * (a @ b) + old)) <= bound), (oa, ob, m, n, k, pad, beta)
    path = str(tmp_path / "c")
    env = {k: v for k, v in os.environ.items() if not k.startswith("DG_GEMM_")}
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), path], timeout=60,
                       env=dict(env, DG_GEMM_TILE="64x64"), capture_output=True, text=True)
    assert r.returncode == 0, (r.stdout[-500:], r.stderr[-2000:])
    for call, x, other in zip(CALLS, got, torch.load(path, weights_only=True)):
        assert torch.equal(x[3].cpu().view(torch.int32), other.view(torch.int32)), call


if __name__ == "__main__":
    torch.save([x[3].cpu() for x in results(torch.device("cuda"))], sys.argv[1])
