"""The tile choice of an FP64 GEMM changes no bit: problems on both sides of
every edge of the rule (one tile to several per CU, strips up to and past 32
wide, odd sizes and leading dimensions, single rows and columns, shifted
bases, short and partial k-stages) give the same result as in child processes
that force 128x128 tiles (direct-to-LDS kernels), 64x64 and 32x32
(register-staged kernel), and all are within 1e-13 of the FP64 product."""
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

# opA, opB, m, n, k, pad of every leading dimension, bases one element off
SHAPES = [
    ("N", "N", 64, 64, 16, 0, 0), ("T", "N", 65, 63, 33, 0, 0), ("N", "T", 33, 31, 15, 1, 1), ("T", "T", 1, 70, 17, 0, 0),
    ("N", "N", 70, 1, 1, 0, 0), ("N", "T", 1, 1, 40, 0, 1), ("N", "N", 512, 512, 512, 0, 0), ("T", "N", 511, 513, 1000, 1, 1),
    ("N", "T", 1031, 777, 272, 1, 0), ("T", "T", 1040, 1056, 256, 0, 0), ("N", "N", 1089, 833, 256, 2, 1),
    ("N", "N", 2048, 2048, 48, 0, 0), ("T", "N", 3000, 40, 128, 0, 0), ("N", "N", 31, 3000, 96, 0, 0),
]


def results(dev):
    out = []
    for i, (oa, ob, m, n, k, pad, off) in enumerate(SHAPES):
        print("tile rule", oa, ob, m, n, k, pad, off, flush=True)
        ra, ca = (m, k) if oa == "N" else (k, m)
        rb, cb = (k, n) if ob == "N" else (n, k)
        dims = ((ra, ca), (rb, cb), (m, n))
        bufs = []
        for j, (r, c) in enumerate(dims):
            # the last column ends with the buffer: no padding after it
            b = torch.empty(off + (r + pad) * (c - 1) + r, dtype=torch.float64, device=dev)
            dgamd.generate_t(3 * i + j + 1, dgamd.DG_DIST_UNIFORM_PM1, b)
            bufs.append(b)
        A, B, C = (b[off:] for b in bufs)
        start = C.clone()
        dgamd.dgemm_t(oa, ob, m, n, k, 1.5, A, ra + pad, B, rb + pad, -0.5, C, m + pad)
        out.append((C.clone(), start, A, B, dims))
    return out


def test_same_bits_on_every_tile(dev, tmp_path):
    got = results(dev)
    for (oa, ob, m, n, k, pad, off), (C, start, A, B, dims) in zip(SHAPES, got):
        dense = [x.as_strided((r, c), (1, r + pad)).cpu().numpy() for x, (r, c) in zip((A, B, C, start), dims + (dims[2],))]
        a, b, c, c0 = dense
        ref = 1.5 * ((a if oa == "N" else a.T) @ (b if ob == "N" else b.T)) - 0.5 * c0
        assert np.linalg.norm(c - ref) <= 1e-13 * np.linalg.norm(ref)
    for tile in ("128x128", "64x64", "32x32"):
        path = str(tmp_path / tile)
        subprocess.run([sys.executable, os.path.abspath(__file__), path], check=True, timeout=100,
                       env=dict(os.environ, DG_GEMM_TILE=tile))
        for shape, mine, other in zip(SHAPES, got, torch.load(path, weights_only=True)):
            assert torch.equal(mine[0].cpu().view(torch.int64), other.view(torch.int64)), (tile, shape)


if __name__ == "__main__":
    torch.save([x[0].cpu() for x in results(torch.device("cuda"))], sys.argv[1])
