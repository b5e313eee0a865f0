"""The tile choice of a GEMM changes no bit: problems on both sides of
every edge of the rule (one tile to several per CU, strips up to and past 32
wide, odd sizes and leading dimensions, single rows and columns, shifted
bases, short and partial k-stages) give the same result as in child processes
that force the direct-to-LDS kernels and the register-staged ones' 128x128
(cut into whole tiles and strips), 64x64 and 32x32 tiles, in FP64 and in FP32, and all are within a
rounding bound of the product (FP64 1e-13; FP32 the a-priori 2^-24 (k + 2) per
element on |A||B|)."""
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
    ("N", "N", 2048, 2048, 48, 0, 0), ("T", "N", 1281, 1125, 80, 1, 0), ("N", "T", 1125, 1058, 96, 0, 1), ("T", "N", 3000, 40, 128, 0, 0), ("N", "N", 31, 3000, 96, 0, 0),
]


def results(dev, dtype):
    out = []
    gemm = dgamd.dgemm_t if dtype == torch.float64 else dgamd.sgemm_t
    for i, (oa, ob, m, n, k, pad, off) in enumerate(SHAPES):
        print("tile rule", dtype, oa, ob, m, n, k, pad, off, flush=True)
        ra, ca = (m, k) if oa == "N" else (k, m)
        rb, cb = (k, n) if ob == "N" else (n, k)
        dims = ((ra, ca), (rb, cb), (m, n))
        bufs = []
        for j, (r, c) in enumerate(dims):
            # the last column ends with the buffer: no padding after it
            b = torch.empty(off + (r + pad) * (c - 1) + r, dtype=dtype, device=dev)
            dgamd.generate_t(3 * i + j + 1, dgamd.DG_DIST_UNIFORM_PM1, b)
            bufs.append(b)
        A, B, C = (b[off:] for b in bufs)
        start = C.clone()
        gemm(oa, ob, m, n, k, 1.5, A, ra + pad, B, rb + pad, -0.5, C, m + pad)
        out.append((C.clone(), start, A, B, dims))
    return out


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_same_bits_on_every_tile(dev, tmp_path, dtype):
    got = results(dev, dtype)
    whole = torch.int64 if dtype == torch.float64 else torch.int32
    for (oa, ob, m, n, k, pad, off), (C, start, A, B, dims) in zip(SHAPES, got):
        a, b, c, c0 = [x.as_strided((r, q), (1, r + pad)).cpu().numpy().astype(np.float64)
                       for x, (r, q) in zip((A, B, C, start), dims + (dims[2],))]
        a, b = a if oa == "N" else a.T, b if ob == "N" else b.T
        ref = 1.5 * (a @ b) - 0.5 * c0
        if dtype == torch.float64:
            assert np.linalg.norm(c - ref) <= 1e-13 * np.linalg.norm(ref)
        else:
            assert np.all(np.abs(c - ref) <= 2.0 ** -24 * (k + 2) * (1.5 * np.abs(a) @ np.abs(b) + 0.5 * np.abs(c0)))
    for tile in ("direct", "128x128", "64x64", "32x32"):
        path = str(tmp_path / tile)
        subprocess.run([sys.executable, os.path.abspath(__file__), path, str(dtype)], check=True, timeout=100,
                       env=dict(os.environ, DG_GEMM_TILE=tile))
        for shape, mine, other in zip(SHAPES, got, torch.load(path, weights_only=True)):
            assert torch.equal(mine[0].cpu().view(whole), other.view(whole)), (tile, shape)


if __name__ == "__main__":
    torch.save([x[0].cpu() for x in results(torch.device("cuda"), getattr(torch, sys.argv[2].split(".")[1]))], sys.argv[1])
