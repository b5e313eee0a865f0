"""The direct-to-LDS kernels, the register-operand ones and the uncut 128x128
tiles at the sizes where each can go wrong, whichever kernel the estimate
would take there: every process below forces one choice (DG_GEMM_TILE) or
switches one kernel off, and all give the same bits, which are within a
rounding bound of the product.  FP64 shapes reach interior tiles with every
length of pipeline tail, cuts with and without a shifted base (operands 8
bytes off 16-byte alignment), edges, odd step counts and partial k-steps;
tests/test_host_route.py checks that they do.  Also as batches in every
scheduling mode, and K-segmented (Cannon, SUMMA)."""
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

OPS = [(a, b) for a in "NT" for b in "NT"]
# opA, opB, m, n, k, elements that A and B start off a 16-byte boundary, what the direct choice makes of it
SHAPES = [(a, b, 384, 512, 8 * s, 0, 0, "areg") for a, b in OPS for s in (2, 4, 6, 8, 10, 12, 14, 24, 26, 28, 50, 52)]
SHAPES += [(a, b, 3 * 128 + 37, 4 * 128 + 66, k, 0, 0, "cut") for a, b in OPS for k in (16, 208)]
SHAPES += [("N", "N", 127 + 3 * 128 + 20, 4 * 128 + 9, 112, 1, 0, "cut"), ("N", "T", 127 + 3 * 128 + 20, 4 * 128 + 9, 112, 1, 0, "cut"),
           ("N", "T", 3 * 128 + 40, 127 + 4 * 128, 208, 0, 1, "cut"), ("N", "T", 127 + 3 * 128, 127 + 4 * 128 + 100, 16, 1, 1, "cut"),
           ("T", "T", 4 * 128, 127 + 4 * 128 + 40, 208, 0, 1, "cut"), ("N", "T", 255 + 3 * 128, 126 + 4 * 128, 48, 1, 1, "cut")]
SHAPES += [(a, b, 200, 151, k, 0, 0, "edge") for a, b in OPS for k in (8, 40, 42)]
SHAPES += [("N", "N", 700, 701, 24, 1, 0, "edge"), ("N", "T", 701, 700, 26, 1, 1, "edge"), ("T", "N", 513, 640, 250, 0, 0, "edge"),
           ("T", "T", 640, 513, 200, 0, 1, "edge")]
EXPECT = {"areg": lambda dma, edge, gen: dma == 1 and edge == gen == 0,
          "cut": lambda dma, edge, gen: dma == 1 and edge == 0 and gen >= 1,
          "edge": lambda dma, edge, gen: dma == 0 and edge == 1 and gen == 0}
# FP32: interior with every kind of step count, cuts, edges; leading dimensions are multiples of 4
SHAPES32 = [(a, b, 384, 512, 32 * s) for a, b in OPS for s in (1, 2, 3, 4, 5, 13)]
SHAPES32 += [(a, b, 3 * 128 + 40, 4 * 128 + 68, k) for a, b in OPS for k in (32, 224)]
SHAPES32 += [(a, b, 200, 152, k) for a, b in OPS for k in (16, 20, 48)]
RUNS = [{"DG_GEMM_TILE": "direct"}, {"DG_GEMM_TILE": "direct", "DG_GEMM_NO_AREG": "1"},
        {"DG_GEMM_TILE": "direct", "DG_GEMM_NO_NARROW": "1"}, {"DG_GEMM_TILE": "128x128whole"}, {"DG_GEMM_TILE": "64x64"}]


def geometry(oa, ob, m, n, k, unit):
    """Stored (rows, columns, leading dimension) of A, B and C, leading dimensions multiples of `unit`."""
    dims = ((m, k) if oa == "N" else (k, m)), ((k, n) if ob == "N" else (n, k)), (m, n)
    return [(r, c, -(-r // unit) * unit) for r, c in dims]


def product(dev, dtype, i, oa, ob, m, n, k, off_a=0, off_b=0):
    """Operands (each buffer ends with its last element) and C of one product."""
    bufs = []
    for j, ((r, c, ld), off) in enumerate(zip(geometry(oa, ob, m, n, k, 2 if dtype == torch.float64 else 4), (off_a, off_b, 0))):
        b = torch.empty(off + ld * (c - 1) + r, dtype=dtype, device=dev)
        dgamd.generate_t(3 * i + j + 1, dgamd.DG_DIST_UNIFORM_PM1, b)
        bufs.append((b[off:], ld))
    return bufs


def results(dev):
    out = []
    for i, (oa, ob, m, n, k, off_a, off_b, _) in enumerate(SHAPES):
        print("f64", oa, ob, m, n, k, off_a, off_b, flush=True)
        (A, lda), (B, ldb), (C, ldc) = product(dev, torch.float64, i, oa, ob, m, n, k, off_a, off_b)
        dgamd.dgemm_t(oa, ob, m, n, k, 1.5, A, lda, B, ldb, -0.5, C, ldc)
        out.append(C)
    for i, (oa, ob, m, n, k) in enumerate(SHAPES32):
        print("f32", oa, ob, m, n, k, flush=True)
        (A, lda), (B, ldb), (C, ldc) = product(dev, torch.float32, i, oa, ob, m, n, k)
        dgamd.sgemm_t(oa, ob, m, n, k, 1.5, A, lda, B, ldb, -0.5, C, ldc)
        out.append(C)
    for mode in (dgamd.DG_PLAN_NONPERSISTENT, dgamd.DG_PLAN_PERSISTENT):
        print("plan", mode, flush=True)
        keep = [product(dev, torch.float64, i, *s[:7]) for i, s in enumerate(SHAPES)]
        plan = dgamd.GroupedPlan([dgamd.gemm_desc(s[0], s[1], s[2], s[3], s[4], 1.5, A, lda, B, ldb, -0.5, C, ldc)
                                  for s, ((A, lda), (B, ldb), (C, ldc)) in zip(SHAPES, keep)], mode)
        plan.execute()
        torch.cuda.synchronize()
        plan.close()
        out += [C for _, _, (C, _) in keep]
    for oa, ob in OPS:
        print("segments", oa, ob, flush=True)
        x = [torch.empty(512 * 512, dtype=torch.float64, device=dev) for _ in range(6)]
        for j, t in enumerate(x):
            dgamd.generate_t(900 + j, dgamd.DG_DIST_UNIFORM_PM1, t)
        dgamd.cannon25d_t(oa, ob, 512, 512, 512, 1.5, x[0], x[1], -0.5, x[2], 2, 1)
        dgamd.summa_t(oa, ob, 512, 512, 512, 1.5, x[3], x[4], -0.5, x[5], 128, 128, 64, 2, 2)
        out += [x[2], x[5]]
    return out


def test_same_bits_whichever_kernel(dev, tmp_path):
    got = results(dev)
    for i, (s, C) in enumerate(zip(SHAPES + SHAPES32, got)):
        dtype = torch.float64 if i < len(SHAPES) else torch.float32
        j = i if i < len(SHAPES) else i - len(SHAPES)
        oa, ob, m, n, k = s[:5]
        bufs = product(dev, dtype, j, oa, ob, m, n, k, *(s[5:7] if dtype == torch.float64 else ()))
        a, b, c0 = [t.as_strided((r, c), (1, ld)).cpu().numpy().astype(np.float64)
                    for (t, _), (r, c, ld) in zip(bufs, geometry(oa, ob, m, n, k, 2 if dtype == torch.float64 else 4))]
        c = C.as_strided((m, n), (1, bufs[2][1])).cpu().numpy().astype(np.float64)
        a, b = a if oa == "N" else a.T, b if ob == "N" else b.T
        ref = 1.5 * (a @ b) - 0.5 * c0
        if dtype == torch.float64:
            assert np.linalg.norm(c - ref) <= 1e-13 * np.linalg.norm(ref), s
        else:
            assert np.all(np.abs(c - ref) <= 2.0 ** -24 * (k + 2) * (1.5 * np.abs(a) @ np.abs(b) + 0.5 * np.abs(c0))), s
    for e, extra in enumerate(RUNS):
        path = str(tmp_path / str(e))
        env = {k: v for k, v in os.environ.items() if not k.startswith("DG_GEMM_")}
        r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__), path], timeout=60, env=dict(env, **extra),
                           capture_output=True, text=True)
        assert r.returncode == 0, (extra, r.stdout[-500:], r.stderr[-2000:])
        for i, (mine, other) in enumerate(zip(got, torch.load(path, weights_only=True))):
            whole = torch.int64 if mine.dtype == torch.float64 else torch.int32
            assert torch.equal(mine.cpu().view(whole), other.view(whole)), (extra, i)


if __name__ == "__main__":
    torch.save([x.cpu() for x in results(torch.device("cuda"))], sys.argv[1])
