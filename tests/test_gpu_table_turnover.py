"""The descriptor-table cache past its limits, in a fresh process: the first
128 tables of a device stay (large ones aside), the next 256 stay beside them,
and beyond those the least recently used make room, but for what a graph was
captured with.  Whether a table is resident shows under capture: a call whose
table is not is refused there.  Every call is checked bit for bit (its alpha is
a power of two), and every graph is replayed after the turnover."""
import os
import subprocess
import sys

import pytest
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "distributed-gemm-thesis_amd"))
import dgamd  # noqa: E402

pytestmark = pytest.mark.gpu

N = 48


class Calls:
    """Distinct tables of one kind of call: two problems, C = 2^e A B."""

    def __init__(self, dev):
        f64 = dict(dtype=torch.float64, device=dev)
        self.A, self.B = torch.empty(N * N, **f64), torch.empty(N * N, **f64)
        dgamd.generate_t(5, dgamd.DG_DIST_UNIFORM_PM1, self.A)
        dgamd.generate_t(6, dgamd.DG_DIST_UNIFORM_PM1, self.B)
        self.out = torch.empty((1000, 2, N * N), **f64)
        self.ref = torch.empty(N * N, **f64)
        dgamd.dgemm_t("N", "N", N, N, N, 1.0, self.A, N, self.B, N, 0.0, self.ref, N)

    def scale(self, i):
        return 2.0 ** (i % 200 - 100)

    def __call__(self, i):
        dgamd.grouped_dgemm_t([dgamd.gemm_desc("N", "N", N, N, N, self.scale(i), self.A, N, self.B, N, 0.0, C, N)
                               for C in self.out[i]])

    def right(self, i):
        return all(torch.equal(C, self.ref * self.scale(i)) for C in self.out[i])

    def capture(self, call, clear):
        """The graph of one call, or None where its table is not resident."""
        g, refused = torch.cuda.CUDAGraph(), False
        torch.cuda.synchronize()
        with torch.cuda.graph(g):
            clear.zero_()
            try:
                call()
            except dgamd.DGError as e:
                assert "not resident" in str(e)
                refused = True
        return None if refused else g

    def resident(self, i):
        return self.capture(lambda: self(i), self.out[i])


def run(dev):
    # a batch whose problem table is larger than 64 KiB, before anything else
    small = torch.zeros((1500, 16), dtype=torch.float64, device=dev)
    x = torch.ones(16, dtype=torch.float64, device=dev)
    large = lambda: dgamd.grouped_dgemm_t([dgamd.gemm_desc("N", "N", 4, 4, 4, 1.0, x, 4, x, 4, 0.0, c, 4) for c in small])
    large()
    assert torch.equal(small, torch.full_like(small, 4.0))
    calls = Calls(dev)
    first = calls.capture(lambda: calls(0), calls.out[0])  # not yet resident
    assert first is None
    graphs = {}
    for i in range(140):   # fills the kept tables and takes a dozen others
        calls(i)
    torch.cuda.synchronize()
    graphs[0] = calls.resident(0)
    graphs[100] = calls.resident(100)
    print("140 tables", flush=True)
    for i in range(200, 400):
        calls(i)
        if i % 50 == 49:
            torch.cuda.synchronize()
    torch.cuda.synchronize()
    assert all(calls.right(i) for i in list(range(140)) + list(range(200, 400)))
    for i in range(200, 400, 9):  # beside the kept tables there is room for 256
        graphs[i] = calls.resident(i)
        assert graphs[i] is not None, i
    print("340 tables", flush=True)
    for i in range(400, 800):
        calls(i)
        if i % 50 == 49:
            torch.cuda.synchronize()  # earlier uses complete: their tables may make room
    torch.cuda.synchronize()
    assert all(calls.right(i) for i in range(400, 800))
    print("740 tables", flush=True)
    assert calls.resident(50) is not None      # one of the first
    assert calls.resident(799) is not None     # one of the last
    assert calls.resident(139) is None and calls.resident(201) is None   # made room
    assert calls.capture(large, small) is None
    for rep in range(3):
        for i, g in graphs.items():
            calls.out[i].fill_(float("nan"))
            g.replay()
            torch.cuda.synchronize()
            assert calls.right(i), (rep, i)
        calls(139)  # a table that made room, made anew
        torch.cuda.synchronize()
        assert calls.right(139)
    print("turnover: ok", flush=True)


def test_kept_pool_and_captured_tables(dev):
    r = subprocess.run([sys.executable, "-u", os.path.abspath(__file__)], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, (r.stdout[-2000:], r.stderr[-3000:])
    assert "turnover: ok" in r.stdout


if __name__ == "__main__":
    run(torch.device("cuda"))
