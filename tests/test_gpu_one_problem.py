"""A single problem goes to the kernel by value, a batch through descriptor
tables: the same bits either way, for every op pair, tile size and edge."""
import pytest
import torch

import dgamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("opA,opB", [("N", "N"), ("N", "T"), ("T", "N"), ("T", "T")])
@pytest.mark.parametrize("m,n,k,pad", [(1, 1, 1, 0), (31, 33, 15, 1), (512, 512, 512, 0), (700, 900, 301, 1),
                                       (1300, 1290, 128, 0), (3001, 2900, 33, 3)])
def test_by_value_matches_batch(dev, opA, opB, m, n, k, pad):
    def matrix(rows, cols, seed):
        t = torch.empty((rows + pad) * cols, dtype=torch.float64, device=dev)
        dgamd.generate_t(seed, dgamd.DG_DIST_WIDE, t)
        return t, rows + pad

    A, lda = matrix(*((m, k) if opA == "N" else (k, m)), 11)
    B, ldb = matrix(*((k, n) if opB == "N" else (n, k)), 12)
    C0, ldc = matrix(m, n, 13)
    one, batch, other = C0.clone(), C0.clone(), C0.clone()
    dgamd.dgemm_t(opA, opB, m, n, k, 1.5, A, lda, B, ldb, -0.5, one, ldc)
    # a second problem keeps the batch on the tables
    plan = dgamd.GroupedPlan([dgamd.gemm_desc(opA, opB, m, n, k, 1.5, A, lda, B, ldb, -0.5, batch, ldc),
                              dgamd.gemm_desc(opA, opB, m, n, k, 1.5, A, lda, B, ldb, -0.5, other, ldc)],
                             dgamd.DG_PLAN_NONPERSISTENT)
    plan.execute()
    torch.cuda.synchronize()
    plan.close()
    assert torch.equal(one, batch) and torch.equal(one, other)
    graph, side = torch.cuda.CUDAGraph(), C0.clone()
    dgamd.dgemm_t(opA, opB, m, n, k, 1.5, A, lda, B, ldb, -0.5, side, ldc)  # tables resident where there are any
    with torch.cuda.graph(graph):
        dgamd.dgemm_t(opA, opB, m, n, k, 1.5, A, lda, B, ldb, -0.5, side, ldc)
    for _ in range(3):
        side.copy_(C0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(side, one)
