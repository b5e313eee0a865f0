"""The register-staged FP64 GEMM's loads (gemm_f64.hip, Staged) on the CPU:
for every tile shape and ragged operands at any leading dimension, every
element that any thread loads lies inside the operand (between its first and
its last element: a pair may take the padding between columns), and every
element of a tile's stage that is inside the operand arrives at its own
place, with zeros past the last k."""
import numpy as np
import pytest

# (rows of the operand's tile, k of a stage): the shapes the kernel is built with
SHAPES = [(128, 16), (64, 16), (32, 16), (32, 32)]
ZERO = -1


def stages(ROWS, BK, rows, ld, klen, row0, kc):
    """(first k, tile rows, k within the stage, offsets loaded, offsets stored) for the two elements of every pair."""
    t = np.arange(256)
    CH, HP = BK // 2, ROWS // 2
    for s in range((klen + BK - 1) // BK):
        left = klen - s * BK
        for q in range(ROWS * BK // 512):
            row = t // CH + 256 // CH * q if kc else 2 * (t % HP)
            kk = 2 * (t % CH) if kc else t // HP + 256 // HP * q
            r = np.minimum(row0 + row, rows - 1)
            at = lambda r_, k_: r_ * ld + k_ + s * BK if kc else r_ + (k_ + s * BK) * ld
            if left > BK:  # read
                x = at(r, kk)
                y = x + 1
                yield s, row, kk, (x, y), x, y
            else:          # read_last
                k = np.minimum(kk, left - 1)
                x = at(r, k)
                y = x + np.where((k + 1 < left) if kc else (r + 1 < rows), 1, 0)
                yield s, row, kk, (x, y), np.where(kk < left, x, ZERO), np.where((kk + 1 if kc else kk) < left, y, ZERO)


@pytest.mark.parametrize("ROWS,BK", SHAPES)
@pytest.mark.parametrize("kc", [True, False])
def test_loads_inside_and_at_their_places(ROWS, BK, kc):
    for rows in (1, 2, 3, 31, 32, 33, 65, 127, 128, 129, 200):
        for klen in (1, 2, 3, 15, 16, 17, 31, 32, 33, 50):
            for ld in ((klen if kc else rows), (klen if kc else rows) + 1):
                ns = (klen + BK - 1) // BK
                end = (rows - 1) * ld + klen if kc else rows + (klen - 1) * ld
                for row0 in range(0, rows, ROWS):
                    got = np.full((ROWS, ns * BK), -2, np.int64)
                    for s, row, k, loaded, x, y in stages(ROWS, BK, rows, ld, klen, row0, kc):
                        assert all(np.all((e >= 0) & (e < end)) for e in loaded)
                        got[row, s * BK + k] = x
                        got[row + (0 if kc else 1), s * BK + k + (1 if kc else 0)] = y
                    inside = min(ROWS, rows - row0)
                    r, kk = np.meshgrid(np.arange(inside), np.arange(klen), indexing="ij")
                    assert np.array_equal(got[:inside, :klen], (row0 + r) * ld + kk if kc else row0 + r + kk * ld)
                    assert np.all(got[:inside, klen:] == ZERO)
