"""The register-staged GEMMs' loads (staged.hpp, Staged) on the CPU:
for every tile shape and ragged operands at any leading dimension, every
element that any thread loads lies inside the operand (between its first and
its last element: a pair may take the padding between columns), and every
element of a tile's stage that is inside the operand arrives at its own
place, with zeros past the last k."""
import numpy as np
import pytest

# (rows of the operand's tile, k of a stage) the kernels are built with
SHAPES = {2: [(128, 16), (64, 16), (32, 32)], 4: [(64, 32), (32, 64)]}  # by elements of a 16-byte load: FP64, FP32
ZERO = -1


def stages(E, ROWS, BK, rows, ld, klen, row0, kc, last):
    """(stage, tile rows, k within it, offsets loaded, offsets stored) for element e of every run."""
    t = np.arange(256)
    CH, HP = BK // E, ROWS // E
    for s in range((klen + BK - 1) // BK):
        left = klen - s * BK
        for q in range(ROWS * BK // (256 * E)):
            row = t // CH + 256 // CH * q if kc else E * (t % HP)
            kk = E * (t % CH) if kc else t // HP + 256 // HP * q
            for e in range(E):
                er, ek = (0, e) if kc else (e, 0)
                at = lambda r, k: r * ld + k + s * BK if kc else r + (k + s * BK) * ld
                if left >= BK + last:  # read
                    x = at(np.minimum(row0 + row, rows - 1), kk) + e
                    yield s, row + er, kk + ek, x, x
                else:                  # read_last
                    x = at(np.minimum(row0 + row + er, rows - 1), np.minimum(kk + ek, left - 1))
                    yield s, row + er, kk + ek, x, np.where(kk + ek < left, x, ZERO)


@pytest.mark.parametrize("E,ROWS,BK", [(E, *x) for E, v in SHAPES.items() for x in v])
@pytest.mark.parametrize("kc", [True, False])
def test_loads_inside_and_at_their_places(E, ROWS, BK, kc):
    for rows in (1, 2, 3, 31, 32, 33, 65, 127, 128, 129, 200):
        for klen in (1, 2, 3, 15, 16, 17, 31, 32, 33, 50, 64, 65, 130):
            for ld in ((klen if kc else rows), (klen if kc else rows) + 1):
                if not kc and ld < E - 1:
                    continue  # loaded by elements
                ns = (klen + BK - 1) // BK
                end = (rows - 1) * ld + klen if kc else rows + (klen - 1) * ld
                for row0 in range(0, rows, ROWS):
                    inside = min(ROWS, rows - row0)
                    got = np.full((ROWS, ns * BK), -2, np.int64)
                    for s, row, k, loaded, stored in stages(E, ROWS, BK, rows, ld, klen, row0, kc,
                                                            0 if kc or inside == ROWS else 1):
                        assert np.all((loaded >= 0) & (loaded < end))
                        got[row, s * BK + k] = stored
                    r, kk = np.meshgrid(np.arange(inside), np.arange(klen), indexing="ij")
                    assert np.array_equal(got[:inside, :klen], (row0 + r) * ld + kk if kc else row0 + r + kk * ld)
                    assert np.all(got[:inside, klen:] == ZERO)
