"""Products whose leading dimension is millions of elements: on both sides of
each tile's limit for 32-bit lane offsets (whole runs below it, single
elements above it), the result has the bits of the same product with the
operand packed close, in FP64 and FP32, for the operand contiguous along k and
along its rows, even and odd leading dimensions.  FP32 also with rows so close
(leading dimension 1, 2) that runs would pass the matrix's end."""
import pytest
import torch

import dgamd

pytestmark = pytest.mark.gpu

BYTES = 12 << 30


@pytest.fixture(scope="module")
def buffer(dev):
    b = torch.empty(BYTES, dtype=torch.uint8, device=dev)
    yield b
    del b
    torch.cuda.empty_cache()


def operand(dev, dtype, rows, cols, seed):
    t = torch.empty(rows * cols, dtype=dtype, device=dev)
    dgamd.generate_t(seed, dgamd.DG_DIST_UNIFORM_PM1, t)
    return t


def same_bits(dev, dtype, oa, ob, m, n, k, far, ld, buf):
    """The product with operand `far` ('A' or 'B') at leading dimension ld against the packed one."""
    gemm = dgamd.dgemm_t if dtype == torch.float64 else dgamd.sgemm_t
    dims = {"A": (m, k) if oa == "N" else (k, m), "B": (k, n) if ob == "N" else (n, k)}
    x = {s: operand(dev, dtype, *dims[s], 40 + i) for i, s in enumerate("AB")}
    lds = {s: dims[s][0] for s in "AB"}
    C0 = operand(dev, dtype, m, n, 43)
    want, got = C0.clone(), C0.clone()
    gemm(oa, ob, m, n, k, 1.5, x["A"], lds["A"], x["B"], lds["B"], -0.5, want, m)
    rows, cols = dims[far]
    wide = buf.view(dtype)[: ld * (cols - 1) + rows]
    wide.as_strided((cols, rows), (ld, 1)).copy_(x[far].view(cols, rows))
    x[far], lds[far] = wide, ld
    print("long columns", dtype, oa, ob, m, n, k, far, ld, flush=True)
    gemm(oa, ob, m, n, k, 1.5, x["A"], lds["A"], x["B"], lds["B"], -0.5, got, m)
    whole = torch.int64 if dtype == torch.float64 else torch.int32
    assert torch.equal(got.view(whole), want.view(whole))


# apart: rows (k-contiguous) or k (row-contiguous) of a tile's stage, less one
@pytest.mark.parametrize("apart", [15, 31, 63, 127])
@pytest.mark.parametrize("oa,ob,far", [("T", "N", "A"), ("N", "N", "B"), ("N", "T", "A"), ("T", "T", "B")])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_limits_of_32_bit_offsets(dev, buffer, dtype, oa, ob, far, apart):
    size = torch.empty(0, dtype=dtype).element_size()
    limit = 2 ** 32 // (size * apart)  # elements between two rows (or k) that are `apart` rows from leaving 32 bits
    other = BYTES // (size * (limit + 2)) - 1  # columns of the far operand that the buffer holds
    assert other >= 33
    for ld in (limit - 130, limit + 1, limit + 2):
        if (oa == "T") if far == "A" else (ob == "N"):  # k along the column: its columns are rows of the product
            m, n, k = (min(other, 130), 70, 50) if far == "A" else (70, min(other, 130), 50)
        else:
            m, n, k = (130, 70, min(other, 50)) if far == "A" else (70, 130, min(other, 50))
        same_bits(dev, dtype, oa, ob, m, n, k, far, ld, buffer)


@pytest.mark.parametrize("oa,ob", [("N", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("ld", [1, 2, 3, 4])
def test_rows_closer_than_a_run(dev, buffer, oa, ob, ld):
    for m, n, k in ((1, 1, 40), (min(ld, 2), 70, 130), (70, min(ld, 2), 17)):
        far = "A" if oa == "N" and m <= ld else "B"
        if (far == "A" and m > ld) or (far == "B" and (n > ld or ob == "N")):
            continue
        same_bits(dev, torch.float32, oa, ob, m, n, k, far, ld, buffer)
