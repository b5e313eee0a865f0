"""The layer reduction of an odd number of elements, on both sides of the
line between its forms (pairs; single elements for up to three layers of more
than 600 MB in all): the additions in layer order, bit for bit."""
import pytest
import torch

import dgamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("layers", [1, 3, 4])
@pytest.mark.parametrize("total", [75000000 - 20, 75000000 + 20])  # elements of C and the layers
def test_both_sides_of_the_line(dev, layers, total):
    n = total // (layers + 1) // 2 * 2 + 1
    C = torch.empty(n, dtype=torch.float64, device=dev)
    partial = torch.empty(n * layers, dtype=torch.float64, device=dev)
    dgamd.generate_t(7, dgamd.DG_DIST_WIDE, C)
    dgamd.generate_t(8, dgamd.DG_DIST_WIDE, partial)
    want = C.clone()
    for l in range(layers):
        want += partial[l * n: (l + 1) * n]
    dgamd.layer_reduce_t(C, partial, n, layers)
    torch.cuda.synchronize()
    assert torch.equal(C, want)
