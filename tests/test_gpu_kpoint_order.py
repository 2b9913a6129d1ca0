"""The complex FP64 back-multiply sums its two real products in one order whichever
tile computes an element and however its operands are loaded: a column block has
the bits it has in the whole product, and so has a psi whose leading dimension
rules out 16-byte loads."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


# n: every remainder of the 16 column stages that a 32 or 64 tile groups by four
# or two, with and without a part of a stage
@pytest.mark.parametrize("trans", [False, True])
@pytest.mark.parametrize("n", [3, 16, 24, 40, 48, 80, 100, 112, 150, 200, 300])
def test_slices_and_odd_leading_dimensions(handle, n, trans):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n)
    npw = 6000
    psi = torch.randn((n, 2 * npw), generator=gen, dtype=torch.float64, device=DEV)
    M = torch.complex(torch.randn((n, n), generator=gen, dtype=torch.float64, device=DEV),
                      torch.randn((n, n), generator=gen, dtype=torch.float64, device=DEV))
    full = handle.zbackmul(M, psi, transM=trans)
    odd = torch.empty((n, 2 * npw + 1), dtype=torch.float64, device=DEV)[:, :2 * npw]
    odd.copy_(psi)
    for cols in (2, 64, 1000, 4000, 2 * npw):
        part = handle.zbackmul(M, psi[:, :cols], transM=trans,
                               out=torch.empty((n, cols), dtype=torch.float64, device=DEV))
        slow = handle.zbackmul(M, odd[:, :cols], transM=trans,
                               out=torch.empty((n, cols), dtype=torch.float64, device=DEV))
        torch.cuda.synchronize()
        assert torch.equal(part, full[:, :cols]), cols
        assert torch.equal(slow, full[:, :cols]), cols
