"""The int8 back-multiply applies its scales, powers of two, as factors, or step by
step where one could leave the range of normal numbers.  Both must round alike:
scaling the operands by a power of two scales the result exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda"


def operands(n, npw):
    g = torch.Generator(device=DEV)
    g.manual_seed(11 * n + npw)
    psi = torch.randn((n, 2 * npw), generator=g, device=DEV, dtype=torch.float64) * 1e-2
    T = torch.eye(n, device=DEV, dtype=torch.float64) + 1e-3 * torch.randn(
        (n, n), generator=g, device=DEV, dtype=torch.float64)
    return T, psi


# exponents of T's and psi's factors and of alpha: each alone beyond the limits of
# the fast way (2^900 for a scale, 1e200 for a diagonal element, 1e30 for alpha)
@pytest.mark.parametrize("kt,kp,ka", [(0, -960, 0), (0, 960, 0), (930, 0, 0), (-930, 0, 0),
                                      (690, 0, 0), (-690, 0, 0), (0, 0, 130), (0, 0, -130)])
@pytest.mark.parametrize("prec", ["int8x4", "int8x6a", "int8x6l"])
def test_scales_round_alike(handle, kt, kp, ka, prec):
    for n, npw in ((40, 300), (200, 2048)):
        T, psi = operands(n, npw)
        ref = handle.backmul(T, psi, prec=prec)
        out = handle.backmul(T * 2.0 ** kt, psi * 2.0 ** kp, alpha=2.0 ** ka, prec=prec)
        assert torch.equal(out * 2.0 ** -(kt + kp + ka), ref), (n, npw)


@pytest.mark.parametrize("prec", ["int8x5", "int8x6a"])
def test_one_wild_row(handle, prec):
    """Rows of unlike size in one tile; the others keep their bits."""
    T, psi = operands(150, 1024)
    ref = handle.backmul(T, psi, prec=prec)
    T2 = T.clone()
    T2[70] *= 2.0 ** 920
    T2[3] *= 2.0 ** -920
    out = handle.backmul(T2, psi, prec=prec)
    assert torch.equal(out[70] * 2.0 ** -920, ref[70])
    assert torch.equal(out[3] * 2.0 ** 920, ref[3])
    keep = [i for i in range(150) if i not in (3, 70)]
    assert torch.equal(out[keep], ref[keep])
