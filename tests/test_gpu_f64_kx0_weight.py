"""The weight 1/2 of a narrow kx = 0 plane in the FP64 overlap.  The plane's product
may exceed the rest by any factor (a state that lives on G = 0), so it must enter
at half from the start: S = alpha (0.5 g + s) with one rounding of the sum, an
infinity in the plane stays one, and errors are relative to the weighted
magnitudes."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd import _lib  # noqa: E402
from openatom_amd.ortho import Batch  # noqa: E402

DEV = "cuda"
EPS = 2.0 ** -52

# (n, npw, nkx0): less than a stage, 64 tiles, ragged, 128 tiles (whole, diagonal)
SHAPES = [(5, 6, 6), (3, 500, 1), (40, 700, 8), (100, 3001, 16), (200, 3000, 9), (300, 9000, 1),
          (512, 9000, 16), (520, 2000, 3)]


def overlaps(handle, psi, nkx0):
    """S by the single call, a batch and the step without allocation."""
    n, K = psi.shape
    out = {"single": handle.overlap_sym(psi, nkx0=nkx0, alpha=2.0)}
    if psi.stride(0) == K:
        b = Batch(handle)
        b.plan([psi, psi], nkx0=nkx0, nspin=2, tol=1e-12, maxit=2, prec="fp64")
        b.run()
        out["batch"] = b.S[1].clone()
        torch.cuda.synchronize()
        b.close()
        S, T, o = torch.empty_like(out["single"]), torch.empty_like(out["single"]), psi.clone()
        torch.cuda.synchronize()
        st = _lib.lib().oa_ortho_step_noalloc(
            handle.h, n, K // 2, psi.data_ptr(), K, nkx0, 2, 1e-12, 2, 0, S.data_ptr(),
            T.data_ptr(), o.data_ptr(), K, None, None)
        assert st == 0
        out["noalloc"] = S
    torch.cuda.synchronize()
    return out


def states(n, npw, pad):
    buf = torch.full((n, 2 * npw + pad), float("nan"), dtype=torch.float64, device=DEV)
    return buf[:, :2 * npw]


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("n,npw,nkx0", SHAPES)
def test_exact_when_the_plane_dominates(handle, n, npw, nkx0, pad):
    psi = states(n, npw + 4, pad)
    K = psi.shape[1]
    psi.zero_()
    psi[:, 2 * nkx0 - 1] = 2.0 ** 27
    r = 1 + torch.arange(n, device=DEV) % 2
    psi[:, K - 1] = r.double()
    want = 2.0 * (2 ** 53 + r[:, None] * r[None, :]).double()  # rounds ties to even, as a sum does
    for name, S in overlaps(handle, psi, nkx0).items():
        assert torch.equal(S, want), name


@pytest.mark.parametrize("n,npw,nkx0", SHAPES)
def test_infinity_in_the_plane(handle, n, npw, nkx0):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n)
    psi = states(n, npw + 4, 0)
    psi.copy_(torch.randn(psi.shape, generator=gen, dtype=torch.float64, device=DEV))
    psi[1, 0] = float("inf")
    sign = torch.sign(psi[:, 0])
    for name, S in overlaps(handle, psi, nkx0).items():
        assert torch.equal(S[1], sign * float("inf")), name
        assert torch.equal(S[:, 1], sign * float("inf")), name
        rest = [i for i in range(n) if i != 1]
        assert bool(torch.isfinite(S[rest][:, rest]).all()), name


@pytest.mark.parametrize("pad", [0, 1])
@pytest.mark.parametrize("n,npw,nkx0", SHAPES)
def test_weighted_bound(handle, n, npw, nkx0, pad):
    """K products of weighted magnitude, each rounded at most K + 8 times."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n + nkx0)
    psi = states(n, npw + 4, pad)
    K = psi.shape[1]
    psi.copy_(torch.randn((n, K), generator=gen, dtype=torch.float64, device=DEV))
    psi[:, :2 * nkx0] *= 1e3
    w = torch.full((K,), 2.0, dtype=torch.float64, device=DEV)
    w[:2 * nkx0] = 1.0
    want = (psi * w) @ psi.T
    bound = (K + 8) * EPS * ((psi.abs() * w) @ psi.abs().T)
    for name, S in overlaps(handle, psi, nkx0).items():
        assert bool(((S - want).abs() <= bound).all()), name
        assert torch.equal(S, S.T), name
