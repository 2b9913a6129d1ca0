"""An S too large for the iteration.  With all elements positive every product
sums terms of one sign, so the iterates overflow to infinities, never to NaN: A
and A' have opposite signs, the residual is infinite, and the loop runs into its
limit, at every size (n is padded to a multiple of 16 inside)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd import _lib  # noqa: E402
from openatom_amd._lib import OrthoNotConverged  # noqa: E402
from openatom_amd.ortho import Batch  # noqa: E402

DEV = "cuda"
MAXIT = 20  # the cubes of the iterates overflow within eight


def positive(n):
    X = np.random.default_rng(n).random((n, n))
    return torch.from_numpy(10.0 * np.eye(n) + X + X.T).to(DEV)


@pytest.mark.parametrize("n", [1, 2, 5, 15, 16, 17, 33, 48, 100, 300])
def test_overflow_ends_at_the_limit(handle, n):
    S = positive(n)
    T = torch.zeros_like(S)
    with pytest.raises(OrthoNotConverged):
        handle.s_to_t(S, nspin=2, tol=1e-12, maxit=MAXIT, T=T)
    assert (handle.last_iterations, handle.last_error) == (MAXIT, float("inf"))
    assert bool(torch.isinf(T).all())
    rep = torch.zeros(24, dtype=torch.uint8, device=DEV)
    handle.s_to_t_async(S, T, rep, nspin=2, tol=1e-12, maxit=MAXIT)
    torch.cuda.synchronize()
    r = _lib.oa_ns_report.from_buffer_copy(bytes(rep.cpu().numpy()))
    assert (r.iterations, r.done, r.status) == (MAXIT, 1, _lib.OA_ERR_NOT_CONVERGED)


@pytest.mark.parametrize("wm", [2, 4])
def test_overflow_in_a_batch(handle, wm):
    """Rows of which the first component is large and positive: S is positive."""
    psis = []
    for n in (5, 17, 100):
        p = torch.full((n, 400), 0.25, dtype=torch.float64, device=DEV)
        p[:, 2:2 + n] += 2.0 * torch.eye(n, dtype=torch.float64, device=DEV)
        psis.append(p)
    b = Batch(handle)
    b.set_table("".join(f"{(p.shape[0] + 31) // 32} 128 {wm}\n" for p in psis))
    b.plan(psis, nkx0=1, nspin=2, tol=1e-12, maxit=MAXIT, prec="fp64")
    b.run()
    for i, r in enumerate(b.reports()):
        assert r[0] == MAXIT and r[2] == _lib.OA_ERR_NOT_CONVERGED, (i, r)
        assert bool(torch.isinf(b.T[i]).all()), i
    b.close()
