"""The S->T iteration at the edges of its launches: sizes around the 16-row
padding and the tile choices, iteration limits on either side of the looks of
the host loop, the asynchronous form, S and T in one buffer, and non-finite S.

Reference: the iteration itself in numpy, FP64 (A = I, B = S/2 or S; C = 3I -
AB; B' = BC/2; A' = CA/2).  A product of two n x n matrices of norm at most 2
(B, and A, C near 2 I) is off by at most about n eps per element relative to
the norms; over the few iterations of a matrix near the fixed point, which
contracts errors, 32 n eps bounds the difference of the two T."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd import _lib  # noqa: E402
from openatom_amd._lib import OrthoNotConverged  # noqa: E402

DEV = "cuda"
EPS = 2.0 ** -52


def make_S(n, nspin, eps, seed):
    g = np.random.default_rng(seed)
    X = g.standard_normal((n, n)) * (eps / np.sqrt(n))
    S = np.eye(n) + 0.5 * (X + X.T)
    return S if nspin == 2 else 2.0 * S


def ref(S, nspin, tol, maxit):
    n = S.shape[0]
    A, B = np.eye(n), (S / 2.0 if nspin == 1 else S)
    for it in range(1, maxit + 1):
        C = 3.0 * np.eye(n) - A @ B
        B, A0 = 0.5 * (B @ C), A
        A = 0.5 * (C @ A)
        err = np.sqrt(((A - A0) ** 2).sum() / n ** 2)
        if not (err > tol and it < maxit):
            break
    return A, it, err


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 31, 33, 64, 65, 100, 191, 300, 448, 577, 777])
@pytest.mark.parametrize("nspin", [1, 2])
def test_matches_the_iteration(handle, n, nspin):
    for eps, tol in ((1e-2, 1e-12), (0.3, 1e-12)):
        S = make_S(n, nspin, eps, n)
        want, it, err = ref(S, nspin, tol, 50)
        T, got_it, got_err = handle.s_to_t(torch.from_numpy(S).to(DEV), nspin=nspin, tol=tol,
                                           maxit=50)
        assert got_it == it
        assert abs(got_err - err) <= 32 * n * EPS
        assert np.abs(T.cpu().numpy() - want).max() <= 32 * n * EPS


@pytest.mark.parametrize("n", [17, 130, 300])
@pytest.mark.parametrize("maxit", [1, 2, 3, 4, 5, 6, 7])
def test_limits_and_async(handle, n, maxit):
    """tol below reach: the loop runs into maxit; the asynchronous form gives
    the same bits and report."""
    S = make_S(n, 2, 0.2, 5)
    want, it, _ = ref(S, 2, 1e-300, maxit)
    Sd = torch.from_numpy(S).to(DEV)
    T = torch.full_like(Sd, float("nan"))
    with pytest.raises(OrthoNotConverged):
        handle.s_to_t(Sd, nspin=2, tol=1e-300, maxit=maxit, T=T)
    assert handle.last_iterations == maxit == it
    assert np.abs(T.cpu().numpy() - want).max() <= 32 * n * EPS
    T2 = torch.full_like(Sd, float("nan"))
    rep = torch.zeros(24, dtype=torch.uint8, device=DEV)
    handle.s_to_t_async(Sd, T2, rep, nspin=2, tol=1e-300, maxit=maxit)
    torch.cuda.synchronize()
    r = _lib.oa_ns_report.from_buffer_copy(bytes(rep.cpu().numpy()))
    assert (r.iterations, r.done, r.status) == (maxit, 1, _lib.OA_ERR_NOT_CONVERGED)
    assert r.error == handle.last_error
    assert torch.equal(T, T2)


def test_guarded_iterations_change_nothing(handle):
    """T and the report after convergence are those of the synchronous form,
    with iterations enqueued past it; S may be its own T."""
    S = make_S(96, 1, 1e-3, 1)
    Sd = torch.from_numpy(S).to(DEV)
    T, it, err = handle.s_to_t(Sd, nspin=1, tol=1e-12, maxit=100)
    rep = torch.zeros(24, dtype=torch.uint8, device=DEV)
    T2 = Sd.clone()
    handle.s_to_t_async(T2, T2, rep, nspin=1, tol=1e-12, maxit=12)
    torch.cuda.synchronize()
    r = _lib.oa_ns_report.from_buffer_copy(bytes(rep.cpu().numpy()))
    assert (r.iterations, r.done, r.status, r.error) == (it, 1, 0, err)
    assert torch.equal(T, T2)


@pytest.mark.parametrize("bad", [float("nan"), float("inf"), -float("inf")])
@pytest.mark.parametrize("n", [5, 40, 200])
def test_non_finite_S(handle, n, bad):
    """One non-finite element of S ends the loop after one iteration with a
    NaN error and an all-NaN T (I S multiplies it with zeros)."""
    S = make_S(n, 2, 1e-3, 2)
    S[1, 3] = bad
    T, it, err = handle.s_to_t(torch.from_numpy(S).to(DEV), nspin=2, tol=1e-12, maxit=50)
    assert it == 1 and np.isnan(err)
    t = T.cpu().numpy()
    keep = np.ones_like(t, dtype=bool)
    keep[1, 3] = False  # the identity leaves this one product an infinity
    assert np.isnan(t[keep]).all()
