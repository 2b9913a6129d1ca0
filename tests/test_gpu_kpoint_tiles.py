"""The complex FP64 products and S->T at the edges of their tiles: the fused
back-multiply Re(M) psi + Im(M) J psi in every tile configuration, J applied
to operand fragments in the Hermitian and the general forward, odd n, leading
dimensions that rule out 16-byte loads, and the complex iteration's limits.

Reference: torch / numpy in complex128.  A part of a complex product of k terms
sums 2 k real products; two orders of summation differ by at most (2 k + 8) eps
times the sum of the products' magnitudes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd._lib import OrthoNotConverged  # noqa: E402

DEV = "cuda"
EPS = 2.0 ** -52


def block(n, npw, pad, gen):
    """[n][2 npw] doubles with leading dimension 2 npw + pad, NaN between."""
    buf = torch.full((n, 2 * npw + pad), float("nan"), dtype=torch.float64, device=DEV)
    v = buf[:, :2 * npw]
    v.copy_(torch.randn((n, 2 * npw), generator=gen, dtype=torch.float64, device=DEV))
    return v


def cplx(v):
    return torch.complex(v[:, 0::2].contiguous(), v[:, 1::2].contiguous())


def mag(z):
    return z.real.abs() + z.imag.abs()


def inside(got, want, bound):
    e = torch.maximum((got.real - want.real).abs(), (got.imag - want.imag).abs())
    return bool((e <= bound).all()), float((e / bound).max())


@pytest.mark.parametrize("pad", [0, 1, 2])
@pytest.mark.parametrize("n,npw", [(1, 1), (20, 31), (33, 600), (64, 9000), (100, 3001),
                                   (130, 20011), (257, 12345), (301, 4000), (512, 9000)])
def test_products(handle, n, npw, pad):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n + npw)
    psi, F, out = (block(n, npw, pad, gen) for _ in range(3))
    M = torch.complex(torch.randn((n, n), generator=gen, dtype=torch.float64, device=DEV),
                      torch.randn((n, n), generator=gen, dtype=torch.float64, device=DEV))
    P, Q = cplx(psi), cplx(F)
    for trans, beta in ((False, 0.0), (True, 0.5)):
        op = M.conj().T if trans else M
        o = out.clone() if beta == 0.0 else out
        want = -0.75 * (op @ P) + beta * cplx(out)
        bound = (2 * n + 8) * EPS * (mag(op) @ mag(P) + mag(cplx(out)))
        handle.zbackmul(M, psi, transM=trans, alpha=-0.75, beta=beta, out=o)
        torch.cuda.synchronize()
        ok, worst = inside(cplx(o), want, bound)
        assert ok, (trans, worst)
    S, L = handle.zoverlap(psi), handle.zlambda(psi, F)
    torch.cuda.synchronize()
    ok, worst = inside(S, P @ P.conj().T, (2 * npw + 8) * EPS * (mag(P) @ mag(P).T))
    assert ok, worst
    assert torch.equal(S, S.conj().T)
    ok, worst = inside(L, P @ Q.conj().T, (2 * npw + 8) * EPS * (mag(P) @ mag(Q).T))
    assert ok, worst


def iterate(S, nspin, tol, maxit, modulus):
    n = S.shape[0]
    A, B = np.eye(n, dtype=complex), (0.5 * S if nspin == 1 else S)
    for it in range(1, maxit + 1):
        C = 3.0 * np.eye(n) - A @ B
        B, A0 = 0.5 * (B @ C), A
        A = 0.5 * (C @ A)
        d = A - A0
        s = (np.abs(d) ** 2).sum() if modulus else (d.real ** 2).sum() - (d.imag ** 2).sum()
        err = np.sqrt(s / n ** 2) if s >= 0 else float("nan")
        if not (err > tol and it < maxit):
            break
    return A, it, err


@pytest.mark.parametrize("n", [1, 2, 15, 17, 33, 64, 101, 200, 300, 450])
@pytest.mark.parametrize("nspin,modulus", [(1, True), (2, True), (1, False)])
def test_s_to_t(handle, n, nspin, modulus):
    g = np.random.default_rng(n)
    X = g.standard_normal((n, n)) + 1j * g.standard_normal((n, n))
    S = (np.eye(n) + (0.05 / np.sqrt(n)) * (X + X.conj().T)) * (2.0 if nspin == 1 else 1.0)
    want, it, err = iterate(S, nspin, 1e-11, 40, modulus)
    Sd = torch.from_numpy(S).to(DEV)
    T, got, gerr = handle.zs_to_t(Sd, nspin=nspin, tol=1e-11, maxit=40, modulus=modulus)
    assert got == it and (np.isnan(gerr) and np.isnan(err) or abs(gerr - err) <= 64 * n * EPS)
    assert np.abs(T.cpu().numpy() - want).max() <= 64 * n * EPS
    # the limit, on both sides of the first look of the host loop (a scalar
    # iteration reaches its fixed point exactly and may end before it)
    for maxit in (1, 2, 4, 5, 6) if n > 2 else ():
        w, it, _ = iterate(S, nspin, 1e-300, maxit, True)
        with pytest.raises(OrthoNotConverged):
            handle.zs_to_t(Sd, nspin=nspin, tol=1e-300, maxit=maxit, modulus=True)
        assert handle.last_iterations == it == maxit
        T, _, _ = handle.zs_to_t(Sd, nspin=nspin, tol=1e-300, maxit=maxit, modulus=True,
                                 raise_on_limit=False)
        assert np.abs(T.cpu().numpy() - w).max() <= 64 * n * EPS


@pytest.mark.parametrize("bad", [complex(float("nan"), 0), complex(0, float("inf"))])
def test_non_finite_S(handle, bad):
    S = torch.eye(40, dtype=torch.complex128, device=DEV)
    S[3, 7] = bad
    T, it, err = handle.zs_to_t(S, nspin=2, tol=1e-12, maxit=30, modulus=True)
    assert it == 1 and np.isnan(err)
    t = T.cpu().numpy()
    keep = np.ones((40, 40), dtype=bool)
    keep[3, 7] = False
    assert np.isnan(t[keep].real).all() and np.isnan(t[keep].imag).all()
