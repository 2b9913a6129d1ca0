"""The FP64-MFMA kernels at the edges of their tiles: every tile configuration
of the GEMM (chosen by the number of 128 and 64 tiles), both layouts of both
operands, remainders of rows, columns and contraction, leading dimensions and
pointers that rule out the 16-byte direct-to-LDS loads, and the partial and
diagonal tiles of the split-K products.

Reference: torch's FP64 product.  Each side sums k terms in some order, each
rounding by at most eps / 2 of a partial sum of |a||b|, so the two differ by at
most (k + 4) eps (|A||B|) elementwise (4 for the scaling by alpha and beta).
The padding between and after the rows is NaN: an access that leaked it would
show in the result."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd.workload import make_states  # noqa: E402

DEV = "cuda"
EPS = 2.0 ** -52


def padded(rows, cols, pad, off, gen):
    """A (rows, cols) view with leading dimension cols + pad at element offset
    `off` of a NaN-filled buffer, filled with normal values."""
    ld = cols + pad
    buf = torch.full((off + rows * ld + 8,), float("nan"), dtype=torch.float64, device=DEV)
    v = buf[off:off + rows * ld].view(rows, ld)[:, :cols]
    v.copy_(torch.randn((rows, cols), generator=gen, dtype=torch.float64, device=DEV))
    return buf, v, ld


# (m, n, k): T32 below 192 tiles of 64; T64W; T64 from 1024; T128 from 512 of 128
SHAPES = [(1, 1, 1), (17, 33, 5), (32, 32, 16), (70, 95, 64), (301, 300, 37), (1000, 900, 47),
          (64 * 260, 250, 30), (64 * 270 + 3, 130, 33), (33000, 301, 50), (32768, 257, 16),
          (33001, 255, 21)]


@pytest.mark.parametrize("pad,off", [(0, 0), (2, 0), (1, 0), (0, 1)])
@pytest.mark.parametrize("ta,tb", [("N", "N"), ("T", "N"), ("N", "T"), ("T", "T")])
@pytest.mark.parametrize("shape", SHAPES)
def test_gemm_tiles(handle, shape, ta, tb, pad, off):
    m, n, k = shape
    gen = torch.Generator(device=DEV)
    gen.manual_seed(m * 7 + n * 3 + k)
    # column-major op(A) [m][k]: the row-major view below is its transpose
    _, A, lda = padded(*((k, m) if ta == "N" else (m, k)), pad, off, gen)
    _, B, ldb = padded(*((n, k) if tb == "N" else (k, n)), pad, off, gen)
    cbuf, C, ldc = padded(n, m, pad, off, gen)
    At = (A if ta == "N" else A.T).T  # [m][k]
    Bt = (B if tb == "N" else B.T).T  # [k][n]
    alpha, beta = -0.75, 0.5
    want = (alpha * (At @ Bt) + beta * C.T).T
    bound = (k + 4) * EPS * (At.abs() @ Bt.abs() + C.T.abs()).T
    before = cbuf.clone()
    st = handle.dgemm(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc)
    assert st == 0
    torch.cuda.synchronize()
    assert bool(((C - want).abs() <= bound).all()), float(((C - want).abs() / bound).max())
    C.copy_(float("nan") * C)  # what lies outside C is untouched
    before[off:off + n * ldc].view(n, ldc)[:, :m] = float("nan")
    assert bool(((cbuf == before) | (cbuf.isnan() & before.isnan())).all())


@pytest.mark.parametrize("ldx", [0, 1, 2])
@pytest.mark.parametrize("n,npw", [(1, 3), (15, 40), (16, 129), (33, 1001), (64, 77), (129, 640),
                                   (255, 2049), (257, 1500), (300, 4097), (400, 333)])
def test_overlap_and_lambda_tiles(handle, n, npw, ldx):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n + npw)
    _, psi, _ = padded(n, 2 * npw, ldx, 0, gen)
    _, F, _ = padded(n, 2 * npw, ldx, 0, gen)
    S = handle.overlap_sym(psi, nkx0=1, alpha=2.0)
    L = handle.lambda_fwd(psi, F)
    torch.cuda.synchronize()
    w = torch.full((2 * npw,), 2.0, dtype=torch.float64, device=DEV)
    w[:2] = 1.0
    K = 2 * npw
    want = (psi * w) @ psi.T
    bound = (K + 8) * EPS * ((psi.abs() * w) @ psi.abs().T)
    assert bool(((S - want).abs() <= bound).all()), float(((S - want).abs() / bound).max())
    assert torch.equal(S, S.T)
    want, bound = psi @ F.T, (K + 8) * EPS * (psi.abs() @ F.abs().T)
    assert bool(((L - want).abs() <= bound).all()), float(((L - want).abs() / bound).max())


def test_tile_choice_keeps_the_sum_order(handle):
    """A column block of T psi has the same bits whichever tile computes it:
    the whole product (128 tiles), and slices of it small enough for each of
    the smaller tiles."""
    n, npw = 200, 40000
    psi = make_states(n, npw, seed=3, device=DEV, rng="torch")
    T = torch.eye(n, dtype=torch.float64, device=DEV) + 1e-3 * torch.randn(
        (n, n), dtype=torch.float64, device=DEV)
    full = handle.backmul(T, psi)
    for cols in (32, 1000, 4000, 24000):
        part = handle.backmul(T, psi[:, :cols])
        torch.cuda.synchronize()
        assert torch.equal(part, full[:, :cols]), cols


@pytest.mark.parametrize("n,npw,nkx0", [(40, 700, 0), (40, 700, 16), (40, 700, 17), (17, 90, 90),
                                        (130, 1501, 16), (301, 20011, 17), (301, 20011, 413),
                                        (300, 5000, 4999)])
def test_overlap_kx0_plane_and_maxdev(handle, n, npw, nkx0):
    """A kx = 0 plane of up to 32 columns comes off in the reduce, a wider one
    is a slice of its own; max|S - d I| from the reduce.  The subtraction adds
    one rounding of the half product to the bound."""
    gen = torch.Generator(device=DEV)
    gen.manual_seed(n + npw)
    psi = torch.randn((n, 2 * npw), generator=gen, dtype=torch.float64, device=DEV)
    md = torch.zeros(1, dtype=torch.float64, device=DEV)
    S = handle.overlap_sym(psi, nkx0=nkx0, alpha=2.0, diag=1.5, maxdev=md)
    torch.cuda.synchronize()
    w = torch.full((2 * npw,), 2.0, dtype=torch.float64, device=DEV)
    w[:2 * nkx0] = 1.0
    want = (psi * w) @ psi.T
    bound = (2 * npw + 10) * EPS * 2.0 * (psi.abs() @ psi.abs().T)
    assert bool(((S - want).abs() <= bound).all()), float(((S - want).abs() / bound).max())
    assert torch.equal(S, S.T)
    eye = torch.eye(n, dtype=torch.float64, device=DEV)
    assert float(md) == float((S - 1.5 * eye).abs().max())
