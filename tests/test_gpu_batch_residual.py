"""The residual that ends S->T is summed in one order whatever the tile of the
launch: a batch reports the single call's error to the last bit, in either GEMM
tile, and so does the asynchronous form."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd import _lib  # noqa: E402
from openatom_amd.ortho import Batch  # noqa: E402
from openatom_amd.workload import make_states  # noqa: E402

DEV = "cuda"
# either side of the 16-row padding, of the 32-row blocks and of the single
# call's change from 32 to 64 tiles
SIZES = [1, 15, 16, 17, 31, 32, 33, 48, 64, 100, 128, 200, 300, 448, 512, 560, 577, 640, 777, 1000]


@pytest.mark.parametrize("wm", [2, 4])
@pytest.mark.parametrize("maxit", [2, 3, 12])
def test_error_of_the_single_call(handle, wm, maxit):
    psis = [make_states(n, 1024, eps=0.02, seed=n, device=DEV, rng="torch") for n in SIZES]
    b = Batch(handle)
    b.set_table("".join(f"{k} 128 {wm}\n" for k in sorted({(n + 31) // 32 for n in SIZES})))
    b.plan(psis, nkx0=1, nspin=2, tol=1e-12, maxit=maxit, prec="fp64")
    b.run()
    reports = b.reports()
    for i, n in enumerate(SIZES):
        rep = torch.zeros(24, dtype=torch.uint8, device=DEV)
        handle.s_to_t_async(b.S[i], torch.empty_like(b.S[i]), rep, nspin=2, tol=1e-12,
                            maxit=maxit)
        torch.cuda.synchronize()
        r = _lib.oa_ns_report.from_buffer_copy(bytes(rep.cpu().numpy()))
        assert reports[i] == (r.iterations, r.done, r.status, r.error), n
    b.close()


@pytest.mark.parametrize("n", [16, 100, 300, 640])
def test_error_of_the_first_step(handle, n):
    """The error itself, after one and after two iterations, against numpy; the
    iterates differ by at most 32 n eps an element, and so does their root mean
    square."""
    g = np.random.default_rng(n)
    X = g.standard_normal((n, n)) * (0.1 / np.sqrt(n))
    S = np.eye(n) + 0.5 * (X + X.T)
    A, B = np.eye(n), S
    for maxit in (1, 2):
        C = 3.0 * np.eye(n) - A @ B
        B, A0 = 0.5 * (B @ C), A
        A = 0.5 * (C @ A)
        want = np.sqrt(((A - A0) ** 2).sum() / n ** 2)
        try:
            handle.s_to_t(torch.from_numpy(S).to(DEV), nspin=2, tol=1e-300, maxit=maxit)
        except _lib.OrthoNotConverged:
            pass
        assert handle.last_iterations == maxit
        assert abs(handle.last_error - want) <= 32 * n * 2.0 ** -52
