"""S and T in shared memory: T is first written after every S has been read, in a
batch after the S of all instances, so T may lie over any S.  Bits of the calls
with buffers of their own."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd.ortho import Batch  # noqa: E402
from openatom_amd.workload import make_kpoint_states, make_states  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("prec", ["fp64", "int8x6a"])
@pytest.mark.parametrize("maxit", [1, 12])
def test_T_over_another_instances_S(handle, prec, maxit):
    """T of 0 and 1 over S of each other, of 2 and 3 inside the larger S of 4."""
    sizes = [(128, 4096), (128, 3000), (65, 2000), (96, 1500), (300, 2048)]
    psis = [make_states(n, k, eps=1e-3, seed=i, device=DEV, rng="torch")
            for i, (n, k) in enumerate(sizes)]
    plan = dict(nkx0=1, nspin=2, tol=1e-12, maxit=maxit, prec=prec)
    ref = Batch(handle)
    ref.plan(psis, **plan)
    ref.run()
    S = [torch.empty((n, n), dtype=torch.float64, device=DEV) for n, _ in sizes]
    inner = S[4].view(-1)
    T = [S[1], S[0], inner[:65 * 65].view(65, 65), inner[-96 * 96:].view(96, 96),
         torch.empty((300, 300), dtype=torch.float64, device=DEV)]
    b = Batch(handle)
    b.plan(psis, S=S, T=T, **plan)
    b.run()
    torch.cuda.synchronize()
    assert b.reports() == ref.reports()
    for i in range(len(sizes)):
        assert torch.equal(b.T[i], ref.T[i]), i
        assert torch.equal(b.outs[i], ref.outs[i]), i
    ref.close()
    b.close()


@pytest.mark.parametrize("n", [5, 64, 300, 600])
@pytest.mark.parametrize("shift", [0, 1, 3])
def test_T_over_S_shifted(handle, n, shift):
    psi = make_states(n, 2 * n, eps=1e-3, seed=n, device=DEV, rng="torch")
    S = handle.overlap_sym(psi)
    want = handle.s_to_t(S, nspin=2, tol=1e-12, maxit=30)
    buf = torch.empty(n * n + shift * n, dtype=torch.float64, device=DEV)
    src, dst = buf[:n * n].view(n, n), buf[shift * n:].view(n, n)
    src.copy_(S)
    torch.cuda.synchronize()
    got = handle.s_to_t(src, nspin=2, tol=1e-12, maxit=30, T=dst)
    assert torch.equal(got[0], want[0]) and got[1:] == want[1:]


@pytest.mark.parametrize("n", [16, 100])
def test_complex_first_iterate(handle, n):
    S = handle.zoverlap(make_kpoint_states(n, 2 * n, eps=1e-3, seed=n, device=DEV, rng="torch"))
    want = handle.zs_to_t(S, nspin=2, tol=1e-12, maxit=1, raise_on_limit=False)
    # one iteration: T = (3 I - S) / 2, stored by the second launch
    eye = torch.eye(n, dtype=torch.complex128, device=DEV)
    assert torch.equal(want[0], 0.5 * (3.0 * eye - S))
