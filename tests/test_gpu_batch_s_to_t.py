"""S->T of many uneven instances in joint launches.  Instances end at different
iterations, so in most launches some end while their other workgroups start and
others go on; each must still take the single call's iterations and give its
bits."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

from openatom_amd.ortho import Batch  # noqa: E402
from openatom_amd.workload import make_states  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("tile,wm", [(128, 2), (128, 4)])
def test_uneven_ends(handle, tile, wm):
    rng = np.random.default_rng(12)
    ns = rng.choice(np.arange(64, 513, 32), size=48)
    eps = 10.0 ** rng.uniform(-4, -2, size=48)
    psis = [make_states(int(n), 1024, eps=float(e), seed=i, device=DEV, rng="torch")
            for i, (n, e) in enumerate(zip(ns, eps))]
    refs = [handle.ortho_step(p, nkx0=1, nspin=2, tol=1e-12, maxit=12, prec="fp64")
            for p in psis]
    b = Batch(handle)
    b.set_table("".join(f"{k} {tile} {wm}\n" for k in sorted({(int(n) + 31) // 32 for n in ns})))
    b.plan(psis, nkx0=1, nspin=2, tol=1e-12, maxit=12, prec="fp64")
    for rep in range(4):
        b.run()
        reports = b.reports()
        for i, (S, T, out, it, _) in enumerate(refs):
            assert reports[i][0] == it, (rep, i, int(ns[i]), reports[i], it)
            assert torch.equal(b.T[i], T) and torch.equal(b.outs[i], out), (rep, i, int(ns[i]))
    b.close()
