"""The workloads whose speed is followed: what programs of this package run,
through its public entry points, from the smallest calls to the largest.

  step      one orthonormalisation step of a state block, Handle.ortho_step:
            S, S -> T, T psi (the call of every MD or minimisation step)
  batch     one step of many independent instances, Batch.launch: path-integral
            beads, tempering replicas, the sessions of a serving loop
  dynamics  the Lambda round trip of Car-Parrinello dynamics: the asymmetric
            forward, Gamma = T Lambda, and the GSpace force from Psi and F
  kpoint    one complex-math step, Handle.zortho_step (k-points)

A case is a dict of plain values.  Sizes: n states of npw plane waves, nkx0 of
them on the kx = 0 plane.  nspin 1 (lda) takes states with S = 2 I, nspin 2
(lsda) states with S = I.
"""
import numpy as np
import torch

from openatom_amd.ortho import Batch, GSpacePlane, Ortho, PairCalculator, default_handle
from openatom_amd.workload import make_force, make_kpoint_states, make_states

DEV = "cuda"
TOL = 1e-12
MAXIT_SYNC = 100   # the host loop ends at the stop rule
MAXIT_ASYNC = 12   # guarded iterations of the asynchronous S -> T
SIZES = (128, 256, 512, 1024)      # serving sessions, npw = 64 n
WEIGHTS = (0.4, 0.3, 0.2, 0.1)
LARGEST = 1.6e12                   # FP64 operations of a drawn batch at most


def _step(name, n, npw, prec, nkx0=1, nspin=2, sync=True, eps=1e-3):
    return {"name": name, "kind": "step", "n": n, "npw": npw, "nkx0": nkx0, "nspin": nspin,
            "prec": prec, "sync": sync, "eps": eps}


def listed():
    return [
        # a molecule in a small box: the call is launches and latency
        _step("step 32x512 fp64", 32, 512, "fp64"),
        # 128 states, 8192 plane waves: the benchmark's small configuration
        _step("step 128x8192 fp64", 128, 8192, "fp64"),
        # a size no tile divides, lda
        _step("step 301x20011 fp64", 301, 20011, "fp64", nspin=1),
        # the benchmark's middle configuration, enqueued without waiting, as an
        # MD loop that keeps its states on the device does
        _step("step 512x65536 fp64", 512, 65536, "fp64", sync=False),
        # the benchmark's large configuration in the drop-in precision
        _step("step 1024x262144 fp64", 1024, 262144, "fp64"),
        # a ragged block on the uniform split with a whole kx = 0 plane
        _step("step 777x50021 int8x5", 777, 50021, "int8x5", nkx0=689, nspin=1),
        # the middle configuration on the adaptive split
        _step("step 512x65536 int8x6a", 512, 65536, "int8x6a", sync=False),
        # the benchmark's headline: the large configuration, adaptive split
        _step("step 1024x262144 int8x6a", 1024, 262144, "int8x6a"),
        # path-integral beads and replicas of uneven size in the drop-in
        # precision (n of 64..512, npw of 8192..65536)
        {"name": "batch 12 beads fp64", "kind": "batch", "mix": "beads", "count": 12,
         "pick": 1, "prec": "fp64"},
        # one iteration of the serving loop at its default precision
        {"name": "batch 10 sessions int8x6a", "kind": "batch", "mix": "sessions", "count": 10,
         "pick": 2, "prec": "int8x6a"},
        # the dynamics force path of a middling system
        {"name": "dynamics 384x40000 fp64", "kind": "dynamics", "n": 384, "npw": 40000,
         "nkx0": 585, "nspin": 2},
        # a k-point of a periodic cell
        {"name": "kpoint 256x32768 fp64", "kind": "kpoint", "n": 256, "npw": 32768, "nspin": 2,
         "prec": "fp64"},
    ]


def _log(rng, lo, hi):
    """A whole number spread over its logarithm."""
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["step"] * 5 + ["batch"] * 2 + ["dynamics", "kpoint"])
    if kind == "batch":
        c = {"kind": "batch", "mix": rng.choice(["beads", "sessions"]),
             "count": rng.randint(2, 14), "pick": rng.randrange(1 << 20),
             "prec": rng.choice(["fp64", "int8x6a"])}
        while work(c)["flops"] > LARGEST:
            c["count"] -= 1
        return c
    if kind == "dynamics":
        n = _log(rng, 24, 700)
        npw = max(n, _log(rng, 1000, 100000))
        return {"kind": "dynamics", "n": n, "npw": npw, "nkx0": int(npw ** (2.0 / 3.0) / 2),
                "nspin": rng.choice([1, 2])}
    if kind == "kpoint":
        n = _log(rng, 16, 512)
        return {"kind": "kpoint", "n": n, "npw": max(n, _log(rng, 600, 100000)), "nspin": 2,
                "prec": rng.choice(["fp64", "fp64", "int8x5"])}
    n = _log(rng, 16, 1024)
    npw = max(n, _log(rng, 500, 262144))
    prec = rng.choice(["fp64", "fp64", "int8x6a", "int8x6a", "int8x5"])
    nkx0 = 1 if prec == "fp64" else rng.choice([1, 1, int(npw ** (2.0 / 3.0) / 2)])
    c = _step("", n, npw, prec, nkx0=nkx0, nspin=rng.choice([1, 2]),
              sync=rng.random() < 0.6, eps=10.0 ** rng.uniform(-4.0, -2.0))
    del c["name"]
    return c


def _instances(case):
    """(n, npw, eps) of a batch's instances, from its `pick`."""
    g = np.random.default_rng(case["pick"])
    if case["mix"] == "sessions":
        ns = [int(n) for n in g.choice(SIZES, size=case["count"], p=WEIGHTS)]
        return [(n, 64 * n, 1e-3) for n in ns]
    ns = g.choice(np.arange(64, 513, 32), size=case["count"])
    npws = (g.integers(8192, 65536 + 1, size=case["count"]) // 256) * 256
    epss = 10.0 ** g.uniform(-4, -2, size=case["count"])
    return [(int(n), int(p), float(e)) for n, p, e in zip(ns, npws, epss)]


def _states(n, npw, eps, seed, nkx0, nspin):
    psi = make_states(n, npw, eps=eps, seed=seed, nkx0=nkx0, device=DEV, rng="torch")
    if nspin == 1:
        psi *= 2.0 ** 0.5
    return psi


def _dyn_inputs(case, seed):
    """(psi, F, T) as the PairCalculator receives them (the kx = 0 points
    rescaled for the Lambda forward), T a symmetric I + O(eps)."""
    n, npw, kx = case["n"], case["npw"], 2 * case["nkx0"]
    psi = _states(n, npw, 1e-3, seed, case["nkx0"], case["nspin"])
    F = make_force(n, npw, seed=seed + (1 << 20), device=DEV, rng="torch")
    psi[:, :kx] *= 0.5 ** 0.5
    F[:, :kx] *= 2.0 ** 0.5
    g = torch.Generator(device=DEV)
    g.manual_seed(seed + (2 << 20))
    X = torch.randn((n, n), generator=g, dtype=torch.float64, device=DEV)
    T = torch.eye(n, dtype=torch.float64, device=DEV) + (0.5e-3 / n ** 0.5) * (X + X.T)
    return psi, F, T


def prepare(case, seed):
    h = default_handle()
    kind = case["kind"]
    if kind == "step":
        return {"case": case, "h": h, "psi": _states(case["n"], case["npw"], case["eps"], seed,
                                                     case["nkx0"], case["nspin"])}
    if kind == "batch":
        psis = [_states(n, npw, eps, seed * 64 + i, 1, 2)
                for i, (n, npw, eps) in enumerate(_instances(case))]
        b = Batch(h)
        b.plan(psis, nkx0=1, nspin=2, tol=TOL, maxit=MAXIT_ASYNC, prec=case["prec"])
        return {"case": case, "batch": b}
    if kind == "dynamics":
        psi, F, T = _dyn_inputs(case, seed)
        nspin, nkx0 = case["nspin"], case["nkx0"]
        return {"case": case, "psi": psi, "F": F, "T": T, "force": torch.empty_like(F),
                "pc": PairCalculator(symmetric=False, nkx0=nkx0, handle=h),
                "ortho": Ortho(nspin=nspin, handle=h),
                "gsp": GSpacePlane(nkx0=nkx0, cp_min_opt=0, nspin=nspin, handle=h)}
    return {"case": case, "h": h,
            "psi": make_kpoint_states(case["n"], case["npw"], eps=1e-3, seed=seed, device=DEV,
                                      rng="torch")}


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "step":
        sync = case["sync"]
        S, T, out, it, _ = state["h"].ortho_step(
            state["psi"], nkx0=case["nkx0"], nspin=case["nspin"], tol=TOL,
            maxit=MAXIT_SYNC if sync else MAXIT_ASYNC, prec=case["prec"], sync=sync)
        return {"S": S, "T": T, "psi": out, "iterations": it}
    if kind == "batch":
        b = state["batch"]
        b.launch()
        return {"S": b.S, "T": b.T, "psi": b.outs}
    if kind == "dynamics":
        L = state["pc"].multiplyForward(state["psi"], state["F"])
        gamma = state["ortho"].gamma(state["T"], L)
        force = state["gsp"].unpackGamma(gamma, state["T"], state["psi"], state["F"],
                                         state["force"])
        return {"lambda": L, "gamma": gamma, "force": force}
    S, T, out, it, _ = state["h"].zortho_step(state["psi"], nspin=case["nspin"], tol=TOL,
                                              maxit=MAXIT_SYNC, modulus=True, prec=case["prec"])
    return {"S": S, "T": T, "psi": out, "iterations": it}


def _step_work(n, npw):
    # S over its upper triangle, three S -> T iterations, T psi; psi read,
    # T psi written, S and T written
    return (32.0 * n * npw + 16.0 * n * n,
            2.0 * n * (n + 1) * npw + 4.0 * n * n * npw + 3 * 6.0 * n ** 3)


def work(case):
    kind = case["kind"]
    if kind == "batch":
        w = [_step_work(n, npw) for n, npw, _ in _instances(case)]
        return {"bytes": sum(x[0] for x in w), "flops": sum(x[1] for x in w)}
    n, npw = case["n"], case["npw"]
    if kind == "dynamics":
        # Lambda, Gamma^T psi and T F; psi, F and T read, the rest written
        return {"bytes": 48.0 * n * npw + 24.0 * n * n,
                "flops": 12.0 * n * n * npw + 2.0 * n ** 3}
    b, f = _step_work(n, npw)
    if kind == "kpoint":
        # Hermitian S and T psi on complex data
        return {"bytes": b + 16.0 * n * n,
                "flops": 4.0 * n * (n + 1) * npw + 8.0 * n * n * npw + 3 * 24.0 * n ** 3}
    return {"bytes": b, "flops": f}


def _inv_sqrt(B):
    lam, V = torch.linalg.eigh(B.cpu())
    return ((V * lam.rsqrt()) @ V.conj().T).to(B.device)


def _exact_step(psi, nkx0, nspin):
    S = 2.0 * (psi @ psi.T)
    kx = psi[:, :2 * nkx0]
    S -= kx @ kx.T
    S = 0.5 * (S + S.T)
    T = _inv_sqrt(S / 2.0 if nspin == 1 else S)
    return S, T, T @ psi


def exact(case, seed):
    kind = case["kind"]
    if kind == "step":
        psi = _states(case["n"], case["npw"], case["eps"], seed, case["nkx0"], case["nspin"])
        S, T, out = _exact_step(psi, case["nkx0"], case["nspin"])
        return {"S": S, "T": T, "psi": out, "iterations": None}
    if kind == "batch":
        r = [_exact_step(_states(n, npw, eps, seed * 64 + i, 1, 2), 1, 2)
             for i, (n, npw, eps) in enumerate(_instances(case))]
        return {"S": [x[0] for x in r], "T": [x[1] for x in r], "psi": [x[2] for x in r]}
    if kind == "dynamics":
        psi, F, T = _dyn_inputs(case, seed)
        L = psi @ F.T
        gamma = T @ (2.0 * L if case["nspin"] != 1 else L)
        force = T @ F - gamma.T @ psi
        force[:, :2 * case["nkx0"]] *= 0.5 ** 0.5
        return {"lambda": L, "gamma": gamma, "force": force}
    Z = torch.view_as_complex(
        make_kpoint_states(case["n"], case["npw"], eps=1e-3, seed=seed, device=DEV,
                           rng="torch").reshape(case["n"], case["npw"], 2))
    S = Z @ Z.conj().T
    S = 0.5 * (S + S.conj().T)
    T = _inv_sqrt(S)
    out = torch.view_as_real(T @ Z).reshape(case["n"], -1)
    return {"S": S, "T": T, "psi": out, "iterations": None}
