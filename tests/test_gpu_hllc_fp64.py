"""The FP64 HLLC fluxes (fp64::hllc_solve_for_flux) against the oracle's over
what the solver accepts: gases whose vacuum fans are products (5/3, 7/5) and
others (pow), vacuum on either side and between two gases, supersonic and
resting states, walls, and states on both sides of the limits (1e-50, 1e50,
1e12 sound speeds) beyond which the expression-by-expression path runs.

Tolerance: some hundred roundings of 1.1e-16 of terms no larger than
rho U max(1, U)^2 with U = |u| + a + |v|, times a factor of 50 for the
quotients in a row: 1e-12 of that scale."""
import numpy as np
import pytest

import oracle as O
from shadowfax_amd import workloads as WK
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu
TOL = 1e-12


def edge_batch(nd, seed):
    b = WK.riemann_batch(6000, seed=seed, family="mixed", ndim=nd, round32=False)
    WL, WR, n = b["WL"], b["WR"], b["n"]
    u = np.random.RandomState(seed).uniform(size=6000)
    k = np.arange(6000)
    for lo, f in ((2000, 1e-49), (2300, 1e-52), (2600, 1e48), (2800, 1e51)):
        m = (k >= lo) & (k < lo + 200)
        WL[0, m] *= f
        WL[-1, m] *= f
        WR[0, m] *= f
        WR[-1, m] *= f
    m = (k >= 3000) & (k < 3300)
    WL[0, m] = WL[-1, m] = 0.0
    m = (k >= 3200) & (k < 3600)
    WR[0, m] = WR[-1, m] = 0.0
    m = (k >= 3600) & (k < 4000)
    WR[:, m] = WL[:, m]
    m = (k >= 4000) & (k < 5000)
    s = 10.0 ** (14 * u[m]) * np.sqrt(WL[-1, m] / WL[0, m])
    WL[1:1 + nd, m] += s * n[:, m]
    WR[1:1 + nd, m] += s * n[:, m]
    m = k >= 5000
    s = 6 * u[m] * np.sqrt(WL[-1, m] / WL[0, m])
    WL[1:1 + nd, m] -= s * n[:, m]
    WR[1:1 + nd, m] += s * n[:, m]
    return WL, WR, n


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 1.66667, 1.05])
def test_hllc_fp64_over_its_range(device, gamma, nd):
    import torch
    print("case", gamma, nd, flush=True)
    WL, WR, n = edge_batch(nd, 23)
    N = WL.shape[1]
    rng = np.random.RandomState(5)
    v = rng.uniform(-1, 1, (nd, N))
    refl = (rng.uniform(size=N) < 0.05).astype(np.uint8)
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
    s = RiemannSolver(1, nd, gamma, 1e-8, -5.0, "fp64")
    F = s.solve_for_flux_batch(t(WL), t(WR), t(n), t(v), t(refl)).cpu().numpy()
    with np.errstate(all="ignore"):
        Fo, _, c = O.solve_for_flux(O.HLLC, nd, WL, WR, n, v=v, refl=refl, gamma=gamma)
        a = [np.where(W[0] > 0, np.sqrt(gamma * W[-1] / W[0]), 0.0) for W in (WL, WR)]
    U = np.maximum(np.abs(WL[1:-1]).sum(0) + a[0], np.abs(WR[1:-1]).sum(0) + a[1])
    U = U + np.abs(v).sum(0)
    scale = np.maximum(WL[0], WR[0]) * U * np.maximum(1.0, U) ** 2
    ok = np.isfinite(Fo).all(0) & (scale > 0)
    err = np.abs(F - Fo).max(0)[ok] / scale[ok]
    print("max %.2e" % err.max(), flush=True)
    assert ok.mean() > 0.9 and np.isfinite(F[:, ok]).all()
    assert err.max() <= TOL
    assert s.stats()["nvacuum"] == c.nvacuum
