"""Vacuum beside a gas, on either side, on both and at walls: every outcome of
solve_vacuum and vacuum_flux (the gas itself, its fan, nothing) and gases on
both sides of the ranges beyond which the step-by-step paths run, against the
oracle.  The fluxes are closed forms of one state: 1e-12 normwise in FP64, the
mixed path's 1e-6 otherwise; status bytes and vacuum counts are equal."""
import numpy as np
import pytest

import oracle as O
from shadowfax_amd import workloads as WK
from shadowfax_amd.metrics import normwise_error
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu
N = 3000


def batch(nd, seed):
    b = WK.riemann_batch(N, seed=seed, family="uniform", ndim=nd, round32=False)
    WL, WR, n = b["WL"], b["WR"], b["n"]
    r = np.random.RandomState(seed)
    k = np.arange(N)
    for W in (WL, WR):  # from -8 to 8 sound speeds along the normal
        W[1:1 + nd] += r.uniform(-8, 8, N) * np.sqrt(W[-1] / W[0]) * n
    for lo, f in ((2400, 1e-48), (2500, 1e-53), (2600, 1e48), (2700, 1e52), (2800, 1e-103)):
        m = (k >= lo) & (k < lo + 100)
        for W in (WL, WR):
            W[0, m] *= f
            W[-1, m] *= f
    empty = r.randint(0, 20, N)
    WL[:, (empty < 9) | (empty == 19)] = 0.0
    WR[:, empty >= 9] = 0.0
    # vacuum is a zero density, whatever the rest says
    WL[1:, (empty < 9) & (k % 3 == 0)] = 3.0
    return WL, WR, n, (r.uniform(size=N) < 0.1).astype(np.uint8), r.uniform(-1, 1, (nd, N))


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 1.66667])
def test_vacuum_sides(device, gamma, kind, nd):
    import torch
    print("case", gamma, kind, nd, flush=True)
    WL, WR, n, refl, v = batch(nd, 31)
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
    with np.errstate(all="ignore"):
        Fo, sto, c = O.solve_for_flux(kind, nd, WL, WR, n, v=v, refl=refl, gamma=gamma)
    for prec, tol in (("fp64", 1e-12), ("mixed", 1e-6)):
        s = RiemannSolver(kind, nd, gamma, 1e-8, -5.0, prec)
        st = torch.full((N,), 9, dtype=torch.uint8, device=device)
        F = s.solve_for_flux_batch(t(WL), t(WR), t(n), t(v), t(refl), status=st).cpu().numpy()
        assert s.stats()["nvacuum"] == c.nvacuum
        # (a wall makes two gases: the mixed path's general iteration holds
        # them in FP32)
        held = (np.arange(N) < 2400) if prec == "mixed" else np.ones(N, bool)
        assert np.array_equal((st.cpu().numpy() != 0)[held], (sto != 0)[held])
        m = np.isfinite(Fo).all(0) & held
        WRe = np.where(refl != 0, WL, WR)
        err = normwise_error(F[:, m], Fo[:, m], WL[:, m], WRe[:, m], gamma)
        print(prec, "max %.2e" % err.max(), flush=True)
        assert m.mean() > 0.7 and np.isfinite(F[:, m]).all()
        assert err.max() <= tol
        if kind == 0 and prec == "fp64":
            W = s.solve_batch(t(WL), t(WR), t(n), t(refl)).cpu().numpy()
            Wo = O.exact_solve(nd, WL, WR, n, refl=refl, gamma=gamma)[0]
            scale = np.abs(Wo).max(0) + 1e-300
            assert (np.abs(W - Wo).max(0) / scale).max() <= 1e-12
