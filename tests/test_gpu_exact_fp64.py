"""The FP64 exact solver's iteration (fp64::ex_solve) against the oracle's
step-by-step one over what it accepts and at the edges of it: the gases with
an integer root (5/3, 7/5) and others (pow), states from near-vacuum to 1e6
jumps, pressure ratios and densities on both sides of the limits beyond which
the step-by-step path runs, walls and moving faces.

Tolerance: both iterations take the same steps and tests; Brent's method may
stop up to 1e-8 from the root, and where it does so, round-off in the pressure
function moves its last iterates by a multiple of that round-off (1e-16)
that grows with the number of steps: 1e-10 normwise leaves six decades.  Newton's
method ends within round-off of the root: 1e-12, as for the fluxes in general."""
import numpy as np
import pytest

import oracle as O
from shadowfax_amd import workloads as WK
from shadowfax_amd.metrics import normwise_error
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu
TOL = 1e-10
TOL_NEWTON = 1e-12


def edge_batch(nd, seed):
    """The mixed family, then blocks of it rescaled: pressures 1e10 to 1e13
    apart each way (ratios to 1e26: the limit is 1e24), densities and pressures
    around 1e-100 and 1e100, colliding and separating streams, and equal
    states."""
    b = WK.riemann_batch(6000, seed=seed, family="mixed", ndim=nd, round32=False)
    WL, WR, n = b["WL"], b["WR"], b["n"]
    u = np.random.RandomState(seed).uniform(size=6000)
    k = np.arange(6000)
    m = (k >= 2000) & (k < 3000)
    WL[-1, m] *= 10.0 ** (10 + 3 * u[m])
    WR[-1, m] *= 10.0 ** -(10 + 3 * u[m])
    for lo, f in ((3000, 1e-100), (3250, 1e100)):  # sound speeds unchanged
        m = (k >= lo) & (k < lo + 250)
        for W in (WL, WR):
            W[0, m] *= f
            W[-1, m] *= f
    m = (k >= 3500) & (k < 4000)
    WR[:, m] = WL[:, m]
    m = (k >= 4000) & (k < 5000)
    s = 10.0 ** (4 * u[m]) * np.sqrt(WL[-1, m] / WL[0, m])
    WL[1:1 + nd, m] += s * n[:, m]
    WR[1:1 + nd, m] -= s * n[:, m]
    m = k >= 5000
    s = 4 * u[m] * np.sqrt(WL[-1, m] / WL[0, m])
    WL[1:1 + nd, m] -= s * n[:, m]
    WR[1:1 + nd, m] += s * n[:, m]
    return WL, WR, n


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 1.4, 1.66667, 2.0, 1.05])
def test_exact_fp64_matches_step_by_step(device, gamma, nd):
    import torch
    print("case", gamma, nd, flush=True)
    WL, WR, n = edge_batch(nd, 17)
    N = WL.shape[1]
    rng = np.random.RandomState(3)
    v = rng.uniform(-1, 1, (nd, N))
    refl = (rng.uniform(size=N) < 0.05).astype(np.uint8)
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
    s = RiemannSolver(0, nd, gamma, 1e-8, -5.0, "fp64")
    st = torch.zeros(N, dtype=torch.uint8, device=device)
    F = s.solve_for_flux_batch(t(WL), t(WR), t(n), t(v), t(refl), status=st)
    Wh = s.solve_batch(t(WL), t(WR), t(n), t(refl))
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        Fo, sto, c = O.solve_for_flux(O.EXACT, nd, WL, WR, n, v=v, refl=refl, gamma=gamma)
        Wo = O.exact_solve(nd, WL, WR, n, refl=refl, gamma=gamma)[0]
        err = normwise_error(F.cpu().numpy(), Fo, WL, WR, gamma)
    assert np.array_equal(st.cpu().numpy() != 0, sto != 0)
    ok = (sto == 0) & np.isfinite(Fo).all(0)
    scale = np.maximum(np.abs(WL), np.abs(np.where(refl, WL, WR))).max(0)
    eh = (np.abs(Wh.cpu().numpy() - Wo) / np.maximum(scale, np.abs(Wo).max(0))).max(0)
    # without Brent's method, and without streams that collide at up to 1e4 sound
    # speeds, whose momenta cancel, both iterations end at the root
    brent = np.array([O.solve_for_flux(O.EXACT, nd, WL[:, i:i + 1], WR[:, i:i + 1], n[:, i:i + 1],
                                       v=v[:, i:i + 1], refl=refl[i:i + 1],
                                       gamma=gamma)[2].nbrent for i in range(N)])
    k = np.arange(N)
    newton = ok & (brent == 0) & ((k < 2000) | ((k >= 3500) & (k < 4000)) | (k >= 5000))
    print("flux %.2e half state %.2e, Newton's alone %.2e %.2e" % (
        err[ok].max(), eh[ok].max(), err[newton].max(), eh[newton].max()), flush=True)
    assert ok.mean() > 0.9 and newton.sum() > 2500
    assert err[ok].max() <= TOL and eh[ok].max() <= TOL
    if gamma >= 1.4:  # (1.05: near vacuum the steps shrink too slowly to tell the root)
        assert err[newton].max() <= TOL_NEWTON and eh[newton].max() <= TOL_NEWTON
    assert s.stats()["nvacuum"] == 2 * c.nvacuum


def two_rarefactions(WL, WR, n, gamma):
    """Half state [rho, p] of problems with two rarefactions, closed forms in
    80 bits."""
    L = np.longdouble
    WL, WR, n, g = WL.astype(L), WR.astype(L), n.astype(L), L(gamma)
    e, m = (g - 1) / (2 * g), 2 / (g - 1)
    uL, uR = (WL[1:-1] * n).sum(0), (WR[1:-1] * n).sum(0)
    aL, aR = np.sqrt(g * WL[-1] / WL[0]), np.sqrt(g * WR[-1] / WR[0])
    q = (WL[-1] / WR[-1]) ** e
    z = (aL + aR - (uR - uL) / m) / (aL + aR * q)  # (p*/pL)^e
    u = uL - m * aL * (z - 1)
    right = u < 0
    W, s = np.where(right, WR, WL), np.where(right, -1, 1)
    uK, a, y = np.where(right, uR, uL), np.where(right, aR, aL), np.where(right, z * q, z)
    b = 2 / (g + 1) + s * (g - 1) / (g + 1) / a * uK
    fan = s * (u - s * a * y) > 0
    out = s * (uK - s * a) >= 0
    y = np.where(out, 1, np.where(fan, b, y))
    return np.stack([W[0] * y ** m, W[-1] * y ** (1 / e)])


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("gamma", [5.0 / 3.0, 5.0 / 3.0 + 9e-13, 1.4, 1.4 - 3e-13, 1.66667])
def test_half_states_to_round_off(device, gamma, nd):
    """Density and pressure behind and inside rarefactions, also for gammas
    next to 5/3 and 7/5.  Streams that separate at up to 0.8 of the vacuum
    speed: the sum of the sound speeds less the separation has 5 times its
    terms' round-off (of 3 roundings each), p* the 7th power of it; with some
    20 roundings behind it 130 times 1.1e-16, 2e-14."""
    import torch
    print("case", gamma, nd, flush=True)
    N = 20000
    b = WK.riemann_batch(N, seed=41, family="uniform", ndim=nd, round32=False)
    WL, WR, n = b["WL"], b["WR"], b["n"]
    r = np.random.RandomState(43)
    WR[-1] = WL[-1] * 10.0 ** r.uniform(-0.5, 0.5, N)
    WR[0] = WL[0] * 10.0 ** r.uniform(-1, 1, N)
    aL, aR = np.sqrt(gamma * WL[-1] / WL[0]), np.sqrt(gamma * WR[-1] / WR[0])
    # the contact from -2 to 2 sound speeds of the faster side
    mid = r.uniform(-2, 2, N) * np.maximum(aL, aR) * n
    sep = 2 / (gamma - 1) * (aL + aR) * r.uniform(0.4, 0.8, N) * n
    WL[1:-1], WR[1:-1] = mid - 0.5 * sep, mid + 0.5 * sep
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
    s = RiemannSolver(0, nd, gamma, 1e-8, -5.0, "fp64")
    W = s.solve_batch(t(WL), t(WR), t(n)).cpu().numpy()
    T = two_rarefactions(WL, WR, n, gamma)
    err = (np.abs(W[[0, -1]] - T) / T).astype(float)
    print("max %.2e median %.2e" % (err.max(), np.median(err)), flush=True)
    assert err.max() <= 2e-14
