"""Results that kernels write to pinned host memory: Ensemble.read of meshes
below, at and above the staging buffer's 2^17 values (in pieces then), equal to
sfx_ensemble_read's rows; and the scalar solves, call after call on one handle,
equal to the batched ones."""
import numpy as np
import pytest

from shadowfax_amd import mesh as M
from shadowfax_amd import serving as S
from shadowfax_amd import workloads as WK
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu
G = 5.0 / 3.0


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_read_is_the_rows(device, precision):
    s = RiemannSolver(1, 2, G, 1e-8, -5.0, precision)
    dms = []
    for side in (2, 9, 181, 190):  # 16, 324, 131,044 and 144,400 values (2^17 = 131,072)
        m = M.voronoi_periodic(M.hilbert_sorted(M.jittered_grid(side, 0.25, seed=side)))
        dms.append(M.DeviceMesh(M.prepare(m, M.kh_ics(m), G, kind=1), precision, device))
    C, F, E = (sum(x) for x in zip(*((d.C, d.F, d.E) for d in dms)))
    ens = S.Ensemble(s, len(dms), C, F, E, C, F)
    ids = [ens.add(d) for d in dms]
    for _ in range(2):
        ens.step(ids)
        for k, d in zip(ids, dms):
            for what in (S.ENS_W, S.ENS_Q, S.ENS_DQ):
                rows = np.empty((d.C, 4))
                S.Cp.check(S._lib().sfx_ensemble_read(ens.h, k, what, S._p(rows, S._dp)))
                got = ens.read(k, what)
                assert got.shape == (4, d.C) and got.flags.c_contiguous
                assert np.array_equal(got, rows.T)


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_scalar_calls_equal_the_batch(device, nd, kind, precision):
    import torch
    b = WK.riemann_batch(40, seed=2, family="mixed", ndim=nd)
    v = np.random.RandomState(1).uniform(-1, 1, (nd, 40))
    refl = (np.arange(40) % 5 == 0).astype(np.uint8)
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
    s = RiemannSolver(kind, nd, G, 1e-8, -5.0, precision)
    F = s.solve_for_flux_batch(t(b["WL"]), t(b["WR"]), t(b["n"]), t(v), t(refl)).cpu().numpy()
    n0 = s.stats()
    for i in range(40):
        got = s.solve_for_flux(b["WL"][:, i], b["WR"][:, i].copy(), b["n"][:, i], v[:, i],
                               bool(refl[i]))
        assert np.array_equal(got, F[:, i]), i
    # the scalar calls are counted as the batch is
    n1 = s.stats()
    assert all(n1[k] == 2 * n0[k] for k in n0), (n0, n1)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_scalar_calls_of_several_threads(device, precision):
    """Threads that solve on one handle each get their own problem's flux."""
    import threading
    import torch
    T, N = 4, 200
    b = WK.riemann_batch(T * N, seed=7, family="uniform", ndim=3)
    t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
    s = RiemannSolver(0, 3, G, 1e-8, -5.0, precision)
    F = s.solve_for_flux_batch(t(b["WL"]), t(b["WR"]), t(b["n"])).cpu().numpy()
    got, errors = np.zeros_like(F), []

    def work(k):
        try:
            for i in range(k * N, (k + 1) * N):
                got[:, i] = s.solve_for_flux(b["WL"][:, i], b["WR"][:, i], b["n"][:, i])
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(T)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    assert not errors, errors
    assert np.array_equal(got, F)
