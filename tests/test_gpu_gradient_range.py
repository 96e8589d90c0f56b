"""FP64 gradients at the ends of the range in which quotients share their
divisor's reciprocal (operands zero or within 2^-200 .. 2^200): states and
geometry inside, outside and on both sides of it, zeros of both signs and
cells at rest, bit for bit the oracle's, which divides."""
import numpy as np
import pytest

import oracle as O
from shadowfax_amd import mesh as M
from shadowfax_amd.fluxpass import FluxPass
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu
G = 5.0 / 3.0


def scaled(m, s):
    m = dict(m)
    nd = m["ndim"]
    for k in ("pos", "centroid", "midpoint", "shift", "box"):
        m[k] = m[k] * s
    m["volume"] = m["volume"] * s ** nd
    m["area"] = m["area"] * s ** (nd - 1)
    return m


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("size", [0, -220, 210, -199])
@pytest.mark.parametrize("states", ["plain", "rest", "tiny", "some_tiny", "huge"])
def test_gradients_bit_exact(device, nd, size, states):
    import torch
    print("case", nd, size, states, flush=True)
    m = M.voronoi_periodic(M.poisson_points(300, seed=5, ndim=nd))
    m = scaled(m, 2.0 ** size)
    rng = np.random.default_rng(7)
    W = rng.uniform(0.5, 2.0, (nd + 2, 300))
    W[1:-1] -= 1.0
    if states == "rest":
        W[1] = 0.0
        W[2] = np.where(rng.uniform(size=300) < 0.5, 0.0, -0.0)
        W[0] = 1.0
    elif states == "tiny":
        W *= 2.0 ** -230
    elif states == "some_tiny":
        W[-1, ::7] = 1e-300
        W[0, ::11] = 2.0 ** -201
    elif states == "huge":
        W[-1, ::5] = 2.0 ** 205
    b = M.prepare(m, W, G, kind=0, vel=np.zeros((nd, 300)), dt=1e-3)
    fp = FluxPass(RiemannSolver(0, nd, G, 1e-8, -5.0, "fp64"), M.DeviceMesh(b, "fp64", device))
    fp.gradients()
    torch.cuda.synchronize()
    with np.errstate(all="ignore"):
        ref = O.gradients(0, b)
    got = fp.m.grad_soa()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    assert np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("nd,size", [(2, 0), (3, 0), (2, -400), (3, 400), (2, -520), (2, 520),
                                     (3, -508)])
@pytest.mark.parametrize("kind", [0, 1])
def test_faces_of_any_size(device, nd, size, kind):
    """FP64 face fluxes of meshes whose squared lengths are in, below (down to
    subnormal) and above the range of the shared reciprocals: the oracle's to
    1e-11 normwise (its fluxes' 1e-12, ten quotients in a row), and infinity
    and NaN where it has them."""
    import torch
    print("case", nd, size, kind, flush=True)
    rng = np.random.default_rng(9)
    W = rng.uniform(0.5, 2.0, (nd + 2, 300))
    W[1:-1] -= 1.0
    with np.errstate(all="ignore"):
        m = scaled(M.voronoi_periodic(M.poisson_points(300, seed=5, ndim=nd)),
                   np.float64(2.0) ** size)
        b = M.prepare(m, W, G, kind=kind, vel=rng.uniform(-1, 1, (nd, 300)), dt=1e-3)
        b["mass"] = np.ones(300)  # the large meshes' fluxes meet the mass limiter
        ob = dict(b, grad=np.zeros((nd, nd + 2, 300)))
        _, ref, _, _ = O.face_flux_pass(kind, ob)
    s = RiemannSolver(kind, nd, G, 1e-8, -5.0, "fp64")
    fp = FluxPass(s, M.DeviceMesh(b, "fp64", device))
    fp.m.grad.zero_()
    fp.face_fluxes()
    torch.cuda.synchronize()
    got = fp.m.dQL_soa()
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    ok = np.isfinite(ref).all(0)
    assert np.array_equal(got[:, ~ok], ref[:, ~ok], equal_nan=True)
    err = np.abs(got - ref)[:, ok].max(0)
    scale = np.abs(ref)[:, ok].max(0)
    print("faces %d of %d, max %.2e" % (ok.sum(), len(ok), (err / scale)[scale > 1e-300].max()
                                        if (scale > 1e-300).any() else 0.0), flush=True)
    assert ok.any() and (err <= 1e-11 * scale + 1e-320).all()


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("size", [0, -190, 190])
def test_gradients_of_extreme_states(device, nd, size):
    """States near the ends of their range (2^-500 .. 2^500) and beyond, each
    component another power of two and a tail that falls through the whole
    range to subnormals and zero, bit for bit the oracle's."""
    import torch
    m = scaled(M.voronoi_periodic(M.poisson_points(300, seed=5, ndim=nd)), 2.0 ** size)
    rng = np.random.default_rng(11)
    for powers in ((-495, -505, 0, -90), (495, 480, 0, 300), (-600, 0, 490, -499)):
        print("case", nd, size, powers, flush=True)
        W = rng.uniform(0.5, 2.0, (nd + 2, 300))
        for k, e in enumerate(powers):
            W[k] *= 2.0 ** e
        W[1] *= rng.choice([-1.0, 1.0], 300)
        W[2, ::2] *= np.exp(-rng.uniform(0, 28, 150) ** 2)
        with np.errstate(all="ignore"):
            b = M.prepare(m, W, G, kind=0, vel=np.zeros((nd, 300)), dt=1e-3)
            ref = O.gradients(0, b)
        fp = FluxPass(RiemannSolver(0, nd, G, 1e-8, -5.0, "fp64"),
                      M.DeviceMesh(b, "fp64", device))
        fp.gradients()
        torch.cuda.synchronize()
        got = fp.m.grad_soa()
        assert np.array_equal(np.isnan(got), np.isnan(ref))
        assert np.array_equal(got, ref, equal_nan=True)
