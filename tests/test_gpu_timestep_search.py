"""sfx_hydro_timestep's step search over time lines of every kind (a power of
two ticks or not, steps from the whole line down to a tick and below), cells
whose remaining time has many or no trailing zero bits, and cell counts around
a block: equal to the oracle's search, which halves down from the whole line,
in every output."""
import numpy as np
import pytest

import oracle as O
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu
G = 5.0 / 3.0


@pytest.mark.parametrize("M", [1 << 60, 3 << 50, (1 << 60) - 1, 1 << 20, 1000])
@pytest.mark.parametrize("nd,kind", [(2, 0), (3, 1)])
@pytest.mark.parametrize("glob", [0, 1])
def test_step_search(device, M, nd, kind, glob):
    import torch
    for C in (1, 255, 1023, 1024, 1025, 5000):
        print("case", M, nd, kind, glob, C, flush=True)
        rng = np.random.default_rng(C)
        W = np.ones((C, nd + 2))
        W[:, 1:-1] = rng.normal(size=(C, nd))
        # sound speeds, and so steps, over 40 decades; some cells at rest
        # without pressure (an infinite step), some so fast that none is left
        W[:, -1] = 10.0 ** rng.uniform(-40, 40, C)
        rest = rng.uniform(size=C) < 0.02
        W[rest, 1:] = 0.0
        vel = np.where(rest[:, None], 0.0, W[:, 1:-1] + 1e-20)
        V = rng.uniform(0.5, 2.0, C)
        now = M // 5
        d = dict(integer_maxtime=M, current_time=now - now // 3, timestep=now // 3,
                 max_timestep=max(1, M // 3), min_timestep=1, tottime=7.3, mintime=0.1,
                 cfl=0.4, global_timestep=glob)
        # the time left: odd, or a multiple of a large power of two, or none
        end = np.where(rng.uniform(size=C) < 0.8, now, now + 1 + rng.integers(0, 4, C))
        end = end.astype(np.uint64)
        if glob:
            end[:] = now
        start = np.zeros(C, np.uint64)
        s0, e0, dt0, a0, ss0, na0, st0 = O.hydro_timestep(kind, nd, W, vel, V, O.timeline(**d),
                                                          start, end, gamma=G)
        s = RiemannSolver(kind, nd, G, 1e-8, -5.0, "fp64")
        t = lambda a: torch.tensor(a, device=device)
        sd, ed = t(start.view(np.int64)), t(end.view(np.int64))
        dt, act, status, res = s.hydro_timestep(t(W), t(vel), t(V), d, sd, ed)
        torch.cuda.synchronize()
        assert np.array_equal(sd.cpu().numpy().view(np.uint64), s0)
        assert np.array_equal(ed.cpu().numpy().view(np.uint64), e0)
        assert np.array_equal(dt.cpu().numpy(), dt0)
        assert np.array_equal(act.cpu().numpy(), a0)
        assert np.array_equal(status.cpu().numpy(), st0)
        r = res.cpu().numpy().view(np.uint64)
        assert r[0] == ss0 and r[1] == na0
