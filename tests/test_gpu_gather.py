"""sfx_gather_dQ over index lists of every shape its blocks meet: sizes around
the cells of a block, cells without entries, ragged counts, and cells with
more entries than a block keeps in LDS.  The sums are the ordered sums of the
rows, bit for bit."""
import ctypes as ct

import numpy as np
import pytest

from shadowfax_amd import _capi as Cp
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu


def ordered(off, ent, dQL):
    acc = np.zeros((len(off) - 1, dQL.shape[1]))
    deg = np.diff(off)
    for p in range(int(deg.max()) if len(deg) else 0):
        c = np.where(deg > p)[0]
        e = ent[off[c] + p]
        x = dQL[e >> 1].astype(np.float64)
        acc[c] += np.where((e & 1)[:, None] == 1, -x, x)
    return acc


@pytest.mark.parametrize("nd", [2, 3])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("counts", ["one", "empty", "ragged", "many", "huge"])
def test_gather_shapes(device, nd, precision, counts):
    import torch
    rng = np.random.RandomState(11)
    dt = np.float64 if precision == "fp64" else np.float32
    s = RiemannSolver(1, nd, 5.0 / 3.0, 1e-8, -5.0, precision)
    for C in (1, 31, 32, 33, 47, 48, 49, 63, 64, 65, 200):
        print("case", nd, precision, counts, C, flush=True)
        deg = {"one": np.ones(C, int), "empty": np.zeros(C, int),
               "ragged": rng.randint(0, 40, C), "many": np.full(C, 45),
               "huge": np.where(np.arange(C) == C // 2, 3000, 5)}[counts]
        off = np.concatenate([[0], np.cumsum(deg)]).astype(np.int64)
        F = max(1, int(off[-1]))
        ent = (2 * rng.randint(0, F, off[-1]) + rng.randint(0, 2, off[-1])).astype(np.int32)
        dQL = rng.standard_normal((F, nd + 2)).astype(dt)
        t = lambda a: torch.tensor(np.ascontiguousarray(a), device=device)
        to, te, tq = t(off), t(np.concatenate([ent, [0]]).astype(np.int32)), t(dQL)
        out = torch.full(((C + 1) * (nd + 2),), 7.25, dtype=torch.float64, device=device)
        d = Cp.MeshDesc()
        d.ndim, d.C, d.F = nd, C, F
        p = lambda x: ct.c_void_p(x.data_ptr())
        d.gather_off, d.gather_entry = p(to), p(te)
        Cp.check(Cp.lib().sfx_gather_dQ(s.handle, ct.byref(d), p(tq), p(out), None))
        torch.cuda.synchronize()
        got = out.cpu().numpy().reshape(C + 1, nd + 2)
        assert np.array_equal(got[:C], ordered(off, ent, dQL))
        assert np.all(got[C] == 7.25)
