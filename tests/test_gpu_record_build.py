"""The grouped entry records (entry_geometry_grouped_kernel) against those in
entry order: record k of slot l of a group lies in row k, lane l, plane by
plane, and everything past a slot's entries is zero.  Meshes whose face and
cell counts leave remainders of 4 and 64, with and without the face records,
and one whose longest cells exceed the rows that a block holds in LDS.  Exact:
the layouts hold the same numbers."""
import numpy as np
import pytest

from shadowfax_amd import mesh as M
from shadowfax_amd.riemann import RiemannSolver

pytestmark = pytest.mark.gpu


def bundle(nd, cells):
    mesh = M.voronoi_periodic(M.poisson_points(cells, seed=cells, ndim=nd))
    W = np.ones((nd + 2, mesh["C"]))
    return M.prepare(mesh, W, gamma=5.0 / 3.0)


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
@pytest.mark.parametrize("nd,cells", [(2, 63), (2, 1001), (3, 130), (3, 3001), (3, 20000)])
def test_grouped_records(device, nd, cells, precision):
    import torch
    print("case", nd, cells, precision, flush=True)
    b = bundle(nd, cells)
    out = {}
    for name, kw in (("order", dict(grouped=False)), ("group", dict(grouped=True)),
                     ("arrays", dict(grouped=True, face_records=False))):
        s = RiemannSolver(1, nd, 5.0 / 3.0, 1e-8, -5.0, precision)
        dm = M.DeviceMesh(b, precision, device, **kw)
        dm.build_entries(s.handle)
        torch.cuda.synchronize()
        out[name] = dm
    d = out["group"]
    off = d.arr["cf_off"].cpu().numpy()
    grp = d.arr["egeo_group"].cpu().numpy()
    rec = out["order"].egeo.cpu().numpy()
    item = rec.dtype.itemsize
    P = rec.shape[1] * item // 16
    want = np.zeros((d.egeo_rows, P, 64, 16 // item), rec.dtype)
    if d.sorted:
        slot = d.arr["egeo_slot"].cpu().numpy()
        cell, n = slot & 0xffffffff, slot >> 32
    else:
        cell, n = np.arange(d.C), np.diff(off)
    for s_ in range(d.C):
        for k in range(int(n[s_])):
            want[grp[s_ // 64] + k, :, s_ % 64] = rec[off[cell[s_]] + k].reshape(P, -1)
    if (nd, cells) == (3, 20000):
        assert np.diff(grp).max() > 24
    for name in ("group", "arrays"):
        got = out[name].egeo.cpu().numpy().reshape(want.shape)
        assert np.array_equal(got.view(np.uint8), want.view(np.uint8)), name
