"""Multipoles of the leaves at the edges of their launch: leaves that do not fill a wavefront's eight,
nor a launch's 64, and leaves from fewer sources than a leaf's eight lanes to many. Device against the
host evaluation of the same plan: the same sums in another order, so 1e-10 of the largest potential
in FP64, and the bounds of test_fmm in mixed precision."""
import numpy as np
import pytest

from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh
from test_fmm import charged, fmm_ref

CASES = [((3, 3, 3), 3), ((5, 4, 3), 8), ((7, 5, 4), 12), ((9, 8, 3), 20), ((12, 12, 6), 700)]


@pytest.mark.gpu
@pytest.mark.parametrize("order", [4, 8, 10])
@pytest.mark.parametrize("cells,leaf", CASES)
def test_leaf_multipoles(cells, leaf, order):
    m = HostMesh.cuboid(tuple(5.0 * c for c in cells), cells, jitter=0.1, seed=6)
    m.prepare({"volume": dict(Ms=8e5)})
    p, u, v = charged(m)
    xyz, qu, qv = p.sources()
    cu, cv = p.corrections()
    pu, pv, _ = fmm_ref(xyz, qu, qv, m.arrays()["pos"], order, leaf, far=order)
    ref = (pu + cu) / (4 * np.pi), (pv + cv) / (4 * np.pi)
    for prec, bound in (("fp64", (1e-10, 1e-10)), ("mixed", (1e-4, 1e-2))):
        g = Engine(m.mesh, demag="fmm", fmm_order=order, fmm_leaf=leaf, fmm_far_order=order, precision=prec)
        g.set_state(nv.FG_BOTH, u=u, v=v)
        g.calc_demag()
        pot = g.get_state(nv.FG_NEXT)[2:]
        err = [np.abs(a - b).max() / np.abs(b).max() for a, b in zip(pot, ref)]
        assert err[0] <= bound[0] and err[1] <= bound[1], (prec, g.fmm_info()["leaves"], err)
        g.close()
