"""Multipoles of the leaves at the edges of their launch: leaves that do not fill a wavefront's eight,
nor a launch's 64, and leaves from fewer sources than a leaf's eight lanes to many. Device against the
host evaluation of the same plan: the same sums in another order, so 1e-10 of the largest potential
in FP64; in mixed precision 2e-6 as in test_fmm_far_field, phi_v with its multipoles cut to degree 4."""
import numpy as np
import pytest

from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh
from test_fmm import charged, fmm_ref
from test_fmm_far_field import far_cut

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
    xyz, pos = xyz.reshape(-1, 3), m.arrays()["pos"]
    pu, pv, L = fmm_ref(xyz, qu, qv, pos, order, leaf, far=order)
    at = np.unique(np.linspace(0, len(pos) - 1, 120).astype(int))
    full = (pu + cu) / (4 * np.pi), (pv + cv) / (4 * np.pi)
    cut = (far_cut(xyz, qv, pv, (pos, at), L, order, order, 4) + cv[at]) / (4 * np.pi)
    for prec in ("fp64", "mixed"):
        g = Engine(m.mesh, demag="fmm", fmm_order=order, fmm_leaf=leaf, fmm_far_order=order, precision=prec)
        g.set_state(nv.FG_BOTH, u=u, v=v)
        g.calc_demag()
        phi, phiv = g.get_state(nv.FG_NEXT)[2:]
        err = [np.abs(a - b).max() / np.abs(b).max() for a, b in zip((phi, phiv), full)]
        if prec == "mixed":
            err[1] = np.abs(phiv[at] - cut).max() / np.abs(full[1]).max()
        assert max(err) <= (1e-10 if prec == "fp64" else 2e-6), (prec, g.fmm_info()["leaves"], err)
        g.close()
