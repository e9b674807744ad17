"""The far field of the device FMM (multipoles evaluated at the targets, one source cell per lane) at
the edges of its tasks: groups of one target to more than three tiles of 16, list chunks of every
size from 1 to 64 entries (the last, partial chunk holds its entries once, twice or four times over),
both expansions in one pass (FP32; FP64 at order 4), one pass per set (FP64 at 6 and 8) and several
passes over columns (FP64 at 10), and the lower far degree. Device against the host evaluation of the
same plan: the same sums in another order and normalisation, so 1e-10 of the largest potential in
FP64; in mixed precision the bounds of test_fmm (far and v expansions cut to lower degrees)."""
import numpy as np
import pytest

from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh
from test_fmm import charged, fmm_ref

CASES = [((6, 5, 4), 4, 0), ((9, 7, 5), 256, 0), ((30, 4, 2), 32, 0), ((14, 13, 12), 1500, 0), ((20, 10, 3), 16, 1),
         ((11, 11, 11), 100, 1)]


@pytest.mark.gpu
@pytest.mark.parametrize("order", [4, 6, 8, 10])
@pytest.mark.parametrize("cells,leaf,low", CASES)
def test_far_field_at_task_edges(cells, leaf, low, order):
    far = {4: 2, 6: 4, 8: 5, 10: 6}[order] if low else order
    m = HostMesh.cuboid(tuple(6.0 * c for c in cells), cells, jitter=0.1, seed=4)
    m.prepare({"volume": dict(Ms=8e5)})
    p, u, v = charged(m)
    xyz, qu, qv = p.sources()
    cu, cv = p.corrections()
    pu, pv, _ = fmm_ref(xyz, qu, qv, m.arrays()["pos"], order, leaf, far=far)
    ref = (pu + cu) / (4 * np.pi), (pv + cv) / (4 * np.pi)
    for prec in ("fp64", "mixed"):
        g = Engine(m.mesh, demag="fmm", fmm_order=order, fmm_leaf=leaf, fmm_far_order=far, precision=prec)
        i = g.fmm_info()
        assert i["m2p_pairs"] <= i["m2p_slots"]
        g.set_state(nv.FG_BOTH, u=u, v=v)
        g.calc_demag()
        pot = g.get_state(nv.FG_NEXT)[2:]
        err = [np.abs(a - b).max() / np.abs(b).max() for a, b in zip(pot, ref)]
        bound = (1e-10, 1e-10) if prec == "fp64" else (1e-4, 1e-2)
        assert err[0] <= bound[0] and err[1] <= bound[1], (prec, err)
        g.close()


@pytest.mark.gpu
def test_order_10_costs_its_operations():
    """In FP64 an order-10 cell takes 1.5 times the operations of an order-8 one and, its sets not
    fitting the registers, two passes per set. Its M2P measures 1.75 times the time; with unequal parts
    that spill, and pieces fetched that a pass does not use, 2.7 times."""
    m = HostMesh.cuboid((180.0, 150.0, 18.0), (60, 50, 6), jitter=0.1, seed=5)
    m.prepare({"volume": dict(Ms=8e5)})
    rng = np.random.default_rng(1)
    u = np.array([1.0, 0.4, 0.0]) + rng.uniform(-0.2, 0.2, size=(m.n_nodes, 3))
    t = {}
    for order in (8, 10):
        g = Engine(m.mesh, demag="fmm", fmm_order=order, profile=True)
        g.set_state(nv.FG_BOTH, u=u / np.linalg.norm(u, axis=1, keepdims=True))
        g.calc_demag()
        g.reset_kernel_stats()
        for _ in range(10):
            g.calc_demag()
        n, ms = g.kernel_stats()["fmm_m2p"]
        t[order] = ms / n
        g.close()
    assert t[10] <= 2.2 * t[8], t
