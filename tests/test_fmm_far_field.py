"""The far field of the device FMM (multipoles evaluated at the targets, one source cell per lane) at
the edges of its tasks: groups of one target to more than three tiles of 16, list chunks of every
size from 1 to 64 entries (the last, partial chunk holds its entries once, twice or four times over),
both expansions in one pass (FP32; FP64 at order 4), one pass per set (FP64 at 6 and 8) and several
passes over columns (FP64 at 10), and the lower far degree. Device against the host evaluation of the
same plan: the same sums in another order and normalisation, so 1e-10 of the largest potential in
FP64; in mixed precision the bounds of test_fmm (far and v expansions cut to lower degrees)."""
import ctypes as C

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


def leaf_cells(x, pos, level):
    """Integer coordinates of the leaves of points x in the octree over a mesh of nodes pos."""
    lo, hi = pos.min(0), pos.max(0)
    half = 0.5 * (hi - lo).max() * (1 + 1e-9)
    return np.floor((x - (0.5 * (lo + hi) - half)) * 2.0**level / (2 * half)).astype(int)


@pytest.mark.gpu
@pytest.mark.parametrize("order", [4, 6, 8, 10])
def test_overflowed_cell_stays_with_its_targets(order):
    """Charges of v beyond FP32 at one node make the expansions of its leaf infinite. Targets whose
    near field holds all of them take them in FP64 and stay finite and accurate, also where other
    targets of the same group evaluate that leaf; so does every potential of u."""
    m = HostMesh.cuboid((84.0, 84.0, 84.0), (14, 14, 14), jitter=0.1, seed=4)
    m.prepare({"volume": dict(Ms=8e5)})
    a = m.arrays()
    pos = a["pos"]
    rng = np.random.default_rng(3)
    u = rng.normal(size=pos.shape) * 0.3 + [1, 0.5, 0]
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    v = rng.normal(size=pos.shape)
    k = int(np.argmin(np.linalg.norm(pos - (pos.min(0) + 0.4 * np.ptp(pos, axis=0)), axis=1)))
    v[k] = 1e60
    out, level = {}, 0
    for prec in ("fp64", "mixed"):
        g = Engine(m.mesh, demag="fmm", fmm_order=order, fmm_leaf=64, fmm_far_order=order, precision=prec)
        level = g.fmm_info()["leaf_level"]
        g.set_state(nv.FG_BOTH, u=u, v=v)
        g.calc_demag()
        out[prec] = g.get_state(nv.FG_NEXT)[2:]
        g.close()
    pg = np.zeros(15 * m.n_tets)
    nv.hip_lib().fg_gauss_points(C.byref(m.mesh), nv.dptr(pg))
    src = leaf_cells(pg.reshape(-1, 5, 3)[np.any(a["tets"] == k, axis=1)].reshape(-1, 3), pos, level)
    tgt = leaf_cells(pos, pos, level)
    near = np.array([np.abs(src - t).max() <= 1 for t in tgt])
    phi, phiv = out["mixed"]
    broken = ~np.isfinite(phiv)
    # groups (the parents of the leaves) with targets of both kinds
    assert set(map(tuple, tgt[near] // 2)) & set(map(tuple, tgt[broken] // 2))
    ref = out["fp64"][1][near]
    assert np.all(np.isfinite(phiv[near])), np.sum(~np.isfinite(phiv[near]))
    assert np.abs(phiv[near] - ref).max() <= 1e-5 * np.abs(ref).max()
    assert np.abs(phi - out["fp64"][0]).max() <= 1e-4 * np.abs(out["fp64"][0]).max()
