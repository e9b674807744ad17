"""The far field of the device FMM (multipoles evaluated at the targets, one source cell per lane) at
the edges of its tasks: groups of one target to more than three tiles of 16, list chunks of every
size from 1 to 64 entries (the last, partial chunk holds its entries once, twice or four times over),
both expansions in one pass (FP32; FP64 at order 4), one pass per set (FP64 at 6 and 8) and several
passes over columns (FP64 at 10), and the lower far degree. Device against the host evaluation of the
same plan: the same sums in another order and normalisation, so 1e-10 of the largest potential in
FP64. In mixed precision the multipoles of v are cut to degree 4 (or the far degree if that is lower):
the reference has the terms above it taken out. What FP32 leaves (2^-24 = 6e-8 in each coefficient and
product, of either sign) is 2e-7 of the largest potential of u and 4e-7 of v, held to 2e-6 for both."""
import ctypes as C

import numpy as np
import pytest

from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh
from test_fmm import charged, fmm_ref

CASES = [((6, 5, 4), 4, 0), ((9, 7, 5), 256, 0), ((30, 4, 2), 32, 0), ((14, 13, 12), 1500, 0), ((20, 10, 3), 16, 1),
         ((11, 11, 11), 100, 1)]


def far_terms(xyz, q, tgt, level, near_degrees, far_degrees):
    """What the multipole-to-target evaluation of a plan of that leaf level adds at targets tgt = (all, index)
    by the degrees of near_degrees = (first, last), and of far_degrees for the entries at distance 3 of
    all the leaves that they serve: sums of q r^n / R^(n+1) P_n about each source's cell."""
    pos, at = tgt
    lo, hi = np.minimum(xyz.min(0), pos.min(0)), np.maximum(xyz.max(0), pos.max(0))
    half = 0.5 * (hi - lo).max() * (1 + 1e-9)
    corner = 0.5 * (lo + hi) - half
    out = np.zeros(len(at))
    for l in (level, level - 1):
        if l < 2:
            continue
        w = 2 * half / 2**l
        sc, tc = np.floor((xyz - corner) / w).astype(int), np.floor((pos - corner) / w).astype(int)
        cen = corner + (sc + 0.5) * w
        for k, i in enumerate(at):
            d = np.abs(sc - tc[i]).max(1)
            pair = (d >= 2) & (np.abs(sc // 2 - tc[i] // 2).max(1) <= 1)
            s, far = sc[pair], d[pair] >= 3
            if l == level:
                octants = 2 * (tc[i] // 2) + np.stack(np.meshgrid([0, 1], [0, 1], [0, 1]), -1).reshape(-1, 3)
                far = ~np.any(np.abs(s[:, None] - octants).max(2) == 2, axis=1)
            a, b = xyz[pair] - cen[pair], pos[i] - cen[pair]
            r, R = np.linalg.norm(a, axis=1), np.linalg.norm(b, axis=1)
            c = (a * b).sum(1) / (np.maximum(r, 1e-300) * R)
            p0, p1, f = np.ones(len(c)), c, q[pair] / R
            for n in range(max(near_degrees[1], far_degrees[1]) + 1):
                keep = np.where(far, far_degrees[0] <= n <= far_degrees[1], near_degrees[0] <= n <= near_degrees[1])
                out[k] += (keep * f * p0).sum()
                f = f * r / R
                p0, p1 = p1, ((2 * n + 3) * c * p1 - (n + 1) * p0) / (n + 2)
    return out


def far_cut(xyz, q, pot, tgt, level, order, far, cut):
    """The potential pot of a plan with its multipole evaluations cut to a degree."""
    return pot[tgt[1]] - far_terms(xyz, q, tgt, level, (cut + 1, order), (min(cut, far) + 1, far))


@pytest.mark.parametrize("cells,leaf", [((6, 5, 4), 256), ((9, 7, 5), 64)])
def test_far_cut(cells, leaf):
    """far_cut against the host FMM: on plans without translations an order-6 plan cut to degree 4 is the
    order-4 one, and an order-8 plan whose far entries lose degrees 6 to 8 the one with far degree 5."""
    m = HostMesh.cuboid(tuple(6.0 * c for c in cells), cells, jitter=0.1, seed=4)
    m.prepare({"volume": dict(Ms=8e5)})
    p, u, v = charged(m)
    xyz, qu, qv = p.sources()
    xyz = xyz.reshape(-1, 3)
    pos = m.arrays()["pos"]
    tgt = pos, np.arange(0, len(pos), 7)
    six, _, L = fmm_ref(xyz, qu, qv, pos, 6, leaf, far=6)
    four = fmm_ref(xyz, qu, qv, pos, 4, leaf, far=4)[0]
    assert L <= 3
    assert np.abs(far_cut(xyz, qu, six, tgt, L, 6, 6, 4) - four[tgt[1]]).max() <= 1e-12 * np.abs(four).max()
    eight, low = (fmm_ref(xyz, qu, qv, pos, 8, leaf, far=f)[0] for f in (8, 5))
    got = eight[tgt[1]] - far_terms(xyz, qu, tgt, L, (9, 8), (6, 8))
    assert np.abs(got - low[tgt[1]]).max() <= 1e-12 * np.abs(low).max()
    if L == 3:  # with four leaves a side no entry is far from all that it serves
        assert np.abs(eight - low).max() >= 1e-6 * np.abs(low).max()


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
    xyz, pos = xyz.reshape(-1, 3), m.arrays()["pos"]
    pu, pv, L = fmm_ref(xyz, qu, qv, pos, order, leaf, far=far)
    ref = (pu + cu) / (4 * np.pi), (pv + cv) / (4 * np.pi)
    at = np.unique(np.linspace(0, len(pos) - 1, 120).astype(int))
    cut = (far_cut(xyz, qv, pv, (pos, at), L, order, far, 4) + cv[at]) / (4 * np.pi)
    for prec in ("fp64", "mixed"):
        g = Engine(m.mesh, demag="fmm", fmm_order=order, fmm_leaf=leaf, fmm_far_order=far, precision=prec)
        i = g.fmm_info()
        assert i["leaf_level"] == L and i["m2p_pairs"] <= i["m2p_slots"]
        g.set_state(nv.FG_BOTH, u=u, v=v)
        g.calc_demag()
        phi, phiv = g.get_state(nv.FG_NEXT)[2:]
        g.close()
        err = [np.abs(a - b).max() / np.abs(b).max() for a, b in zip((phi, phiv), ref)]
        if prec == "fp64":
            assert max(err) <= 1e-10, err
        else:
            err[1] = np.abs(phiv[at] - cut).max() / np.abs(ref[1]).max()
            assert max(err) <= 2e-6, err


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
