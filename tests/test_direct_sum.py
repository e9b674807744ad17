"""The direct demag sum at the edges of its split into target blocks and source shares: one node more
or less than a block of 256 or 512 targets, source counts that are no multiple of 4, 64 or 256, and
batches whose instances meet inside a block. Against the oracle's plain sum; the two add the same
terms in different orders, so they differ by at most S roundings of the sum of magnitudes."""
import ctypes as C

import numpy as np
import pytest

import oracle
from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh

TRI = np.array([[1 / 3] * 3, [.6, .2, .2], [.2, .6, .2], [.2, .2, .6]])
TRI_W = np.array([-27 / 96, 25 / 96, 25 / 96, 25 / 96])


def mesh(cells, seed):
    m = HostMesh.cuboid(tuple(4.0 * c for c in cells), cells, jitter=0.1, seed=seed)
    return m.prepare({"volume": dict(Ms=8e5)})


def unit(n, seed):
    u = np.random.default_rng(seed).normal(size=(n, 3))
    return u / np.linalg.norm(u, axis=1, keepdims=True)


def magnitudes(m, u):
    """sum_s |q_s| / |x_i - y_s| / 4 pi per node, and the number of sources."""
    a = m.arrays()
    X = a["pos"][a["tets"]]
    J = X[:, 1:] - X[:, :1]
    g = np.linalg.inv(J).transpose(0, 2, 1)
    da = np.concatenate([-g.sum(1, keepdims=True), g], axis=1)
    pg = np.zeros(15 * m.n_tets)
    nv.hip_lib().fg_gauss_points(C.byref(m.mesh), nv.dptr(pg))
    w = np.linalg.det(J)[:, None] * np.array([2 / 15] + [3 / 40] * 4)
    q = np.abs(8e5 * w * np.einsum("tak,tak->t", da, u[a["tets"]])[:, None])
    P = a["pos"][a["tris"]]
    cr = np.cross(P[:, 1] - P[:, 0], P[:, 2] - P[:, 0])
    n = cr / np.linalg.norm(cr, axis=1, keepdims=True)
    s = np.einsum("fak,fk->fa", u[a["tris"]], n) @ TRI.T
    qf = np.abs(a["dMs"][:, None] * np.linalg.norm(cr, axis=1)[:, None] * TRI_W * s)
    y = np.concatenate([pg.reshape(-1, 3), np.einsum("ga,fak->fgk", TRI, P).reshape(-1, 3)])
    r = np.linalg.norm(a["pos"][:, None] - y[None], axis=2)
    return (1.0 / r) @ np.concatenate([q.ravel(), qf.ravel()]) / (4 * np.pi), len(y)


def check(m, u, phi):
    p = oracle.Problem(m.mesh, tol=1e-10, max_iter=100)
    p.set_state(nv.FG_BOTH, u=u)
    p.calc_demag()
    ref = p.get_state(nv.FG_NEXT)[2]
    A, S = magnitudes(m, u)
    # plus 8 for each term's own roundings and the triangles' self terms
    assert np.all(np.abs(phi - ref) <= (S + 8) * 2.0**-53 * A), np.max(np.abs(phi - ref) / A)


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(1, 1, 1), (4, 16, 2), (7, 7, 3), (7, 7, 7), (18, 8, 2), (19, 8, 2), (10, 9, 9)])
def test_direct_sum_at_block_edges(cells):
    m = mesh(cells, 1)
    u = unit(m.n_nodes, 2)
    g = Engine(m.mesh)
    g.set_state(nv.FG_BOTH, u=u, v=-3.0 * u)
    g.calc_demag()
    _, _, phi, phiv = g.get_state(nv.FG_NEXT)
    check(m, u, phi)
    # v = -3 u: the same charges scaled by a factor that is exact up to one rounding each
    assert np.allclose(phiv, -3.0 * phi, rtol=1e-9, atol=1e-11 * np.abs(phi).max())


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[(2, 2, 2), (3, 5, 1), (1, 1, 1)], [(7, 7, 3), (7, 7, 3)], [(9, 9, 5), (2, 1, 1), (6, 6, 6)]])
def test_direct_sum_batch(sizes):
    ms = [mesh(c, 3 + k) for k, c in enumerate(sizes)]
    us = [unit(m.n_nodes, 20 + k) for k, m in enumerate(ms)]
    g = Engine.batch([m.mesh for m in ms])
    g.set_state(nv.FG_BOTH, u=np.concatenate(us))
    g.calc_demag()
    phi = g.get_state(nv.FG_NEXT)[2]
    off, _ = g.layout()
    for k, (m, u) in enumerate(zip(ms, us)):
        check(m, u, phi[off[k]:off[k + 1]])


def touching_tets(n_pairs):
    """Pairs of tetrahedra whose second one has a corner at the first one's centroid, a Gauss point (both
    exact in binary: the centroid takes a quarter of each corner), far apart from one another."""
    pos, tets = [], []
    for k in range(n_pairs):
        o = np.array([0.0, 0.0, 64.0 * k])
        tets += [np.arange(4) + 8 * k, np.arange(4) + 8 * k + 4]
        pos += [o, o + [4, 0, 0], o + [0, 4, 0], o + [0, 0, 4], o + [1, 1, 1], o + [9, 1, 1], o + [1, 9, 1], o + [1, 1, 9]]
    pos, tets = np.array(pos, float) * 2.0**-30, np.array(tets, np.int32)
    treg, vol, surf = np.zeros(len(tets), np.int32), (nv.VolumeRegion * 1)(), (nv.SurfaceRegion * 1)()
    vol[0].Ms, vol[0].Ae, vol[0].alpha = 8e5, 1e-11, 0.1
    m = nv.Mesh()
    m.n_nodes, m.n_tets, m.n_tris, m.n_vol_regions, m.n_surf_regions = len(pos), len(tets), 0, 1, 1
    m.pos = pos.ctypes.data_as(C.POINTER(C.c_double))
    m.tet_nodes, m.tet_region = (x.ctypes.data_as(C.POINTER(C.c_int32)) for x in (tets, treg))
    m.vol, m.surf = C.cast(vol, C.POINTER(nv.VolumeRegion)), C.cast(surf, C.POINTER(nv.SurfaceRegion))
    return m, (pos, tets, treg, vol, surf)


@pytest.mark.gpu
@pytest.mark.parametrize("n_pairs,batch", [(2, 1), (80, 1), (2, 3)])
def test_source_at_a_node(n_pairs, batch):
    """A node of a body that overlaps another one can lie on a Gauss point: its potential is infinite, as
    the plain sum has it (no number without charge), and the other nodes' are not touched."""
    m, own = touching_tets(n_pairs)
    u = unit(m.n_nodes, 4)
    v = unit(m.n_nodes, 5)
    if n_pairs > 2:
        v[8:16] = 0  # no charge of v at the second pair's node
    p = oracle.Problem(m, tol=1e-10, max_iter=100)
    p.set_state(nv.FG_BOTH, u=u, v=v)
    p.calc_demag()
    g = Engine.batch([m] * batch) if batch > 1 else Engine(m)
    g.set_state(nv.FG_BOTH, u=np.tile(u, (batch, 1)), v=np.tile(v, (batch, 1)))
    g.calc_demag()
    at = np.arange(4, m.n_nodes, 8)
    for out, ref in zip(g.get_state(nv.FG_NEXT)[2:], p.get_state(nv.FG_NEXT)[2:]):
        assert not np.isfinite(ref[at]).any() and np.isfinite(np.delete(ref, at)).all()
        for phi in out.reshape(batch, -1):
            assert np.array_equal(phi[at], ref[at], equal_nan=True)
            assert np.allclose(np.delete(phi, at), np.delete(ref, at), rtol=1e-11, atol=1e-12 * np.nanmax(np.abs(np.delete(ref, at))))
