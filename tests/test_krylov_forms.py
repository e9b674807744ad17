"""The solver's kernels in each of their forms (a whole solve in one block of 256, 512 or 1,024 threads;
four lanes per row; a lane per row in one pass of the grid; a lane per row in several passes) at the
edges between them: 256, 512 and 1,024 nodes, 32,768 and 262,144, and the next mesh after each (and
65,536, the most that four lanes per row could take). A batch's
blocks with the lifted vector in LDS (up to 6,400 nodes in the largest instance) and in memory. The accepted solution's residual is recomputed in
numpy from the assembled system; BiCGSTAB tests its recursive residual, which drifts from the true
one by rounding only, so it is held to twice the tolerance. In FP32 iterations the accepted residual is
the true one."""
import numpy as np
import pytest
import scipy.sparse as sp

from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh

TOL = 1e-9


@pytest.mark.gpu
@pytest.mark.parametrize("krylov", ["fp64", "mixed"])
@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 2, 6), (7, 7, 3), (7, 7, 7), (8, 7, 7), (15, 7, 7), (16, 7, 7), (31, 31, 31), (31, 31, 32), (31, 31, 63), (32, 31, 63), (63, 63, 63), (64, 63, 63)])
def test_solution_at_form_edges(cells, krylov):
    m = HostMesh.cuboid(tuple(3.0 * c for c in cells), cells, jitter=0.1, seed=5)
    m.prepare({"volume": dict(Ms=8e5, Ae=1.3e-11, alpha=0.1)})
    rng = np.random.default_rng(1)
    u = np.array([1.0, 0.4, 0.0]) + rng.uniform(-0.2, 0.2, size=(m.n_nodes, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    g = Engine(m.mesh, tol=TOL, max_iter=1000, krylov=krylov)
    g.set_state(nv.FG_BOTH, u=u)
    dt = 2e-14
    g.base_projection(0.3)
    g.prepare_elements(np.array([1e4, 2e4, -3e3]), dt, 1.05)
    failed, info = g.solve(dt)
    assert not failed and info.iterations > 0
    rp, col, val, rhs = g.system()
    A = sp.csr_matrix((val, col, rp), shape=(len(rhs), len(rhs)))
    x = g.solution()
    assert np.linalg.norm(rhs - A @ x) <= 2 * TOL * np.linalg.norm(rhs)
    assert info.rhs_norm == pytest.approx(np.linalg.norm(rhs), rel=1e-12)
    v = np.sqrt((x.reshape(-1, 2) ** 2).sum(1).max())
    assert info.v_max == pytest.approx(1.76085962784e11 * nv.MU0 * v, rel=1e-12)


@pytest.mark.gpu
@pytest.mark.parametrize("block", [256, 512, 1024])
@pytest.mark.parametrize("sizes", [[(15, 19, 19), (2, 2, 2)], [(2, 1, 1), (15, 19, 20), (7, 7, 7)]])
def test_batch_blocks(sizes, block):
    ms = []
    for k, c in enumerate(sizes):
        m = HostMesh.cuboid(tuple(3.0 * n for n in c), c, jitter=0.1, seed=5 + k)
        ms.append(m.prepare({"volume": dict(Ms=8e5, Ae=1.3e-11, alpha=0.1)}))
    assert max(m.n_nodes for m in ms) in (6400, 6720)
    rng = np.random.default_rng(1)
    n = sum(m.n_nodes for m in ms)
    u = np.array([1.0, 0.4, 0.0]) + rng.uniform(-0.2, 0.2, size=(n, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    g = Engine.batch([m.mesh for m in ms], tol=TOL, max_iter=1000, batch_solver="persistent", batch_block=block)
    g.set_state(nv.FG_BOTH, u=u)
    g.base_projection(0.3)
    g.prepare_elements(np.array([1e4, 2e4, -3e3]), 2e-14, 1.05)
    failed, info = g.solve(2e-14)
    assert not failed and info.iterations > 0
    rp, col, val, rhs = g.system()
    r = rhs - sp.csr_matrix((val, col, rp), shape=(n * 2, n * 2)) @ g.solution()
    off = 2 * g.layout()[0]
    for a, b in zip(off[:-1], off[1:]):
        assert np.linalg.norm(r[a:b]) <= 2 * TOL * np.linalg.norm(rhs[a:b])


@pytest.mark.gpu
@pytest.mark.parametrize("krylov", ["fp64", "mixed"])
@pytest.mark.parametrize("cells", [(31, 31, 63), (47, 47, 47), (63, 63, 63), (64, 63, 63)])
def test_iterations_queued_past_the_end_read_no_rows(cells, krylov):
    """The second solve of a system starts from the first one's solution and ends at its first test, so
    the two iterations queued behind it have nothing to do: their products take about as long as an empty
    launch between two events (6 us, against 14 to 50 for the one that forms the first residual)."""
    m = HostMesh.cuboid(tuple(3.0 * c for c in cells), cells, jitter=0.1, seed=5)
    m.prepare({"volume": dict(Ms=8e5, Ae=1.3e-11, alpha=0.1)})
    rng = np.random.default_rng(1)
    u = np.array([1.0, 0.4, 0.0]) + rng.uniform(-0.2, 0.2, size=(m.n_nodes, 3))
    u /= np.linalg.norm(u, axis=1, keepdims=True)
    g = Engine(m.mesh, tol=TOL, max_iter=1000, krylov=krylov, profile=True)
    g.set_state(nv.FG_BOTH, u=u)
    g.base_projection(0.3)
    g.prepare_elements(np.array([1e4, 2e4, -3e3]), 2e-14, 1.05)
    assert not g.solve(2e-14)[0] and not g.solve(2e-14)[0]
    g.reset_kernel_stats()
    for _ in range(5):
        failed, info = g.solve(2e-14)
        assert not failed and info.iterations == 0
    t = {k: ms / n for k, (n, ms) in g.kernel_stats().items() if n}
    empty = min(t.values())
    assert t["spmv"] - empty <= 0.3 * (t["spmv_r0"] - empty), t
