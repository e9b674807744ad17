"""The spin solver's phases past one pass of their grids (more than 65,536 nodes, 262,144 unknowns):
diffusion alone on a bar against the closed form of tests/test_spin_accumulation.py, whose P1 error at
this cell size is below 1e-3; and a second solve, whose first chunk of iterations has the length of the
first one's, gives the same field; and a solve after one that failed."""
import time

import numpy as np
import pytest

from feellgood_amd.engine import SpinSolver
from test_electrostatic import bar
from test_spin_accumulation import JN, MUB_E, S0, SURF, UP, vol


@pytest.mark.gpu
def test_diffusion_on_a_fine_bar():
    m, own, pos = bar(0.0, cells=(60, 38, 38))
    assert m.n_nodes > 87381
    u = np.tile([0.0, 0.0, 1.0], (m.n_nodes, 1))
    sp = SpinSolver(m, [vol(), vol()], SURF, np.zeros(m.n_nodes), tol=1e-10, max_iter=3000)
    s, info = sp.solve(u, accumulate=False)
    assert info.status == 0 and info.iterations > 16
    x = pos[:, 0] - pos[:, 0].min()
    L, lsf = np.ptp(pos[:, 0]), 10e-9
    s1 = -JN * MUB_E * np.array(UP)
    ref = (np.outer(np.sinh((L - x) / lsf), S0) + np.outer(np.sinh(x / lsf), s1)) / np.sinh(L / lsf)
    assert np.abs(s - ref).max() <= 1e-3 * np.abs(ref).max()
    again, info2 = sp.solve(u, accumulate=False)
    assert info2.iterations == info.iterations and np.array_equal(again, s)


@pytest.mark.gpu
def test_solve_after_a_failed_one():
    """A long solve that did not converge (magnetizations far from unit length, of which the longest solve
    is taken) leaves nothing behind: the next one gives the same field, and takes about as long, as one
    after a solve that converged. With the failed one's iterations queued ahead of it, empty launches
    took more than twice its own time."""
    m, own, pos = bar(0.0, cells=(20, 6, 6), ms=(8e5, 8e5))
    u = np.tile([0.0, 0.0, 1.0], (m.n_nodes, 1))
    sp = SpinSolver(m, [vol(), vol()], SURF, np.zeros(m.n_nodes), tol=1e-8, max_iter=2000)
    tries = [(sp.solve(k * u, accumulate=False)[1], k) for k in (30.0, 50.0, 100.0, 200.0, 300.0, 500.0, 1000.0, 2000.0)]
    long = max((i.iterations, k) for i, k in tries if i.status != 0)
    assert long[0] >= 150
    ref, info = sp.solve(0 * u, accumulate=False)
    assert info.status == 0 and info.iterations < 60
    t = {False: [], True: []}
    for k in range(10):
        failed = k % 2 == 1
        sp.solve(long[1] * u if failed else 0 * u, accumulate=False)
        t0 = time.perf_counter()
        s, again = sp.solve(0 * u, accumulate=False)
        t[failed].append(time.perf_counter() - t0)
        assert again.iterations == info.iterations and np.array_equal(s, ref)
    assert min(t[True]) <= 1.5 * min(t[False]), t
