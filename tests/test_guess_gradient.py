"""Weight gradients of the learned guess at the edges of their node chunks: one node short of and past
a tile of 64, and chunks of several tiles (beyond 64 x 512 nodes). Against the oracle's FP64 backward pass on the recorded features: the products and sums are FP32, a
unit's relative error is that of its 64-term sums (64 x 2^-24 = 4e-6) through two layers."""
import numpy as np
import pytest

import oracle
from feellgood_amd import native as nv
from feellgood_amd.engine import Engine
from feellgood_amd.mesh import HostMesh
from test_guess import adjacency, field, initial_u


@pytest.mark.gpu
@pytest.mark.parametrize("cells", [(1, 1, 1), (2, 2, 6), (3, 3, 3), (10, 2, 1), (12, 4, 1), (40, 40, 19)])
def test_weight_gradient_chunks(cells):
    m = HostMesh.cuboid(tuple(4.0 * c for c in cells), cells, jitter=0.1, seed=2)
    m.prepare({"volume": dict(Ms=8e5, alpha=0.1)})
    mag = np.ones(m.n_nodes, dtype=np.int32)
    n = m.n_nodes
    e = Engine(m.mesh, tol=1e-10, max_iter=1000)
    rng = np.random.default_rng(6)
    u = initial_u(m)
    v = rng.normal(size=(n, 3)) * 2e9
    e.set_state(nv.FG_BOTH, u=u, v=v - np.sum(v * u, axis=1, keepdims=True) * u)
    e.guess_init(1)
    p = (rng.normal(size=nv.FG_GUESS_NPARAM) * 0.15).astype(np.float32)
    p[-nv.FG_GUESS_NSCALE:] = [1 / 3e4, 1 / 2e9, 5e8, 1 / 1e7]
    e.guess_set(p)
    e.base_projection(0.2)
    e.prepare_elements(field(0.4), 2e-14, 1.05)
    assert not e.solve(2e-14)[0]
    grad, loss, _ = e.guess_gradient()
    ptr, idx = adjacency(m)
    _, L, _, go = oracle.guess_eval(p, e.guess_features(), ptr, idx, mag, e.get_state(nv.FG_NEXT)[1])
    assert loss == pytest.approx(L, rel=1e-5)
    assert np.linalg.norm(grad - go) <= 1e-5 * np.linalg.norm(go)
