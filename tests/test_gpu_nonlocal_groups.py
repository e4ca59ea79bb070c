"""The cell-grid nonlocal search (eight lanes per particle) against the test of every pair in numpy, at particle
counts around eight and thirty-two, cutoffs from none accepted to all, different ones per particle, uneven clouds."""
import numpy as np
import pytest

import lpmgpu as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 8, 9, 31, 33, 257, 1001])
@pytest.mark.parametrize("shape", [(1, 1, 1), (40, 0.5, 0.5), (3, 20, 1), (2, 2, 30)])
def test_lists(n, shape):
    rng = np.random.default_rng(n)
    xyz = rng.random((n, 3)) * shape
    xyz[rng.random(n) < 0.3] *= 0.1  # crowded cells
    L = rng.choice([0.0, 0.2, 0.7, 1.0], n)
    print("[gpu] nonlocal groups", n, shape, flush=True)
    ptr = np.zeros(n + 1, dtype=np.int32)
    g = G.Context(G.SC3D, 0.5, G.ELASTIC, xyz, bonds=(ptr, ptr[:n], np.zeros(0, dtype=np.int32)))
    g.set("nonlocal_L", L)
    g.search_nonlocal(1.5)
    d = xyz[:, None] - xyz[None]
    # the kernel's sum order: x^2 + y^2 + z^2
    hit = np.sqrt(d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1] + d[..., 2] * d[..., 2]) < (1.5 * L)[:, None]
    np.testing.assert_array_equal(g.get("nl_ptr"), np.r_[0, np.cumsum(hit.sum(1))])
    np.testing.assert_array_equal(np.asarray(g.get("nl_idx"))[:hit.sum()], np.nonzero(hit)[1])
