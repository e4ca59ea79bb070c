"""The cell-grid nonlocal search on both sides of its choice of lanes per particle (65,536 particles; 36 items per range of
three cells) against the test of every pair: uneven clouds, short and long lists."""
import numpy as np
import pytest

import lpmgpu as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("L", [0.5, 1.0, 3.2])
@pytest.mark.parametrize("n,two", [(65536, False), (65537, False), (65539, True), (70001, False)])
def test_lists(n, two, L):
    print("[gpu] nonlocal lanes", n, "2D" if two else "3D", "L", L, flush=True)
    rng = np.random.default_rng(n)
    size = (260, 260, 0) if two else (40, 41, 40)
    xyz = rng.random((n, 3)) * size
    some = rng.random(n) < 0.05
    xyz[some] = xyz[some] * 0.3 + 0.1  # a denser corner
    ptr = np.zeros(n + 1, dtype=np.int32)
    g = G.Context(G.HEXAGON2D if two else G.SC3D, 0.5, G.ELASTIC, xyz, bonds=(ptr, ptr[:n], np.zeros(0, dtype=np.int32)))
    g.set("nonlocal_L", L * rng.choice([0.0, 0.6, 1.0], n))
    got = []
    for cells in (0, 1):
        g.mode(nl_cells=cells)
        g.search_nonlocal(1.5)
        p = np.array(g.get("nl_ptr"))
        got.append((p, np.array(g.get("nl_idx"))[:p[-1]]))
    np.testing.assert_array_equal(got[1][0], got[0][0])
    np.testing.assert_array_equal(got[1][1], got[0][1])
