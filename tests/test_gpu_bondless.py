"""Particles without any bond: an empty matrix, which every preconditioner takes."""
import numpy as np
import pytest

import lpmgpu as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("persist", [0, 1])
@pytest.mark.parametrize("precond", [0, 1, 2])
@pytest.mark.parametrize("lattice,n", [(G.SC3D, 5), (G.SC3D, 700), (G.HEXAGON2D, 70)])
def test_zero_solution(lattice, n, precond, persist, precision):
    print("[gpu] bondless", lattice, n, "precond", precond, "persist", persist, "precision", precision, flush=True)
    xyz = np.random.default_rng(n).random((n, 3)) * [40, 40, 40 if lattice == G.SC3D else 0]
    ptr = np.zeros(n + 1, dtype=np.int32)
    g = G.Context(lattice, 0.5, G.ELASTIC, xyz, bonds=(ptr, ptr[:n], np.zeros(0, dtype=np.int32)))
    g.set_elastic(0.0, lattice != G.SC3D, 69e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=precision, precond=precond, cg_persist=persist)
    g.apply_bc(g.load_step(disp=[(np.arange(2), "x", 0.0), (np.arange(3, 5), "y", 0.1)]))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    it, _ = g.solve_linear_system()
    assert it == 0
    np.testing.assert_array_equal(g.get("disp"), np.zeros(n * g.dim))
