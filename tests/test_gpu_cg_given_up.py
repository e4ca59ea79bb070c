"""A persistent CG solve that gives up a wait: the context stays with launches until its settings change."""
import numpy as np
import pytest

import lpmgpu as G
from scenarios import faces, hex_plate

pytestmark = pytest.mark.gpu


def test_later_solves_do_not_wait_again():
    print("[gpu] persistent CG: given up once", flush=True)
    xyz, _ = hex_plate(60, 60)
    g = G.Context(G.HEXAGON2D, 0.5, G.ELASTIC, xyz, bonds="device")
    g.set_elastic(0.0, True, 69e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=1, precond=2, cg_tol=1e-9, cg_maxit=20000, cg_wait_ms=0)
    lo, hi = faces(xyz, 1)
    g.apply_bc(g.load_step(disp=[(lo, "x", 0.0), (lo, "y", 0.0), (hi, "y", 0.001)]))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    x = []
    for _ in range(3):
        g.solve_linear_system()
        x.append(np.array(g.get("disp")))
    assert int(g.stat("cg_persist_given_up")) == 1 and int(g.stat("cg_persistent")) == 0
    np.testing.assert_array_equal(x[0], x[1])
    np.testing.assert_array_equal(x[0], x[2])
    g.mode(cg_wait_ms=2000)  # tried again, and done
    g.solve_linear_system()
    assert int(g.stat("cg_persistent")) == 1 and int(g.stat("cg_persist_given_up")) == 1
    g.mode(cg_wait_ms=0)  # tried once more
    for _ in range(2):
        g.solve_linear_system()
    assert int(g.stat("cg_persist_given_up")) == 2
    g.mode(cg_persist=1)  # and again
    g.solve_linear_system()
    assert int(g.stat("cg_persist_given_up")) == 3
