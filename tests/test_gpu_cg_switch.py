"""A caller that switches the preconditioner from solve to solve: the persistent CG prepares once for each kind."""
import numpy as np
import pytest

import lpmgpu as G
from scenarios import faces, sc_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("n", [5, 27])
def test_two_plans(n, precision):
    print("[gpu] preconditioner switched, SC", n, "precision", precision, flush=True)
    xyz, _ = sc_cube(n)
    g = G.Context(G.SC3D, 0.5, G.ELASTIC, xyz, bonds="device")
    g.set_elastic(0.0, False, 200e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=precision, cg_tol=1e-3 if precision == 0 else 1e-9,
           cg_maxit=20000)
    lo, hi = faces(xyz, 2)
    g.apply_bc(g.load_step(disp=[(lo, a, 0.0) for a in "xyz"] + [(hi, "z", 0.001)]))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    got = {}
    for _ in range(3):
        for precond in (2, 0, 1):
            g.mode(precond=precond)
            g.solve_linear_system()
            x = np.array(g.get("disp"))
            np.testing.assert_array_equal(x, got.setdefault(precond, x))
    assert int(g.stat("cg_persistent")) == 9
    assert int(g.stat("cg_persist_plans")) == 2


def test_contexts_of_different_coarse_size_in_turn():
    # the LDS limit belongs to the kernel: a context with a small coarse space leaves it large enough for the other
    print("[gpu] persistent CG: contexts with 8 and 125 aggregates in turn", flush=True)
    ctx = []
    for n, cells in [(9, 4), (26, 5)]:
        xyz, _ = sc_cube(n)
        g = G.Context(G.SC3D, 0.5, G.ELASTIC, xyz, bonds="device")
        g.set_elastic(0.0, False, 200e3, 0.3, 1.0, elmap_literal=0)
        g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=1, precond=2, cg_tol=1e-9, cg_maxit=20000, coarse_cells=cells)
        lo, hi = faces(xyz, 2)
        g.apply_bc(g.load_step(disp=[(lo, a, 0.0) for a in "xyz"] + [(hi, "z", 0.001)]))
        g.update_geometry()
        g.update_force_state()
        g.update_rr()
        g.calc_stiffness()
        g.update_stiffness_disp_bc()
        ctx.append(g)
    for _ in range(3):
        for g in reversed(ctx):
            g.solve_linear_system()
    assert [int(g.get_mode("ncoarse")) for g in ctx] == [48, 750]
    assert [int(g.stat("cg_persistent")) for g in ctx] == [3, 3]
