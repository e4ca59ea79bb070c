"""Persistent CG solves of several contexts at the same time, one thread each: small grids that run side by side, grids
that fill the device and wait for each other, and both together. Each gives its own bits and none gives up."""
import threading

import numpy as np
import pytest

import lpmgpu as G
from scenarios import faces, sc_cube

pytestmark = pytest.mark.gpu


def context(n, precision, precond):
    xyz, _ = sc_cube(n)
    g = G.Context(G.SC3D, 0.5, G.ELASTIC, xyz, bonds="device")
    g.set_elastic(0.0, False, 200e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=precision, precond=precond, cg_tol=1e-30, cg_maxit=40)
    lo, hi = faces(xyz, 2)
    g.apply_bc(g.load_step(disp=[(lo, a, 0.0) for a in "xyz"] + [(hi, "z", 0.001)]))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    return g


@pytest.mark.parametrize("sizes", [(9, 9, 10, 11, 12, 12), (27, 30, 26), (40, 8, 27, 8, 12)])
def test_side_by_side(sizes):
    print("[gpu] persistent CG in threads, SC", sizes, flush=True)
    ctx = [context(n, k % 2, (2, 0, 2)[k % 3]) for k, n in enumerate(sizes)]
    want = []
    for g in ctx:
        g.solve_linear_system()
        want.append(np.array(g.get("disp")))
    wrong = []

    def work(k):
        for _ in range(15):
            ctx[k].solve_linear_system()
            if not np.array_equal(ctx[k].get("disp"), want[k]):
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(ctx))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    assert all(int(g.stat("cg_persistent")) == 16 and int(g.stat("cg_persist_given_up")) == 0 for g in ctx)
