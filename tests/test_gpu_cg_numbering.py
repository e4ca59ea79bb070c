"""Where the persistent CG hands over to the launches because of the particles' numbering, and that both give the
solution: lattices in their own order, shuffled, and shuffled within windows."""
import numpy as np
import pytest
import scipy.sparse as sp

import lpmgpu as G
from scenarios import faces, sc_cube

pytestmark = pytest.mark.gpu


def box(nx, ny, nz):
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    return np.stack([i.ravel(), j.ravel(), k.ravel()], axis=1).astype(np.float64)


def shuffled(x, window):
    rng = np.random.default_rng(3)
    return np.concatenate([rng.permutation(x[a:a + window]) for a in range(0, len(x), window)])


# persistent: for (precond 0, precond 2) in (FP32, FP64)
CASES = [
    ("own order", box(36, 36, 36), 0, [[1, 1], [1, 1]]),
    ("own order, columns beyond int16", box(150, 150, 3), 0, [[1, 1], [1, 1]]),
    ("shuffled, small", sc_cube(12)[0], 10**9, [[1, 1], [1, 1]]),
    ("shuffled, int16 columns", box(31, 31, 31), 10**9, [[1, 0], [1, 0]]),
    ("shuffled in windows, int16 columns", box(30, 30, 30), 256, [[1, 1], [1, 1]]),
    ("shuffled", box(36, 36, 36), 10**9, [[0, 0], [0, 0]]),
    ("shuffled, few reads of u", box(190, 190, 1), 10**9, [[1, None], [1, None]]),
]


@pytest.mark.parametrize("name,xyz,window,want", CASES, ids=[c[0] for c in CASES])
def test_route_and_solution(name, xyz, window, want):
    two = not np.ptp(xyz[:, 2])
    if window:
        xyz = shuffled(xyz, window)
    g = G.Context(G.SQUARE2D if two else G.SC3D, 0.5, G.ELASTIC, xyz, bonds="device")
    g.set_elastic(0.0, two, 200e3, 0.3, 1.0, elmap_literal=0)
    lo, hi = faces(xyz, 0)
    disp = [(lo, "xyz"[k], 0.0) for k in range(g.dim)] + [(hi, "x", 0.001)]
    for precision in (0, 1):
        tol = 1e-2 if precision == 0 else 1e-9
        g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=precision, cg_tol=tol, cg_maxit=20000)
        g.set("xyz", xyz)
        g.apply_bc(g.load_step(disp=disp))
        g.update_geometry()
        g.update_force_state()
        g.update_rr()
        b = np.array(g.get("residual"))
        g.calc_stiffness()
        g.update_stiffness_disp_bc()
        r, c, v = g.matrix()
        K = sp.csr_matrix((v, c, r), shape=(len(b), len(b)))
        for k, precond in enumerate((0, 2)):
            print("[gpu] numbering:", name, "precision", precision, "precond", precond, flush=True)
            g.mode(precond=precond)
            g.reset_stats()
            g.solve_linear_system()
            assert want[precision][k] in (None, int(g.stat("cg_persistent")))
            # the recurrence's residual follows the true one: the tolerance in FP64; in FP32 twice it (rounding
            # 2^-24 times |K||x|/|b|, below 1e3 for these loads, stays under it)
            assert np.linalg.norm(b - K @ g.get("disp")) <= 2 * tol * np.linalg.norm(b)
            g.set("xyz", xyz)  # the solve has moved the particles
