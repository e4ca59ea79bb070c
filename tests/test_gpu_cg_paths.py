"""Paths of the persistent CG that depend on sizes: rows of Ac^-1 that do not fit the LDS, coarse ranges at and beyond
2,048 DoFs, a two-level solve longer than one launch, and FP32 iterates against the launched ones."""
import numpy as np
import pytest
import scipy.sparse as sp

import lpmgpu as G
from scenarios import faces, sc_cube
from test_gpu_cg_persistent import plate, solve, system
from test_gpu_coarse_groups import CELL, ensemble, preconditioned

pytestmark = pytest.mark.gpu


# aggregates of the specimens (three coarse DoFs each), and whether the solve is persistent
@pytest.mark.parametrize("sizes,ran", [
    ([(16, 16)] * 8, 1),  # 177 workgroups of 35 rows of 768 entries: 215 KB, read from memory
    ([(1, 1), (11, 31), (1, 1), (10, 34)], 1),  # coarse DoFs 1020-1031 span 1023 + 3 + 1020 = 2046
    ([(1, 1), (11, 31), (1, 1), (11, 31)], 0),  # 2049
])
def test_coarse_rows_and_ranges(sizes, ran):
    print("[gpu] persistent CG, coarse blocks", sizes, flush=True)
    xyz, agg, na, first, bonds = ensemble(sizes)
    g = G.Context(G.SQUARE2D, 0.5, G.ELASTIC, xyz, bonds=bonds)
    g.set_specimens(first)
    g.set_elastic(0.0, True, 69e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=1, precond=2, cg_tol=1e-12, cg_maxit=1, coarse_cells=CELL)
    pick = lambda f: np.concatenate([a + np.nonzero(f(xyz[a:b, 1]))[0] for a, b in zip(first[:-1], first[1:])])  # noqa: E731
    lo, hi = pick(lambda y: y == y.min()), pick(lambda y: y == y.max())
    g.apply_bc(g.load_step(disp=[(lo, "x", 0.0), (lo, "y", 0.0), (hi, "y", 0.001)]))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    b = np.asarray(g.get("residual"))
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    g.solve_linear_system()
    assert int(g.stat("cg_persistent")) == ran
    r, c, v = g.matrix()
    K = sp.csr_matrix((v, c, r), shape=(len(b), len(b)))
    u, worst = preconditioned(K, b, xyz, agg, na, np.concatenate([2 * lo, 2 * lo + 1, 2 * hi + 1]))
    x = u * (b @ u) / (u @ (K @ u))
    # the bound of test_gpu_coarse_groups.py
    assert np.linalg.norm(g.get("disp") - x) <= 2 * worst * 2.3e-16 * np.linalg.norm(x)


def test_two_level_longer_than_one_launch():
    print("[gpu] persistent CG: two-level, 1,500 iterations", flush=True)
    xyz = plate(60, 300)
    g, ls = system(G.SQUARE2D, xyz, 1, 2, 1e-300, True, cells=40)
    g.mode(cg_maxit=1500)
    x1, b, it1, ran = solve(g, ls, 1, xyz)
    x0, _, it0, _ = solve(g, ls, 0, xyz)
    assert ran == 1 and it1 == it0 == 1500
    # both have long converged: rounding, amplified by at most the condition number of K (below 1e6 here)
    assert np.linalg.norm(x1 - x0) <= 1e6 * 2.3e-16 * np.linalg.norm(x0)


@pytest.mark.parametrize("precond", [0, 1, 2])
@pytest.mark.parametrize("lattice,size", [("square", (37, 41)), ("square", (129, 128)), ("square", (512, 256)), ("sc", 11), ("sc", 26)])
def test_fp32_iterates(lattice, size, precond):
    print("[gpu] persistent CG, FP32 after 8 iterations,", lattice, size, "precond", precond, flush=True)
    two = lattice == "square"
    xyz = plate(*size) if two else sc_cube(size)[0]
    g, ls = system(G.SQUARE2D if two else G.SC3D, xyz, 0, precond, 1e-30, two, cells=max(4, size[0] // 12) if two else 6)
    g.mode(cg_maxit=8)
    x1, _, it1, ran = solve(g, ls, 1, xyz)
    x0, _, it0, _ = solve(g, ls, 0, xyz)
    assert ran == 1 and it1 == it0 == 8
    # one product rounds sums of up to 61 blocks: 61 * 2^-24 = 3.6e-6 relative; eight iterations, each at most
    # doubling what it is given, 1e-3
    assert np.linalg.norm(x1 - x0) <= 1e-3 * np.linalg.norm(x0)
