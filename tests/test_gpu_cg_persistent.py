"""The persistent CG (mode cg_persist) against the launched CG and the matrix itself: sizes at the
edges of its slices and workgroups, every preconditioner, both precisions, an ensemble, solves longer
than one launch, and the fallback when a wait inside the kernel is given up."""
import numpy as np
import pytest
import scipy.sparse as sp

import lpmgpu as G
import oracle as O
from scenarios import faces, hex_plate, sc_cube

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)


def plate(nx, ny):
    """Square lattice plate, nx x ny particles."""
    j, i = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    return np.stack([i.ravel(), j.ravel(), np.zeros(nx * ny)], axis=1).astype(np.float64)


def system(lattice, xyz, precision, precond, tol, plane_stress, cells=4):
    g = G.Context(lattice, 0.5, G.ELASTIC, xyz, bonds="device")
    g.set_elastic(0.0, plane_stress, 200e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=precision, precond=precond, cg_tol=tol,
           cg_maxit=20000, coarse_cells=cells)
    ax = g.dim - 1
    lo, hi = faces(xyz, ax)
    disp = [(lo, "xyz"[k], 0.0) for k in range(g.dim)] + [(hi, "xyz"[ax], 0.001)]
    return g, g.load_step(disp=disp)


def solve(g, ls, persist, xyz):
    """One linear solve from the undeformed state; returns (x, iterations, persistent solves)."""
    g.mode(cg_persist=persist)
    g.reset_stats()
    g.set("xyz", xyz)
    g.apply_bc(ls)
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    b = g.get("residual")
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    it, _ = g.solve_linear_system()
    return g.get("disp"), b, it, int(g.stat("cg_persistent"))


def residual(g, x, b):
    r, c, v = g.matrix()
    K = sp.csr_matrix((v, c, r), shape=(len(b), len(b)))
    return np.linalg.norm(b - K @ x) / np.linalg.norm(b)


# particles: below one slice, one slice, one more, a partly filled last slice; one slice per
# workgroup up to 256 slices (16,384 rows), two from there; the largest (8 slices each: 131,072 rows)
PLATES = [(7, 9), (8, 8), (13, 5), (37, 41), (128, 128), (129, 128), (200, 231), (512, 256)]


@pytest.mark.parametrize("precision", [0, 1])
@pytest.mark.parametrize("precond", [0, 1, 2])
@pytest.mark.parametrize("nx,ny", PLATES)
def test_plates(nx, ny, precond, precision):
    # FP64: the recurrence's residual follows the true one to far below 1e-9. FP32: the true residual
    # is that of an FP32 solution, whose rounding (2^-24 per entry, times |K||x|/|b|, below 1e3 for these
    # loads) stays under the tolerance of 1e-2.
    tol = 1e-2 if precision == 0 else 1e-9
    say("[gpu] persistent CG, square", nx, "x", ny, "precond", precond, "precision", precision)
    xyz = plate(nx, ny)
    g, ls = system(G.SQUARE2D, xyz, precision, precond, tol, True, cells=max(4, nx // 12))
    x1, b, it1, ran = solve(g, ls, 1, xyz)
    assert ran == 1
    assert residual(g, x1, b) <= 2 * tol
    x2, _, it2, _ = solve(g, ls, 1, xyz)
    assert it1 == it2
    np.testing.assert_array_equal(x1, x2)  # a fixed order of every sum
    x0, _, it0, ran = solve(g, ls, 0, xyz)
    assert ran == 0
    assert abs(it1 - it0) <= 2 + it0 // 20
    assert residual(g, x0, b) <= 2 * tol


@pytest.mark.parametrize("precision,idx16", [(0, 1), (0, 0), (1, 1), (1, 0)])
@pytest.mark.parametrize("n", [4, 11, 26])
def test_cubes(n, precision, idx16):
    tol = 1e-2 if precision == 0 else 1e-9
    say("[gpu] persistent CG, SC", n, "precision", precision, "idx16", idx16)
    xyz, _ = sc_cube(n)
    g, ls = system(G.SC3D, xyz, precision, 2, tol, False, cells=6)
    g.mode(spmv_idx16=idx16)
    x1, b, it1, ran = solve(g, ls, 1, xyz)
    x0, _, it0, _ = solve(g, ls, 0, xyz)
    assert ran == 1 and abs(it1 - it0) <= 2 + it0 // 20
    assert residual(g, x1, b) <= 2 * tol


def test_one_row_more_is_launched():
    say("[gpu] persistent CG: one slice above its range")
    xyz = plate(512, 257)
    g, ls = system(G.SQUARE2D, xyz, 0, 0, 1e-1, True)
    assert solve(g, ls, 1, xyz)[3] == 0


def test_longer_than_one_launch():
    # 1,024 iterations a launch: the state passes through memory twice here
    say("[gpu] persistent CG: 2,500 iterations")
    xyz = plate(60, 300)
    g, ls = system(G.SQUARE2D, xyz, 1, 0, 1e-300, True)
    g.mode(cg_maxit=2500)
    x1, b, it1, ran = solve(g, ls, 1, xyz)
    x0, _, it0, _ = solve(g, ls, 0, xyz)
    assert ran == 1 and it1 == it0 == 2500
    # both have long converged: the difference is rounding, amplified by at most the condition
    # number of K (below 1e6 here)
    assert np.linalg.norm(x1 - x0) <= 1e6 * 2.3e-16 * np.linalg.norm(x0)


def test_zero_right_hand_side_and_no_iterations():
    say("[gpu] persistent CG: zero right-hand side, cg_maxit 0")
    xyz, _ = sc_cube(6)
    g, ls = system(G.SC3D, xyz, 1, 2, 1e-9, False)
    still = g.load_step(disp=[(faces(xyz, 2)[0], a, 0.0) for a in "xyz"])
    x, b, it, ran = solve(g, still, 1, xyz)
    assert ran == 1 and it == 0 and not x.any() and not b.any()
    g.mode(cg_maxit=0)
    x, b, it, ran = solve(g, ls, 1, xyz)
    assert ran == 1 and it == 0 and not x.any() and b.any()


def test_given_up_wait_is_solved_by_launches():
    # cg_wait_ms = 0: a workgroup that finds a slot empty once leaves, all others follow, and the
    # solve is repeated launch by launch with the same bits as without the persistent kernel
    say("[gpu] persistent CG: waits given up")
    xyz, _ = hex_plate(60, 60)
    g, ls = system(G.HEXAGON2D, xyz, 1, 2, 1e-9, True)
    x0 = solve(g, ls, 0, xyz)[0]
    g.mode(cg_wait_ms=0)
    x1, _, _, ran = solve(g, ls, 1, xyz)
    assert ran == 0
    np.testing.assert_array_equal(x0, x1)
    g.mode(cg_wait_ms=2000)
    assert solve(g, ls, 1, xyz)[3] == 1


def test_ensemble_groups():
    # specimens of 1 to 9 aggregates, several of them inside one workgroup's rows
    say("[gpu] persistent CG: ensemble with one coarse block per specimen")
    parts, first, bp, bs, p2 = [], [0], [np.zeros(1, np.int64)], [], []
    for nx, ny in [(6, 7), (30, 20), (5, 9), (12, 33), (41, 25), (7, 7)]:
        x, _ = hex_plate(nx, ny)
        a, b, c = (np.asarray(v, dtype=np.int64) for v in G.build_bonds(G.HEXAGON2D, 0.5, x))
        off = int(bp[-1][-1])
        bp.append(a[1:] + off)
        bs.append(b + off)
        p2.append(c + first[-1])
        first.append(first[-1] + len(x))
        parts.append(x)
    xyz = np.vstack(parts)
    res = []
    for persist in (1, 0):
        g = G.Context(G.HEXAGON2D, 0.5, G.ELASTIC, xyz, bonds=tuple(np.concatenate(v).astype(np.int32) for v in (bp, bs, p2)))
        g.set_specimens(first)
        g.set_elastic(0.0, True, 69e3, 0.3, 1.0, elmap_literal=0)
        g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=1, precond=2, coarse_cells=10, cg_tol=1e-12,
               tol_NR=1e-10, max_NR_iter=40, cg_maxit=20000, cg_persist=persist)
        disp = []
        for x, off in zip(parts, first):
            ids, y = np.arange(off, off + len(x)), x[:, 1]
            lo, hi = ids[y < y.min() + 1e-6], ids[y > y.max() - 1e-6]
            disp += [(lo, "x", 0.0), (lo, "y", 0.0), (hi, "y", 0.001)]
        g.update_geometry()
        g.update_force_state()
        assert g.solve_step_static(g.load_step(disp=disp), -1)
        assert (g.stat("cg_persistent") > 0) == bool(persist)
        res.append((g.get("xyz"), g.specimen_stat("newton_iters")))
    np.testing.assert_array_equal(res[0][1], res[1][1])
    u0, u1 = res[1][0] - xyz.ravel(), res[0][0] - xyz.ravel()
    assert np.linalg.norm(u1 - u0) <= 1e-9 * np.linalg.norm(u0)
