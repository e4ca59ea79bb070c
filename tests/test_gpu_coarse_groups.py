"""The coarse inversion over groups of different block sizes, in fused steps and in three kernels per step (the line
lies at 2,048 tiles of 32 x 32), with dropped and dead coarse DoFs: the first CG iterate, alpha M^-1 b, against numpy."""
import numpy as np
import pytest
import scipy.sparse as sp

import lpmgpu as G

pytestmark = pytest.mark.gpu

CELL = 4  # lattice spacings per aggregate


def plate(cx, cy):
    nx, ny = CELL * cx + 1, CELL * cy + 1
    j, i = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    x = np.stack([i.ravel(), j.ravel(), np.zeros(nx * ny)], axis=1).astype(np.float64)
    cell = np.minimum(cy - 1, x[:, 1] // CELL) * cx + np.minimum(cx - 1, x[:, 0] // CELL)
    return x, cell.astype(int)


def ensemble(sizes):
    parts, cells, first, bp, bs, p2, na = [], [], [0], [np.zeros(1, np.int64)], [], [], 0
    for cx, cy in sizes:
        x, cell = plate(cx, cy)
        a, b, c = (np.asarray(v, dtype=np.int64) for v in G.build_bonds(G.SQUARE2D, 0.5, x))
        off = int(bp[-1][-1])
        bp.append(a[1:] + off)
        bs.append(b + off)
        p2.append(c + first[-1])
        parts.append(x)
        cells.append(cell + na)
        na += cx * cy
        first.append(first[-1] + len(x))
    bonds = tuple(np.concatenate(v).astype(np.int32) for v in (bp, bs, p2))
    return np.vstack(parts), np.concatenate(cells), na, first, bonds


def preconditioned(K, b, xyz, agg, na, fixed):
    """M^-1 b with M^-1 = D^-1 + P (P^T K P)^+ P^T, block by block, and the largest condition number of a block's
    range times its size."""
    n = len(xyz)
    size = np.bincount(agg, minlength=na)
    cen = np.stack([np.bincount(agg, xyz[:, k], na) / size for k in range(2)], axis=1)
    d = xyz[:, :2] - cen[agg]
    i = np.arange(n)
    P = sp.csr_matrix((np.concatenate([np.ones(2 * n), -d[:, 1], d[:, 0]]),
                       (np.concatenate([2 * i, 2 * i + 1, 2 * i, 2 * i + 1]),
                        np.concatenate([3 * agg, 3 * agg + 1, 3 * agg + 2, 3 * agg + 2]))), shape=(2 * n, 3 * na))
    free = np.ones(2 * n)
    free[fixed] = 0
    P = sp.diags(free) @ P
    Ac = (P.T @ (K @ P)).toarray()
    y, t, worst = np.zeros(3 * na), P.T @ b, 0.0
    lo = 0
    while lo < 3 * na:  # the diagonal blocks
        hi = lo + 3
        while hi < 3 * na and (np.any(Ac[lo:hi, hi:]) or np.any(Ac[hi:hi + 3, lo:hi])):
            hi += 3
        w, V = np.linalg.eigh(0.5 * (Ac[lo:hi, lo:hi] + Ac[lo:hi, lo:hi].T))
        keep = w > 1e-9 * max(w.max(), 1.0)
        if keep.any():  # else no DoF of the block is free
            y[lo:hi] = V[:, keep] @ ((V[:, keep].T @ t[lo:hi]) / w[keep])
            worst = max(worst, (hi - lo) * w.max() / w[keep].min())
        lo = hi
    return b / K.diagonal() + P @ y, worst


# aggregates of the specimens, three coarse DoFs each: one, two and three tiles of a block; blocks that end at a tile's
# edge; the last one with 768 DoFs four times, 2,331 tiles, which run as three kernels a step
SIZES = [[(1, 1), (2, 5), (7, 3), (11, 3)], [(8, 4), (1, 2), (16, 4)], [(11, 1)], [(16, 16)] * 2 + [(3, 2)],
         [(16, 16), (3, 2), (16, 16), (6, 4), (16, 16), (11, 3), (16, 16), (1, 1)]]


@pytest.mark.parametrize("persist", [0, 1])
@pytest.mark.parametrize("dropped", [False, True])
@pytest.mark.parametrize("sizes", SIZES)
def test_first_iterate(sizes, dropped, persist):
    print("[gpu] coarse groups", sizes, "dropped", dropped, "persist", persist, flush=True)
    xyz, agg, na, first, bonds = ensemble(sizes)
    g = G.Context(G.SQUARE2D, 0.5, G.ELASTIC, xyz, bonds=bonds)
    if len(sizes) > 1:
        g.set_specimens(first)
    g.set_elastic(0.0, True, 69e3, 0.3, 1.0, elmap_literal=0)
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=1, precond=2, cg_tol=1e-12, cg_maxit=1,
           coarse_cells=CELL, cg_persist=persist)
    disp, fixed = [], []
    held = np.zeros(len(xyz), dtype=bool)
    for a, b in zip(first[:-1], first[1:]):
        held[a:b] = xyz[a:b, 1] == 0
    if dropped:  # in every third aggregate one particle stays free (its rotation is a combination of the translations),
        # in every fifth none
        for k in range(0, na, 3):
            held[np.nonzero(agg == k)[0][1:]] = True
        for k in range(1, na, 5):
            held[agg == k] = True
    top = np.concatenate([a + np.nonzero(xyz[a:b, 1] == xyz[a:b, 1].max())[0] for a, b in zip(first[:-1], first[1:])])
    top = top[~held[top]]
    held = np.nonzero(held)[0]
    disp = [(held, "x", 0.0), (held, "y", 0.0), (top, "y", 0.001)]
    fixed = np.concatenate([2 * held, 2 * held + 1, 2 * top + 1])
    g.apply_bc(g.load_step(disp=disp))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    b = np.asarray(g.get("residual"))
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    it, _ = g.solve_linear_system()
    assert it == 1 and int(g.get_mode("ncoarse")) == 3 * na
    r, c, v = g.matrix()
    K = sp.csr_matrix((v, c, r), shape=(len(b), len(b)))
    u, worst = preconditioned(K, b, xyz, agg, na, fixed)
    x = u * (b @ u) / (u @ (K @ u))
    # an inverse without pivoting of a positive definite block of n DoFs is off by n cond eps relative to its largest
    # entry at most; the same for the sums that form the block
    assert np.linalg.norm(g.get("disp") - x) <= 2 * worst * 2.3e-16 * np.linalg.norm(x)
