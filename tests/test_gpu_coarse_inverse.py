"""The coarse inversion (32 pivots per launch, the next pivot block inverted by the launch before) at
block sizes around its tiles. A wrong entry of the inverse leaves the preconditioner indefinite or of a
different size than the coarse space needs, which the CG's iteration count shows at once."""
import numpy as np
import pytest
import scipy.sparse as sp
import scipy.sparse.linalg as spla

import lpmgpu as G
from scenarios import faces

pytestmark = pytest.mark.gpu


def plate(nx, ny):
    j, i = np.meshgrid(np.arange(ny), np.arange(nx), indexing="ij")
    return np.stack([i.ravel(), j.ravel(), np.zeros(nx * ny)], axis=1).astype(np.float64)


def host_iterations(K, b, xyz, nx_cells, ny_cells, fixed, tol):
    """Iterations of CG with D^-1 + P (P^T K P)^-1 P^T on the same rigid-body modes, in numpy."""
    n = len(xyz)
    ext = np.ptp(xyz, axis=0)
    cx = np.minimum(nx_cells - 1, (xyz[:, 0] / (ext[0] / nx_cells)).astype(int))
    cy = np.minimum(ny_cells - 1, (xyz[:, 1] / (ext[1] / ny_cells)).astype(int))
    agg = cy * nx_cells + cx
    na = nx_cells * ny_cells
    P = np.zeros((2 * n, 3 * na))
    for a in range(na):
        m = np.nonzero(agg == a)[0]
        d = xyz[m] - xyz[m].mean(axis=0)
        P[2 * m, 3 * a] = 1
        P[2 * m + 1, 3 * a + 1] = 1
        P[2 * m, 3 * a + 2] = -d[:, 1]
        P[2 * m + 1, 3 * a + 2] = d[:, 0]
    P[fixed] = 0
    Ac = np.linalg.pinv(P.T @ (K @ P), rcond=1e-9, hermitian=True)
    dinv = 1 / K.diagonal()
    M = spla.LinearOperator(K.shape, matvec=lambda r: dinv * r + P @ (Ac @ (P.T @ r)))
    count = []
    spla.cg(K, b, rtol=tol, atol=0, M=M, maxiter=2000, callback=lambda x: count.append(1))
    return len(count)


# coarse DoFs 3 (nx cells x ny cells): below, at and above one, two and three tiles of 32
@pytest.mark.parametrize("cells", [(1, 1), (5, 2), (11, 1), (7, 3), (11, 2), (8, 4), (11, 3)])
def test_block_sizes(cells):
    nx, ny = 8 * cells[0] + 1, 8 * cells[1] + 1
    print("[gpu] coarse inverse,", 3 * cells[0] * cells[1], "coarse DoFs", flush=True)
    xyz = plate(nx, ny)
    g = G.Context(G.SQUARE2D, 0.5, G.ELASTIC, xyz, bonds="device")
    g.set_elastic(0.0, True, 69e3, 0.3, 1.0, elmap_literal=0)
    tol = 1e-8
    g.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=1, precond=2, cg_tol=tol, cg_maxit=2000, coarse_cells=8)
    lo, hi = faces(xyz, 1)
    g.apply_bc(g.load_step(disp=[(lo, "x", 0.0), (lo, "y", 0.0), (hi, "y", 0.001)]))
    g.update_geometry()
    g.update_force_state()
    g.update_rr()
    b = g.get("residual")
    g.calc_stiffness()
    g.update_stiffness_disp_bc()
    it, _ = g.solve_linear_system()
    assert int(g.get_mode("ncoarse")) == 3 * cells[0] * cells[1]
    r, c, v = g.matrix()
    K = sp.csr_matrix((v, c, r), shape=(len(b), len(b)))
    assert np.linalg.norm(b - K @ g.get("disp")) <= 2 * tol * np.linalg.norm(b)
    fixed = np.concatenate([2 * lo, 2 * lo + 1, 2 * hi + 1])
    want = host_iterations(K, b, xyz, cells[0], cells[1], fixed, tol)
    assert abs(it - want) <= 3 + want // 10, (it, want)
