"""A new context: what every state array holds, by model and by the way the bonds come (lists, device search)."""
import numpy as np
import pytest

import lpmgpu as G
from scenarios import hex_plate, sc_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bonds", [None, "device"])
@pytest.mark.parametrize("model", [G.ELASTIC, G.ELASTIC_DAMAGE, G.J2, G.HCF])
@pytest.mark.parametrize("lattice,size", [("sc", 2), ("sc", 7), ("hex", (9, 31))])
def test_initial_state(lattice, size, model, bonds):
    xyz, _ = sc_cube(size) if lattice == "sc" else hex_plate(*size)
    n = len(xyz)
    print("[gpu] setup state", lattice, size, "n", n, "model", model, bonds, flush=True)
    g = G.Context(G.SC3D if lattice == "sc" else G.HEXAGON2D, 0.5, model, xyz, bonds=bonds)
    for f in ("xyz", "xyz_initial", "xyz_last"):
        np.testing.assert_array_equal(np.asarray(g.get(f)).reshape(-1, 3), xyz, err_msg=f)
    for f in ("Pin", "Pex", "stress", "damage", "damage_last", "damage_visual", "Ddot_local", "Ddot_nonlocal", "nonlocal_L",
              "dLe_total", "TdLe_total", "cs_sum", "type", "disp_constraint", "dLe", "dLp", "dLp_last", "bstrain", "Kn", "Tv",
              "bforce", "bforce_last", "bdamage", "bdamage_last"):
        assert not np.any(g.get(f)), f
    sv, last, mat = (np.asarray(g.get(f)).reshape(n, -1) for f in ("state_var", "state_var_last", "mat"))
    want_sv, want_mat = np.zeros_like(sv), np.zeros_like(mat)
    if model == G.HCF:
        want_sv[:, 1] = 2**31 - 1
        want_mat[:, 5], want_mat[:, 6] = 1.0, 1.108
    for a, b in ((sv, want_sv), (last, want_sv), (mat, want_mat)):
        np.testing.assert_array_equal(a, b)
    dis = np.asarray(g.get("dis_initial"))
    i = np.repeat(np.arange(n), np.diff(g.get("bond_ptr")))
    d = np.linalg.norm(xyz[i] - xyz[g.get("bond_p2")], axis=1)
    np.testing.assert_allclose(dis, d, rtol=4e-16, atol=0)
    np.testing.assert_array_equal(g.get("dis"), dis)
    np.testing.assert_array_equal(g.get("dis_last"), dis)
    g.close()
