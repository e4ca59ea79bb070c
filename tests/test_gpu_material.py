"""Material values per bond and particle: all particles at once, then single ones (first, last, inner), each against
the values of a context that holds them everywhere."""
import numpy as np
import pytest

import lpmgpu as G
from scenarios import hex_plate, sc_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", ["elastic", "damage", "j2", "hcf"])
@pytest.mark.parametrize("lattice,size", [("sc", 2), ("sc", 5), ("hex", (9, 8))])
def test_values(lattice, size, model):
    sc = lattice == "sc"
    xyz, _ = sc_cube(size) if sc else hex_plate(*size)
    n = len(xyz)
    print("[gpu] material", lattice, size, model, flush=True)
    kind = {"elastic": G.ELASTIC, "damage": G.ELASTIC_DAMAGE, "j2": G.J2, "hcf": G.HCF}[model]
    args = {"elastic": (1e-2,), "damage": (1e-3, 2.0, 10.0, 0.99), "j2": (300.0, 0.25, 2e3, 0.5, 1.0), "hcf": (5e-5, 2.019, 0.5)}[model]

    def make():
        return G.Context(G.SC3D if sc else G.HEXAGON2D, 0.5, kind, xyz, bonds="device")

    def setm(g, L, E, pid=-1):
        getattr(g, {"elastic": "set_elastic", "damage": "set_elastic_damage", "j2": "set_j2", "hcf": "set_hcf"}[model])(
            L, not sc, E, 0.3, *args, elmap_literal=0, pid=pid)

    def state(g):
        return {k: np.asarray(g.get(k)) for k in ("Kn", "Tv", "mat", "nonlocal_L")}

    g, a, b = make(), make(), make()
    setm(a, 1.5, 200e3)
    setm(b, 2.5, 70e3)
    A, B = state(a), state(b)
    ptr, split = a.get("bond_ptr"), a.get("bond_split")
    # all bonds of a layer alike (hexagon: of the plate), a layer's stiffness in proportion to E
    first = np.arange(ptr[-1]) < np.repeat(split, np.diff(ptr))
    for layer in (first, ~first):
        if layer.any():
            assert len(np.unique(A["Kn"][layer])) == 1 and A["Kn"][layer][0] > 0
    assert len(np.unique(A["Tv"])) == 1 and np.all(A["nonlocal_L"] == 1.5)
    np.testing.assert_allclose(A["Kn"] / B["Kn"], 200e3 / 70e3, rtol=1e-14)
    want_mat = {"elastic": [1e-2], "damage": [1e-3, 2.0, 0.99, 10.0], "j2": [200e3, 0.3, 300.0, 0.25, 2e3, 0.5, 0.0, 1.0],
                "hcf": [5e-5, 2.019, 0.5, 200e3, 0.3, 1.0, 1.108]}[model]
    m = A["mat"].reshape(n, -1)
    np.testing.assert_array_equal(m, np.tile(np.r_[want_mat, np.zeros(m.shape[1] - len(want_mat))], (n, 1)))
    setm(g, 1.5, 200e3)
    one = sorted({0, n // 2, n - 1})
    for i in one:
        setm(g, 2.5, 70e3, pid=i)
    got = state(g)
    bond = np.isin(np.repeat(np.arange(n), np.diff(ptr)), one)
    part = np.isin(np.arange(n), one)
    for k, sel in (("Kn", bond), ("Tv", bond), ("mat", np.repeat(part, m.shape[1])), ("nonlocal_L", part)):
        np.testing.assert_array_equal(got[k], np.where(sel, B[k], A[k]), err_msg=k)
    with pytest.raises(G.LPMError):
        setm(g, 1.0, 1.0, pid=n)
