"""The force kernels (a workgroup takes eight consecutive particles) against the oracle, bit for bit, at
particle counts around the group size, in 2D and 3D, with broken and damaged bonds."""
import numpy as np
import pytest

import oracle as O
from scenarios import Pair, hex_plate, sc_cube

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("model", [O.ELASTIC, O.ELASTIC_DAMAGE])
@pytest.mark.parametrize("lattice,size", [("hex", (3, 4)), ("hex", (4, 4)), ("hex", (9, 7)), ("sc", 2), ("sc", 3), ("sc", 7)])
def test_forces_bitwise(lattice, size, model):
    rng = np.random.default_rng(5)
    sc = lattice == "sc"
    xyz, box = sc_cube(size) if sc else hex_plate(*size)
    n = len(xyz)
    print("[gpu] forces", lattice, size, "n", n, "n % 8 =", n % 8, flush=True)
    p = Pair(O.SC3D if sc else O.HEXAGON2D, 0.5, model, xyz, box)
    if model == O.ELASTIC:
        p.set_elastic(0.0, not sc, 200e3, 0.3, 1.0)
    else:
        p.set_elastic_damage(1.0, not sc, 200e3, 0.3, 1e-3, 1.0, 10.0, 0.99)
    x = xyz + 2e-3 * rng.standard_normal(xyz.shape) * ([1, 1, 1] if sc else [1, 1, 0])
    bd = rng.choice([0.0, 0.25, 1.0], p.o.info("nbonds"))
    for f, v in (("xyz", x), ("bdamage", bd), ("damage", np.linspace(0, 0.5, n))):
        p.o.setd(f, v)
        p.g.set(f, v)
    p.o.update_geometry()
    p.o.update_force_state()
    p.g.update_geometry()
    p.g.update_force_state()
    for f in ("dis", "dLe", "bstrain", "cs", "bforce", "bdamage", "dLe_total", "TdLe_total", "cs_sum", "Pin", "stress",
              "damage_visual"):
        np.testing.assert_array_equal(p.g.get(f), p.o.getd(f), err_msg=f)
