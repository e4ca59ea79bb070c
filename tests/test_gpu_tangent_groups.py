"""The Jacobian product kernels (a workgroup takes eight consecutive particles) against the formulas in
numpy, at particle counts around the group size, in 2D and 3D, with broken, half-broken and damaged bonds."""
import numpy as np
import pytest

import lpmgpu as G
from scenarios import hex_plate, sc_cube

pytestmark = pytest.mark.gpu


def reference(g, v, w):
    n, dim = g.n, g.dim
    ptr, split, p2, opp = (g.get(k) for k in ("bond_ptr", "bond_split", "bond_p2", "opp"))
    cs, dis, Kn, Tv = g.get("cs").reshape(-1, 3), g.get("dis"), g.get("Kn"), g.get("Tv")
    bd, f = g.get("bdamage"), g.get("bforce")
    i = np.repeat(np.arange(n), np.diff(ptr))
    slot = 2 * i + (np.arange(len(p2)) >= split[i])
    broken = np.abs(bd - 1) < 1e-6
    V, W = np.zeros((n, 3)), np.zeros((n, 3))
    V[:, :dim], W[:, :dim] = v.reshape(n, dim), w.reshape(n, dim)

    def per_particle(b):
        out = np.zeros((n, 3))
        np.add.at(out, i, b)
        return out[:, :dim].ravel()

    dd = V[i] - V[p2]
    ddis = np.where(broken, 0, (cs * dd).sum(1))
    inv = np.where(broken, 0, 1 / dis)
    tot = np.bincount(slot, ddis, 2 * n)
    df = (2 * Kn * ddis + 2 * Tv * tot[slot]) * (1 - bd)
    jv = per_particle((dd - cs * ddis[:, None]) * (inv * 0.5 * (f + f[opp]))[:, None] + cs * (0.5 * (df + df[opp]))[:, None])
    t = 0.5 * ((cs * W[i]).sum(1) + (cs[opp] * W[p2]).sum(1))
    T = np.bincount(slot, 2 * Tv * t * (1 - bd), 2 * n)
    c = np.where(broken, 0, 2 * Kn * t * (1 - bd) + T[slot])
    h = 0.5 * (f + f[opp])
    a, ao = h * inv, h * np.where(broken[opp], 0, 1 / dis[opp])
    co = cs[opp]
    y = per_particle(a[:, None] * (W[i] - cs * (cs * W[i]).sum(1)[:, None]) -
                     ao[:, None] * (W[p2] - co * (co * W[p2]).sum(1)[:, None]) + c[:, None] * cs - c[opp][:, None] * co)
    return jv, y


@pytest.mark.parametrize("damage", [False, True])
@pytest.mark.parametrize("lattice,size", [("hex", (2, 1)), ("hex", (3, 4)), ("hex", (9, 7)), ("sc", 2), ("sc", 3), ("sc", 7)])
def test_products_match_the_formulas(lattice, size, damage):
    rng = np.random.default_rng(11)
    xyz, _ = sc_cube(size) if lattice == "sc" else hex_plate(*size)
    g = G.Context(G.SC3D if lattice == "sc" else G.HEXAGON2D, 0.5, G.ELASTIC_DAMAGE, xyz)
    print("[gpu] tangent", lattice, size, "n", g.n, "n % 8 =", g.n % 8, flush=True)
    g.set_elastic_damage(0.0, lattice == "hex", 69e3, 0.3, 1e9, 1.0, 1.0, 1.0, elmap_literal=0)
    nb = g.size("nbonds")
    g.set("Kn", g.get("Kn") * rng.uniform(0.5, 1.5, nb))
    g.set("Tv", g.get("Tv") * rng.uniform(0.5, 1.5, nb))
    if damage:
        bd = rng.uniform(0, 0.9, nb)
        bd[rng.random(nb) < 0.2] = 1.0  # a bond may be broken and its reverse not
        g.set("bdamage", bd)
    x = xyz + 1e-3 * rng.normal(size=xyz.shape) * ([1, 1, 1] if lattice == "sc" else [1, 1, 0])
    g.set("xyz", x)
    g.update_geometry()
    g.update_force_state()
    v, w = rng.normal(size=g.dim * g.n), rng.normal(size=g.dim * g.n)
    jv, y = reference(g, v, w)
    # sums of at most 32 bonds of three products each: 1e-14 of the largest entry covers their rounding
    for got, want in ((g.force_jvp(v), jv), (g.force_vjp(w), y)):
        assert np.max(np.abs(got - want)) <= 1e-13 * max(np.max(np.abs(want)), 1e-30)
