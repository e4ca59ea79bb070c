"""The sparsity pattern (sorted, each particle once) against numpy: lattices, rings of bonds up to the limit of 512
candidates of a row, particles without bonds; beyond the limit the context is refused."""
import numpy as np
import pytest

import lpmgpu as G
from scenarios import hex_plate, sc_cube

pytestmark = pytest.mark.gpu


def ring(n, offsets, alone=0):
    """n particles, each bonded to those `offsets` to both sides, and `alone` ones without bonds."""
    k = np.array([-o for o in offsets] + list(offsets))
    p2 = (np.arange(n)[:, None] + k) % n
    deg = len(k)
    ptr = np.r_[np.arange(n + 1) * deg, np.full(alone, n * deg)]
    split = np.r_[ptr[1:n + 1], ptr[n + 1:]]  # all bonds in layer 0
    xyz = np.random.default_rng(2).random((n + alone, 3)) * 50
    return xyz, (ptr, split, np.sort(p2, axis=1).ravel())


def check(g):
    n = g.n
    ptr, split, p2 = (np.asarray(g.get(k)) for k in ("bond_ptr", "bond_split", "bond_p2"))
    rows = []
    for i in range(n):
        c = [p2[ptr[i]:ptr[i + 1]]]
        for b in range(ptr[i], ptr[i + 1]):
            k = p2[b]
            c.append(p2[ptr[k]:split[k]] if b < split[i] else p2[split[k]:ptr[k + 1]])
        rows.append(np.unique(np.concatenate(c)))
    np.testing.assert_array_equal(g.get("conn_ptr"), np.r_[0, np.cumsum([len(r) for r in rows])])
    np.testing.assert_array_equal(g.get("conn_idx"), np.concatenate(rows))


@pytest.mark.parametrize("lattice,size", [("sc", 2), ("sc", 6), ("hex", (3, 4)), ("hex", (9, 15))])
def test_lattices(lattice, size):
    xyz, _ = sc_cube(size) if lattice == "sc" else hex_plate(*size)
    print("[gpu] pattern", lattice, size, flush=True)
    check(G.Context(G.SC3D if lattice == "sc" else G.HEXAGON2D, 0.5, G.ELASTIC, xyz, bonds="device"))


@pytest.mark.parametrize("n,offsets,alone", [
    (700, (1, 4, 13, 32, 71, 124, 218, 259, 301, 317, 330), 3),  # 22 bonds, 506 candidates, few alike
    (4096, (64, 128, 192, 256, 320, 384, 448, 512), 0),  # ids a constant apart
    (65, (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11), 1),
    (3, (1,), 0),
])
def test_rings(n, offsets, alone):
    print("[gpu] pattern ring", n, offsets, alone, flush=True)
    xyz, bonds = ring(n, offsets, alone)
    check(G.Context(G.SC3D, 0.5, G.ELASTIC, xyz, bonds=bonds))


def test_too_many_candidates_refused():
    xyz, bonds = ring(600, tuple(range(1, 13)))  # 24 bonds, 600 candidates
    with pytest.raises(G.LPMError, match="two-hop candidates"):
        G.Context(G.SC3D, 0.5, G.ELASTIC, xyz, bonds=bonds)
