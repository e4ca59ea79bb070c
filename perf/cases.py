"""Timed cases of the load-step path: what they are, how their inputs are made, one pass of each, and
what the pass returns in 64 bits (plain torch, no code of the library).

Every case goes through lpmgpu.Context, the binding of the C ABI. Lattices, solver settings and
materials are those of the repository's own benchmark and tests; sizes run from about a thousand
particles to the benchmark's 262,144. The kinds:

  forces   new positions from the caller -> geometry, bond forces, Pin, stress, residual norms
  tangent  Jacobian products of the internal force, forward (jvp) and transposed (vjp)
  linear   one linear solve from scratch: assembly, Dirichlet elimination, CG
  path     a converged state restored, then `steps` static load steps (Newton + CG each)
  fatigue  an ensemble of HCF dogbones: static start, then `steps` simulated load cycles
  adjoint  gradient of a linear objective of the equilibrium in every bond's Kn, Tv and damage
  setup    a new particle system: bond search, sparsity pattern, nonlocal neighbour lists
"""
import functools
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "lpm-mac_amd"))

import lpmgpu as G  # noqa: E402

LATTICE = {"square": G.SQUARE2D, "hex": G.HEXAGON2D, "sc": G.SC3D, "fcc": G.FCC3D, "bcc": G.BCC3D}
DIM = {"square": 2, "hex": 2, "sc": 3, "fcc": 3, "bcc": 3}
RADIUS = {"square": 0.5, "hex": 0.5, "sc": 0.5, "fcc": 0.5 / math.sqrt(2), "bcc": math.sqrt(3) / 4}
BONDS = {"square": 8, "hex": 12, "sc": 18, "fcc": 18, "bcc": 14}  # of an interior particle
BLOCKS = {"square": 17, "hex": 31, "sc": 61, "fcc": 61, "bcc": 41}  # of an interior matrix row


def listed():
    def case(name, kind, lattice, nx, ny, nz=1, **kw):
        return dict(dict(name=name, kind=kind, lattice=lattice, nx=nx, ny=ny, nz=nz, model="elastic", precision=0, precond=2,
                         steps=1, rotated=False), **kw)

    return [
        # the smallest call: a caller that moves a small plate itself and asks for the forces
        case("forces hex 31x33", "forces", "hex", 31, 33),
        # the same for a rotated crystal (ragged surfaces) of ordinary size
        case("forces fcc 20 rotated", "forces", "fcc", 20, 20, 20, rotated=True),
        # forward and transposed Jacobian products, as a matrix-free solver or a sensitivity uses them
        case("tangent sc 30x31x29", "tangent", "sc", 30, 31, 29),
        # the reference's own algorithm on the 10k-particle plate: one FP64 Jacobi CG solve
        case("linear hex 100 fp64", "linear", "hex", 100, 115, precision=1, precond=0),
        # one load step of a small cube with the mixed-precision solver: launches and waits count
        case("step sc 12", "path", "sc", 12, 12, 12),
        # one load step all in FP64, odd sizes, the third 3D lattice
        case("step bcc 21x20x19 fp64", "path", "bcc", 21, 20, 19, precision=1),
        # the headline workload: 64^3 cube in tension, quadratic predictor, kept coarse space
        case("path sc 64", "path", "sc", 64, 64, 64, steps=6),
        # crystal plasticity: a rotated FCC crystal through yield
        case("path fcc 24 J2", "path", "fcc", 24, 24, 24, model="j2", steps=3, rotated=True),
        # edge-cracked plate with bonds breaking during the load steps
        case("path hex 200 crack", "path", "hex", 200, 231, model="crack", steps=3),
        # parameter calibration: eight dogbones of uneven size through fatigue cycles together
        case("fatigue 8 dogbones", "fatigue", "hex", 90, 0, model="hcf", steps=2),
        # gradients in every bond parameter at the converged state of a plate
        case("adjoint hex 120x141 fp64", "adjoint", "hex", 120, 141, precision=1),
        # a new specimen: bonds, pattern and nonlocal lists searched on the device
        case("setup sc 41x40x39", "setup", "sc", 41, 40, 39),
    ]


def draw(rng):
    kind = rng.choice(["forces", "tangent", "linear", "path", "path", "path", "fatigue", "adjoint", "setup"])
    model, steps, rotated = "elastic", 1, False
    if kind == "path":
        model = rng.choice(["elastic", "elastic", "j2", "crack"])
        steps = rng.randint(1, 4)
    if kind == "fatigue":
        lattice, model, steps = "hex", "hcf", rng.randint(1, 3)
    elif model == "crack":
        lattice = "hex"
    elif model == "j2":
        lattice, rotated = "fcc", True
    else:
        lattice = rng.choice(["hex", "square", "sc", "sc", "fcc", "bcc"])
    # particles, spread over the logarithm; what takes many solves stays below the largest listed
    top = {"forces": 150e3, "tangent": 150e3, "linear": 60e3, "path": 130e3, "fatigue": 5e3, "adjoint": 50e3, "setup": 130e3}[kind]
    low = 8e3 if model == "crack" else 1e3  # a short crack in a small plate runs through it at once
    n = math.exp(rng.uniform(math.log(low), math.log(top)))
    if DIM[lattice] == 2:
        nx = max(12, round(math.sqrt(n / 1.15) * rng.uniform(0.8, 1.2)))
        ny, nz = (0 if kind == "fatigue" else max(12, round(n / nx))), 1
    else:
        per = {"sc": 1, "fcc": 4, "bcc": 2}[lattice]
        nx = max(6, round((n / per) ** (1 / 3) * rng.uniform(0.9, 1.1)))
        ny = max(6, round(math.sqrt(n / per / nx) * rng.uniform(0.9, 1.1)))
        nz = max(6, round(n / per / nx / ny))
        if rotated:
            ny = nz = nx
    precision = rng.choice([0, 0, 1]) if kind in ("path", "adjoint") and model == "elastic" else int(kind == "linear")
    precond = 0 if kind == "linear" else 2
    return dict(kind=kind, lattice=lattice, nx=nx, ny=ny, nz=nz, model=model, precision=precision, precond=precond, steps=steps,
                rotated=rotated)


# ---------------------------------------------------------------- particles and bonds
@functools.lru_cache(maxsize=4)
def _lattice(lattice, nx, ny, nz, rotated):
    """Positions (x fastest, then y, then z) and integer lattice coordinates."""
    if lattice in ("sc", "square"):
        i, j, k = np.meshgrid(np.arange(nx), np.arange(ny), np.arange(nz if lattice == "sc" else 1), indexing="ij")
        ic = np.stack([a.transpose(2, 1, 0).ravel() for a in (i, j, k)], axis=1)
        return ic.astype(np.float64), ic
    if lattice == "hex":  # half-spacing units in x, rows of alternating length
        ic = np.concatenate([np.stack([2 * np.arange(nx - j % 2) + j % 2, np.full(nx - j % 2, j), np.zeros(nx - j % 2, int)], axis=1)
                             for j in range(ny)])
        return ic * np.array([0.5, math.sqrt(3) / 2, 0.0]), ic
    # fcc, bcc: half-edge units of the unit cell
    if not rotated:
        grid = [np.arange(2 * m + 1) for m in (nx, ny, nz)]
    else:  # a box cut out of a crystal in a general orientation
        a = int(math.ceil(math.sqrt(3) * max(nx, ny, nz))) + 2
        grid = [np.arange(-a, a + 1)] * 3
    k, j, i = np.meshgrid(grid[2], grid[1], grid[0], indexing="ij")
    even = (i + j + k) % 2 == 0 if lattice == "fcc" else ((i - j) % 2 == 0) & ((j - k) % 2 == 0)
    ic = np.stack([i[even], j[even], k[even]], axis=1)
    x = 0.5 * ic
    if rotated:
        q, _ = np.linalg.qr(np.random.default_rng(7).normal(size=(3, 3)))
        x = x @ q.T + 0.5 * np.array([nx, ny, nz])
        keep = np.all((x >= 0) & (x <= np.array([nx, ny, nz])), axis=1)
        x, ic = x[keep], ic[keep]
    return np.ascontiguousarray(x), ic


NEIGHBOURS = {  # integer offsets of the first and of the second layer
    "square": ([(1, 0, 0), (0, 1, 0)], [(1, 1, 0), (1, -1, 0)]),
    "hex": ([(2, 0, 0), (1, 1, 0), (-1, 1, 0)], [(3, 1, 0), (-3, 1, 0), (0, 2, 0)]),
    "sc": ([(1, 0, 0), (0, 1, 0), (0, 0, 1)], [(1, 1, 0), (1, -1, 0), (1, 0, 1), (1, 0, -1), (0, 1, 1), (0, 1, -1)]),
    "fcc": ([(1, 1, 0), (1, -1, 0), (1, 0, 1), (1, 0, -1), (0, 1, 1), (0, 1, -1)], [(2, 0, 0), (0, 2, 0), (0, 0, 2)]),
    "bcc": ([(1, 1, 1), (1, 1, -1), (1, -1, 1), (1, -1, -1)], [(2, 0, 0), (0, 2, 0), (0, 0, 2)]),
}


@functools.lru_cache(maxsize=4)
def _bonds(lattice, nx, ny, nz, rotated):
    """Directed bonds (p1, p2, layer), by particle, layer and partner id."""
    _, ic = _lattice(lattice, nx, ny, nz, rotated)
    lo = ic.min(axis=0) - 3
    dims = ic.max(axis=0) + 4 - lo
    flat = np.full(int(np.prod(dims)), -1, dtype=np.int64)
    key = lambda c: ((c[:, 2] - lo[2]) * dims[1] + c[:, 1] - lo[1]) * dims[0] + c[:, 0] - lo[0]  # noqa: E731
    flat[key(ic)] = np.arange(len(ic))
    rows = []
    for layer, half in enumerate(NEIGHBOURS[lattice]):
        for off in half + [tuple(-v for v in o) for o in half]:
            j = flat[key(ic + np.array(off))]
            i = np.nonzero(j >= 0)[0]
            rows.append(np.stack([i, np.full(len(i), layer), j[i]]))
    b = np.concatenate(rows, axis=1)
    b = b[:, np.lexsort((b[2], b[1], b[0]))]
    return b[0], b[2], b[1]


def _csr(n, p1, p2, layer):
    ptr = np.concatenate([[0], np.cumsum(np.bincount(p1, minlength=n))])
    split = ptr[:-1] + np.bincount(p1[layer == 0], minlength=n)
    return ptr.astype(np.int32), split.astype(np.int32), p2.astype(np.int32)


def _cracked(x, p1, p2, layer):
    """The bonds that do not cross an edge crack of a quarter of the width at mid-height."""
    y0 = 0.5 * (x[:, 1].min() + x[:, 1].max()) + 0.25
    tip = x[:, 0].min() + 0.25 * np.ptp(x[:, 0])
    ya, yb = x[p1, 1], x[p2, 1]
    cross = (ya - y0) * (yb - y0) < 0
    t = np.where(cross, (y0 - ya) / np.where(cross, yb - ya, 1.0), 0.0)
    keep = ~(cross & (x[p1, 0] + t * (x[p2, 0] - x[p1, 0]) < tip))
    return p1[keep], p2[keep], layer[keep]


def _dogbones(case, rng):
    """Eight 2D dogbones of 0.6 to 1.4 times the mean size: positions, specimen offsets, bonds."""
    parts, first, bonds = [], [0], []
    for s in range(8):
        w = max(16, int(round(case["nx"] * math.sqrt(0.6 + 0.8 * s / 7) * 0.62)))
        x, _ = _lattice("hex", w, 2 * int(w / 0.866), 1, False)
        p1, p2, layer = _bonds("hex", w, 2 * int(w / 0.866), 1, False)
        y = x[:, 1] / x[:, 1].max()
        d = np.abs(y - 0.5)
        width = np.where(d <= 0.15, 0.5, np.where(d >= 0.25, 1.0, 0.5 + 0.5 * (d - 0.15) / 0.10)) * (w - 1)
        keep = np.abs(x[:, 0] - 0.5 * (w - 1)) <= 0.5 * width + 1e-9
        new = np.cumsum(keep) - 1
        both = keep[p1] & keep[p2]
        bonds.append((new[p1[both]] + first[-1], new[p2[both]] + first[-1], layer[both]))
        parts.append(x[keep])
        first.append(first[-1] + int(keep.sum()))
    return parts, first, tuple(np.concatenate(b) for b in zip(*bonds))


# ---------------------------------------------------------------- inputs
def _stiffness(lattice, E, nu, plane_stress):
    """(Kn of layer 0, Kn of layer 1, Tv) of a bond."""
    if plane_stress:
        c11, c12 = E / (1 - nu) / (1 + nu), E * nu / (1 + nu) / (1 - nu)
    else:
        c11, c12 = E * (1 - nu) / (1 + nu) / (1 - 2 * nu), E * nu / (1 + nu) / (1 - 2 * nu)
    c44, r, s2, s3 = E / 2 / (1 + nu), RADIUS[lattice], math.sqrt(2), math.sqrt(3)
    if lattice == "hex":
        k = s3 / 12 * (c11 - c12)
        return k, k, s3 / 144 * (3 * c12 - c11)
    if lattice == "square":
        return 0.5 * (c11 - c12), 0.5 * c44, (c12 - c44) / 12
    if lattice == "sc":
        return (c11 - c12 - c44) * r, c44 * r, (c12 - c44) / 18 * r
    if lattice == "fcc":
        return s2 * c44 * r, s2 / 4 * (c11 - c12 - c44) * r, s2 / 24 * (c12 - c44) * r
    return s3 * c44 * r, (c11 - c12) / s3 * r, s3 / 14 * (c12 - c44) * r


@functools.lru_cache(maxsize=8)
def _inputs(items, seed):
    """Everything of a case that its seed makes, on the host: positions, bonds, bond stiffness (a
    random field over the particles, as a calibration has it), loads and moved positions."""
    case = dict(items)
    rng = np.random.default_rng(seed)
    key = (case["lattice"], case["nx"], case["ny"], case["nz"], case["rotated"])
    d = {"dim": DIM[case["lattice"]], "first": None}
    if case["kind"] == "fatigue":
        parts, d["first"], bonds = _dogbones(case, rng)
        d["x"] = np.concatenate(parts)
    else:
        d["x"], _ = _lattice(*key)
        bonds = _bonds(*key)
        if case["model"] == "crack":
            bonds = _cracked(d["x"], *bonds)
    d["p1"], d["p2"], d["layer"] = bonds
    x, n = d["x"], len(d["x"])
    two = d["dim"] == 2
    E = {"j2": 200e3, "hcf": 110e3}.get(case["model"], 69e3 if two else 200e3) * rng.uniform(0.9, 1.1)
    nu = 0.3 if case["model"] != "hcf" else 0.34
    d["E"], d["nu"], d["plane_stress"] = E, nu, two
    k0, k1, tv = _stiffness(case["lattice"], E, nu, two)
    field = 1 + 0.05 * rng.uniform(-1, 1, n)
    d["Kn"] = np.where(d["layer"] == 0, k0, k1) * 0.5 * (field[d["p1"]] + field[d["p2"]])
    d["Tv"] = np.full(len(d["p1"]), tv)
    ax = d["dim"] - 1
    h = x[:, ax]
    span = h.max() - h.min()
    edge = 0.4 if case["rotated"] else 1e-6
    d["lo"], d["hi"] = np.nonzero(h < h.min() + edge)[0], np.nonzero(h > h.max() - edge)[0]
    # strain per step: the elastic benchmark's 0.5% in 20 steps; through yield; until the crack grows
    crack = 1.12e-4 * math.sqrt(400 / case["nx"]) / case["steps"]
    vary = 0.02 if case["model"] == "crack" else 0.1
    d["pull"] = {"j2": 8e-4, "crack": crack}.get(case["model"], 2.5e-4) * span * rng.uniform(1 - vary, 1 + vary)
    # moved positions: a smooth stretch and a little noise
    moved = x * (1 + 1e-3 * rng.uniform(0.5, 1.5, 3)) + 1e-4 * rng.normal(size=x.shape)
    if two:
        moved[:, 2] = 0.0
    d["moved"] = np.ascontiguousarray(moved)
    d["v"], d["w"] = rng.normal(size=d["dim"] * n), rng.normal(size=d["dim"] * n)
    d["A"] = rng.uniform(3e-5, 8e-5, 8)
    return d


def _loads(d):
    """Held face and pulled face, along the last axis."""
    if d["dim"] == 3:
        return [(d["lo"], "x", 0.0), (d["lo"], "y", 0.0), (d["lo"], "z", 0.0), (d["hi"], "z", d["pull"])]
    return [(d["lo"], "x", 0.0), (d["lo"], "y", 0.0), (d["hi"], "y", d["pull"])]


def prepare(case, seed):
    d = _inputs(tuple(sorted((k, v) for k, v in case.items() if k != "name")), int(seed))
    s = {"case": case, "in": d}
    if case["kind"] == "setup":
        return s
    model = {"elastic": G.ELASTIC, "crack": G.ELASTIC, "j2": G.J2, "hcf": G.HCF}[case["model"]]
    # cracked and concatenated specimens bring their bond lists, others have them searched on the device
    lists = case["model"] in ("crack", "hcf")
    ctx = G.Context(LATTICE[case["lattice"]], RADIUS[case["lattice"]], model, d["x"],
                    bonds=_csr(len(d["x"]), d["p1"], d["p2"], d["layer"]) if lists else "device")
    s["ctx"] = ctx
    args = (d["plane_stress"], d["E"], d["nu"])
    if case["model"] == "j2":
        ctx.set_j2(0.0, *args, 300.0, 0.0, 2e3, 0.0, 1.0, damage_threshold=1.0, elmap_literal=0)
    elif case["model"] == "hcf":
        t = np.zeros(len(d["x"]), dtype=np.int32)
        groups, amp = [], []
        for a, b in zip(d["first"][:-1], d["first"][1:]):
            y = d["x"][a:b, 1]
            top, bottom = a + np.nonzero(y > y.max() - 1e-6)[0], a + np.nonzero(y < y.min() + 1e-6)[0]
            t[top] = t[bottom] = 4
            groups.append([top, bottom])
            amp.append(1e-3 * (y.max() - y.min()))
        ctx.set_specimens(d["first"])
        ctx.set("type", t)
        ctx.set_hcf(4.0, *args, 5e-5, 2.019, 0.5, elmap_literal=0)
        mat = ctx.get("mat").reshape(-1, 10)
        for k, (a, b) in enumerate(zip(d["first"][:-1], d["first"][1:])):
            mat[a:b, 0] = d["A"][k]
        ctx.set("mat", mat)
        ctx.search_nonlocal(1.5)
        s["groups"], s["amp"] = groups, amp
        s["start"] = ctx.load_step(disp=[bc for (top, bottom), a in zip(groups, amp)
                                         for bc in [(top, "x", 0.0), (top, "y", 0.1 * a), (top, "z", 0.0), (bottom, "x", 0.0),
                                                    (bottom, "y", 0.0), (bottom, "z", 0.0)]])
    else:
        ctx.set_elastic(0.0, *args, 1e-3 if case["model"] == "crack" else 1.0, elmap_literal=0)
    ctx.set("Kn", d["Kn"])
    ctx.set("Tv", d["Tv"])
    fp64 = case["precision"] == 1
    ctx.mode(dirichlet_static=1, cg_transpose=0, diag10_literal=0, precision=case["precision"], precond=case["precond"],
             cg_tol=1e-12 if fp64 and case["kind"] != "path" else 1e-3, cg_forcing=int(case["kind"] in ("path", "fatigue")),
             tol_NR=1e-8 if case["model"] == "crack" else 1e-10 if d["dim"] == 2 else 1e-11, max_NR_iter=50, cg_maxit=50000)
    if case["kind"] == "adjoint" and not fp64:
        ctx.mode(cg_tol=1e-6)
    if case["kind"] == "path":
        ctx.mode(predictor={"crack": 1}.get(case["model"], 2), coarse_reuse=1)
        s["load"] = ctx.load_step(disp=_loads(d))
    if case["kind"] in ("forces", "tangent"):
        ctx.set("xyz", d["moved"])
    if case["kind"] in ("linear", "adjoint"):
        s["load"] = ctx.load_step(disp=_loads(d))
    ctx.update_geometry()
    ctx.update_force_state()
    if case["kind"] == "linear":
        ctx.apply_bc(s["load"])
        ctx.update_geometry()
        ctx.update_force_state()
    if case["kind"] == "adjoint":
        if not ctx.solve_step_static(s["load"], -1):
            raise RuntimeError("the state of the adjoint does not converge")
    if case["kind"] in ("path", "linear", "fatigue"):
        ctx.store()
        ctx.checkpoint_save(0)
    return s


# ---------------------------------------------------------------- one pass
def run(state):
    case, d = state["case"], state["in"]
    kind = case["kind"]
    if kind == "setup":
        ctx = G.Context(LATTICE[case["lattice"]], RADIUS[case["lattice"]], G.HCF, d["moved"], bonds="device")
        ctx.set_hcf(4.0 * RADIUS[case["lattice"]], d["plane_stress"], d["E"], d["nu"], 5e-5, 2.019, 0.5, elmap_literal=0)
        ctx.search_nonlocal(1.5)
        out = {k: ctx.get(k) for k in ("bond_ptr", "bond_p2", "opp", "dis_initial", "conn_ptr", "conn_idx", "nl_ptr", "nl_idx")}
        ctx.close()
        return out
    ctx = state["ctx"]
    if kind == "forces":
        ctx.set("xyz", d["moved"])
        ctx.update_geometry()
        ctx.update_force_state()
        norms = ctx.update_rr()
        return {"Pin": ctx.get("Pin"), "stress": ctx.get("stress"), "norms": list(norms)}
    if kind == "tangent":
        return {"jv": ctx.force_jvp(d["v"]), "jtw": ctx.force_vjp(d["w"])}
    if kind == "linear":
        ctx.checkpoint_restore(0)
        ctx.update_rr()
        ctx.calc_stiffness()
        ctx.update_stiffness_disp_bc()
        ctx.solve_linear_system()
        return {"disp": ctx.get("disp"), "xyz": ctx.get("xyz")}
    if kind == "path":
        ctx.checkpoint_restore(0)
        for _ in range(case["steps"]):
            if not ctx.solve_step_static(state["load"], -1):
                raise RuntimeError("a load step does not converge")
        if case["model"] == "crack":
            return {"xyz": ctx.get("xyz"), "bdamage": ctx.get("bdamage")}
        if d["dim"] == 2:  # the Newton test of a tall plate leaves Pin at its free DoFs at 1e-8 of the reactions
            return {"xyz": ctx.get("xyz"), "dis": ctx.get("dis")}
        out = {"xyz": ctx.get("xyz"), "Pin": ctx.get("Pin"), "stress": ctx.get("stress")}
        if case["model"] == "j2":
            out["state_var"] = ctx.get("state_var")
        return out
    if kind == "fatigue":
        ctx.checkpoint_restore(0)
        ctx.solve_problem_fatigue_static([state["start"]])
        ctx.solve_problem_cyclic_specimens(G.LOAD_DOGBONE_DISP, 1, [0.1] + [1.0, 0.1] * 200, state["groups"], state["amp"], 0.05,
                                           4, max_cycles_run=case["steps"])
        return {"xyz": ctx.get("xyz"), "damage": ctx.get("damage"), "state_var": ctx.get("state_var")}
    w_pin = np.zeros(d["dim"] * ctx.n)
    w_pin[d["dim"] * d["hi"] + d["dim"] - 1] = 1.0
    value, g_kn, g_tv, g_damage, _, _ = ctx.adjoint_linear(w_pin=w_pin, w_x=1e3 * d["w"])
    return {"value": value, "dKn": g_kn, "dTv": g_tv, "dbdamage": g_damage}


# ---------------------------------------------------------------- the least work of a pass
def work(case):
    """Positions and bond parameters read and results written once; where a matrix is formed, its
    blocks written and read once per load step (or half cycle)."""
    d = _inputs(tuple(sorted((k, v) for k, v in case.items() if k != "name")), 1)
    n, nb, dim = len(d["x"]), len(d["p1"]), d["dim"]
    force = {"bytes": 24 * n + 44 * nb + 72 * n, "flops": 70 * nb}
    if case["kind"] == "forces":
        return force
    if case["kind"] == "tangent":
        return {"bytes": 32 * dim * n + 72 * nb, "flops": 120 * nb}
    if case["kind"] == "setup":
        return {"bytes": 24 * n + 16 * nb + 4 * n * BLOCKS[case["lattice"]], "flops": 10 * nb}
    blocks = n * BLOCKS[case["lattice"]]
    solves = {"fatigue": 2 * case["steps"] + 1}.get(case["kind"], case["steps"])
    matrix = 2 * blocks * dim * dim * (8 if case["precision"] else 4)
    out = 24 * nb if case["kind"] == "adjoint" else 0
    return {"bytes": solves * (force["bytes"] + matrix) + out,
            "flops": solves * (force["flops"] + blocks * dim * dim * 12)}


# ---------------------------------------------------------------- the same in 64 bits
class _Exact:
    """Internal force and its Jacobian in plain torch, FP64."""

    def __init__(self, d):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        t = lambda a: torch.as_tensor(np.ascontiguousarray(a), device=dev)  # noqa: E731
        self.n, self.dim, self.dev = len(d["x"]), d["dim"], dev
        self.x0 = t(d["x"])[:, :self.dim]
        self.p1, self.p2, layer = t(d["p1"]), t(d["p2"]), t(d["layer"])
        self.slot = 2 * self.p1 + layer
        order = np.lexsort((d["p1"], d["layer"], d["p2"]))  # the k-th bond in reverse order is the reverse of the k-th
        opp = np.empty(len(order), dtype=np.int64)
        opp[order] = np.arange(len(order))
        self.opp = t(opp)
        self.kn, self.tv = t(d["Kn"]), t(d["Tv"])
        self.dis0 = (self.x0[self.p1] - self.x0[self.p2]).norm(dim=1)

    def total(self, le):
        return torch.zeros(2 * self.n, dtype=torch.float64, device=self.dev).index_add_(0, self.slot, le)

    def gather(self, per_bond):
        return torch.zeros(self.n, self.dim, dtype=torch.float64, device=self.dev).index_add_(0, self.p1, per_bond)

    def at(self, x):
        r = x[self.p1] - x[self.p2]
        self.dis = r.norm(dim=1)
        self.cs = r / self.dis[:, None]
        self.le = self.dis - self.dis0
        self.tot = self.total(self.le)
        f = 2 * self.kn * self.le + 2 * self.tv * self.tot[self.slot]
        self.ff = 0.5 * (f + f[self.opp])
        return self.gather(self.cs * self.ff[:, None])

    def jvp(self, v):  # symmetric here: no damage, one Tv, the Kn of a bond and of its reverse equal
        dv = v[self.p1] - v[self.p2]
        dd = (self.cs * dv).sum(dim=1)
        df = 2 * self.kn * dd + 2 * self.tv * self.total(dd)[self.slot]
        df = 0.5 * (df + df[self.opp])
        return self.gather((dv - self.cs * dd[:, None]) * (self.ff / self.dis)[:, None] + self.cs * df[:, None])

    def solve(self, b, free, tol=1e-13, most=20000):
        diag = self.gather((2 * self.kn + 2 * self.tv)[:, None] * self.cs * self.cs).abs() + 1e-300
        x, r = torch.zeros_like(b), b * free
        z = r / diag
        p, rz, stop = z.clone(), (r * z).sum(), tol * r.norm()
        for k in range(most):
            q = self.jvp(p) * free
            a = rz / (p * q).sum()
            x += a * p
            r -= a * q
            if k % 16 == 0 and r.norm() <= stop:
                break
            z = r / diag
            new = (r * z).sum()
            p = z + (new / rz) * p
            rz = new
        return x

    def equilibrium(self, d, steps):
        """Positions under `steps` of the case's loads, and the free DoFs."""
        free = torch.ones(self.n, self.dim, dtype=torch.float64, device=self.dev)
        x = self.x0.clone()
        h = x[:, -1]
        x[:, -1] = h + (h - h.min()) / (h.max() - h.min()) * steps * d["pull"]
        for ids, axis, step in _loads(d):
            a = "xyz".index(axis)
            free[ids, a] = 0.0
            x[ids, a] = self.x0[ids, a] + steps * step
        for _ in range(12):
            r = -self.at(x) * free
            scale = self.gather(self.cs * self.ff[:, None]).norm()
            if r.norm() <= 1e-14 * scale:
                break
            x = x + self.solve(r, free)
        self.at(x)
        return x, free

    def three(self, v):
        out = torch.zeros(self.n, 3, dtype=torch.float64, device=self.dev)
        out[:, :self.dim] = v
        return out.reshape(-1)


def exact(case, seed):
    d = _inputs(tuple(sorted((k, v) for k, v in case.items() if k != "name")), int(seed))
    kind = case["kind"]
    if kind == "setup":
        x = d["moved"]
        length = np.linalg.norm(x[d["p1"]] - x[d["p2"]], axis=1)
        return dict.fromkeys(("bond_ptr", "bond_p2", "opp", "conn_ptr", "conn_idx", "nl_ptr", "nl_idx"), None) | {"dis_initial": length}
    if case["model"] != "elastic" or (kind in ("path", "linear", "adjoint") and len(d["x"]) > 40000):
        return None
    e = _Exact(d)
    if kind in ("forces", "tangent"):
        pin = e.at(torch.as_tensor(d["moved"], device=e.dev)[:, :e.dim])
        if kind == "forces":  # no DoF is held and none loaded: the residual is -Pin
            return {"Pin": e.three(pin), "stress": None, "norms": [float(pin.norm()), None]}
        as2 = lambda v: torch.as_tensor(v, device=e.dev).reshape(e.n, e.dim)  # noqa: E731
        return {"jv": e.jvp(as2(d["v"])).reshape(-1), "jtw": e.jvp(as2(d["w"])).reshape(-1)}
    if kind == "linear":  # the library's matrix drops small terms of the Jacobian on purpose
        return None
    x, free = e.equilibrium(d, case["steps"])
    if kind == "path":
        if e.dim == 2:
            return {"xyz": e.three(x), "dis": e.dis}
        return {"xyz": e.three(x), "Pin": e.three(e.gather(e.cs * e.ff[:, None])), "stress": None}
    a = torch.zeros(e.n, e.dim, dtype=torch.float64, device=e.dev)
    a[d["hi"], e.dim - 1] = 1.0
    b = 1e3 * torch.as_tensor(d["w"], device=e.dev).reshape(e.n, e.dim)
    pin = e.gather(e.cs * e.ff[:, None])
    lam = e.solve((e.jvp(a) + b) * free, free)
    w = a - lam
    t2 = ((w[e.p1] - w[e.p2]) * e.cs).sum(dim=1)  # 2 t_b
    tot = e.tot[e.slot]
    return {"value": float((a * pin).sum() + (b * x).sum()), "dKn": t2 * e.le, "dTv": t2 * tot,
            "dbdamage": -t2 * (e.kn * e.le + e.tv * tot)}
