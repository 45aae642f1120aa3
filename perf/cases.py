"""Performance cases: what programs that use this engine have it do.

A pass is one frame of a program's loop: advance by ``step(dt, substeps)`` (or
one request per resident scene through the server), then read the state back,
as the reference's update() does after its substeps.  The scenes are cantilever
beams of 1.0 x 0.25 x 0.25 m in the sizes of the repository's workloads, caught
in mid-motion: bent, moving at about 1 m/s, with a little noise on every vertex.

``exact`` advances the same scene in 64 bits with torch and numpy alone.  It
makes its own meshes, shape functions and colourings (the colour orders decide
the Gauss-Seidel results, so the same saturation-degree and smallest-last rules
are restated here).
"""
from __future__ import annotations

import heapq
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import octopusengine_amd as oe

SIZE = (1.0, 0.25, 0.25)
GRAVITY = -9.81
DENSITY = 1000.0
ELEMENTS = {"p1": oe.TETRA, "q1": oe.HEXA, "p2": oe.TETRA10, "p3": oe.TETRA20, "q2": oe.HEXA27}
MATERIALS = {"neohooke": oe.NEOHOOKE, "stable": oe.STABLE_NEOHOOKE}


# ------------------------------------------------------------------ the cases
def _vbd(name, element, cells, **kw):
    c = dict(kind="vbd", element=element, nx=cells[0], ny=cells[1], nz=cells[2], young=5e5, poisson=0.49,
             material="stable", iterations=10, rho=0.0, damping=0.0, curve=0.0, dt=0.02, substeps=4)
    c.update(kw)
    return dict(c, name=name) if name else c


def _xpbd(name, element, cells, **kw):
    c = dict(kind="xpbd", element=element, nx=cells[0], ny=cells[1], nz=cells[2], young=1e6, poisson=0.45,
             material="neohooke", damping=0.0, curve=0.0, dt=0.01, substeps=50)
    c.update(kw)
    return dict(c, name=name) if name else c


def _explicit(name, element, cells, **kw):
    c = dict(kind="explicit", element=element, nx=cells[0], ny=cells[1], nz=cells[2], young=1e6, poisson=0.45,
             material="neohooke", damping=0.0, curve=0.0, dt=1e-3, substeps=100)
    c.update(kw)
    return dict(c, name=name) if name else c


def listed():
    return [
        # An interactive object: one step of a small quadratic beam per frame,
        # where a frame is a chain of small launches.
        _vbd("vbd_p2_16x4x4", "p2", (16, 4, 4), dt=0.005, substeps=1),
        # The usual linear meshes of the VBD experiments, with the Chebyshev
        # acceleration and the stiffer material that those runs use.
        _vbd("vbd_p1_64x16x16", "p1", (64, 16, 16), young=1e7, poisson=0.45, rho=0.75),
        # Trilinear hexahedra on a mesh that follows a curved shape (an asset
        # rather than a generated box), with damping.
        _vbd("vbd_q1_64x16x16", "q1", (64, 16, 16), young=1e7, poisson=0.45, curve=0.02, damping=1e-4),
        # The single-scene workload: 140,481 vertices, soft and nearly incompressible.
        _vbd("vbd_p2_64x16x16", "p2", (64, 16, 16)),
        # Quadratic hexahedra at the size of the reference's comparisons.
        _vbd("vbd_q2_32x8x8", "q2", (32, 8, 8), young=1e7, poisson=0.45),
        # The small linear XPBD scene: one frame of 20 substeps.
        _xpbd("xpbd_p1_16x4x4", "p1", (16, 4, 4), substeps=20),
        # The high-order XPBD frames, 50 substeps each.
        _xpbd("xpbd_q2_32x8x8", "q2", (32, 8, 8)),
        _xpbd("xpbd_p3_32x8x8", "p3", (32, 8, 8)),
        # High-order explicit integration at dt = 1e-5 s, read back every millisecond.
        _explicit("explicit_q2_32x8x8", "q2", (32, 8, 8)),
        _explicit("explicit_p3_32x8x8", "p3", (32, 8, 8), damping=1e-5),
        # Batched simulation of mixed beams (grids of 8-64 x 4-16 x 4-16 cells,
        # P2 or Q2), recorded at 25 frames per second of simulated time.
        dict(kind="batch", name="batch_mixed_32", scenes=32, nx_max=64, nyz_max=16, layout=4, iterations=10, dt=0.04,
             substeps=8),
        # A serving program's frame: one step request for each resident scene,
        # sizes log-normal around 20,000 vertices, then every state is read.
        dict(kind="served", name="served_30", scenes=30, median=20000.0, layout=5, iterations=10, dt=0.005,
             substeps=1, max_batch=64, streams=2),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["vbd", "vbd", "vbd", "xpbd", "explicit", "batch", "served"])
    if kind == "batch":
        return dict(kind="batch", scenes=_log_int(rng, 2, 32), nx_max=rng.randint(9, 64), nyz_max=rng.randint(5, 16),
                    layout=rng.randrange(1 << 20), iterations=rng.choice([2, 5, 10]), dt=0.02, substeps=4)
    if kind == "served":
        return dict(kind="served", scenes=_log_int(rng, 2, 30), median=float(_log_int(rng, 1000, 20000)),
                    layout=rng.randrange(1 << 20), iterations=rng.choice([5, 10]), dt=0.005, substeps=1,
                    max_batch=rng.choice([16, 64]), streams=2)
    element = rng.choice(["p1", "q1", "p2", "p3", "q2"])
    material = rng.choice(["neohooke", "stable"])
    curve = rng.choice([0.0, 0.0, 0.02])
    # vertices per cell edge: the finer the element, the fewer cells per axis
    per = {"p1": 1, "q1": 1, "p2": 2, "q2": 2, "p3": 3}[element]
    nyz_hi = {1: 16, 2: 12, 3: 8}[per]
    ny = _log_int(rng, 1, nyz_hi)
    nz = max(1, min(nyz_hi, ny + rng.randint(-2, 2)))
    nx = max(1, min(4 * nyz_hi, int(round(rng.uniform(2.0, 5.0) * ny))))
    if kind == "vbd":
        return _vbd("", element, (nx, ny, nz), material=material, curve=curve,
                    young=10.0 ** rng.uniform(5.0, 7.0), poisson=round(rng.uniform(0.3, 0.49), 3),
                    iterations=rng.choice([2, 5, 10]), rho=rng.choice([0.0, 0.0, 0.75]),
                    damping=rng.choice([0.0, 0.0, 1e-4]), dt=0.005 * (n := rng.choice([1, 2, 4])), substeps=n)
    if kind == "xpbd":
        n = _log_int(rng, 5, 50)
        return _xpbd("", element, (nx, ny, nz), curve=curve, dt=2e-4 * n, substeps=n)
    n = _log_int(rng, 10, 100)
    return _explicit("", element, (nx, ny, nz), material=material, curve=curve, damping=rng.choice([0.0, 1e-5]),
                     dt=1e-5 * n, substeps=n)


# --------------------------------------------------------------------- meshes
# Reference nodes per element, in the engine's node order.  Tetrahedra: corners,
# then edge nodes, then face nodes; hexahedra: corners, edges, faces, centre.
_TET_NODES = {
    "p1": [(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)],
    "p2": [(0, 0, 0), (2, 0, 0), (0, 2, 0), (0, 0, 2), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1),
           (0, 1, 1)],
    "p3": [(0, 0, 0), (3, 0, 0), (0, 3, 0), (0, 0, 3), (1, 0, 0), (2, 0, 0), (2, 1, 0), (1, 2, 0), (0, 2, 0),
           (0, 1, 0), (0, 0, 1), (0, 0, 2), (2, 0, 1), (1, 0, 2), (0, 2, 1), (0, 1, 2), (1, 0, 1), (1, 1, 1),
           (0, 1, 1), (1, 1, 0)],
}
_ORDER = {"p1": 1, "p2": 2, "p3": 3, "q1": 1, "q2": 2}
_HEX8 = [(-1, -1, -1), (1, -1, -1), (1, 1, -1), (-1, 1, -1), (-1, -1, 1), (1, -1, 1), (1, 1, 1), (-1, 1, 1)]
_HEX27 = _HEX8 + [(0, -1, -1), (1, 0, -1), (0, 1, -1), (-1, 0, -1), (-1, -1, 0), (1, -1, 0), (1, 1, 0), (-1, 1, 0),
                  (0, -1, 1), (1, 0, 1), (0, 1, 1), (-1, 0, 1), (0, 0, -1), (0, -1, 0), (1, 0, 0), (0, 1, 0),
                  (-1, 0, 0), (0, 0, 1), (0, 0, 0)]
# the six tetrahedra of a cell, by cell corner
_TETS = np.array([[0, 4, 6, 5], [3, 6, 2, 0], [0, 4, 7, 6], [3, 6, 0, 7], [2, 0, 6, 1], [6, 0, 5, 1]])
# lattice offsets of a cell's corners
_CORNERS = np.array([(0, 0, 0), (1, 0, 0), (1, 0, 1), (0, 0, 1), (0, 1, 0), (1, 1, 0), (1, 1, 1), (0, 1, 1)])


def _beam(element, nx, ny, nz, curve=0.0):
    """(xyz float32 (N, 3), topology int32 (E, S)): grid corners first (x
    fastest), the other nodes in the order in which the elements meet them."""
    p = _ORDER[element]
    k, j, i = np.meshgrid(np.arange(nz), np.arange(ny), np.arange(nx), indexing="ij")
    cells = np.stack([i.ravel(), j.ravel(), k.ravel()], 1)
    corners = p * (cells[:, None, :] + _CORNERS[None])                      # (cells, 8, 3), lattice units
    if element in _TET_NODES:
        ref = np.array(_TET_NODES[element])
        bary = np.concatenate([p - ref.sum(1, keepdims=True), ref], 1)      # in units of 1 / p
        tets = corners[:, _TETS].reshape(-1, 4, 3)
        nodes = np.einsum("sk,ekd->esd", bary, tets) // p
    else:
        # trilinear weights of the cell's corners at the reference nodes
        ref = np.array(_HEX8 if element == "q1" else _HEX27)
        w = np.stack([np.prod(1 + ref * c, axis=1) for c in np.array(_HEX8)], 1)     # (S, 8), eighths
        nodes = np.einsum("sk,ekd->esd", w, corners) // 8
    lx, ly = p * nx + 1, p * ny + 1
    key = (nodes[..., 2] * ly + nodes[..., 1]) * lx + nodes[..., 0]
    uniq, first, inv = np.unique(key.ravel(), return_index=True, return_inverse=True)
    lattice = np.stack([uniq % lx, uniq // lx % ly, uniq // (lx * ly)], 1)
    corner = (lattice % p == 0).all(1)
    rank = np.where(corner, uniq, first + int(key.max()) + 1)
    order = np.argsort(rank, kind="stable")
    ids = np.empty(len(uniq), np.int64)
    ids[order] = np.arange(len(uniq))
    xyz = lattice[order] * (np.array(SIZE) / (p * np.array([nx, ny, nz])))
    if curve:
        x, y, z = xyz.T.copy()
        xyz[:, 1] += curve * np.sin(3.0 * x) * (1.0 + 4.0 * z)
        xyz[:, 2] += curve * np.cos(2.0 * x) * y * 4.0
    return xyz.astype(np.float32), ids[inv].reshape(key.shape).astype(np.int32)


def _fixed(xyz):
    return xyz[:, 0] < 1e-6


def _motion(xyz, seed, spacing):
    """(positions, velocity) float32 of a bent, swinging beam with noise; the
    fixed face at rest."""
    rng = np.random.default_rng(seed)
    x = xyz[:, 0:1].astype(np.float64)
    bend = np.array([0.0, -1.0, 0.0]) * rng.uniform(0.02, 0.08) + np.array([0.0, 0.0, 1.0]) * rng.uniform(-0.04, 0.04)
    swing = np.array([0.0, -1.0, 0.0]) * rng.uniform(0.8, 1.6) + np.array([0.1, 0.0, 1.0]) * rng.uniform(-0.5, 0.5)
    noise = rng.uniform(-1.0, 1.0, xyz.shape) * min(1e-3, 0.06 * spacing)
    free = ~_fixed(xyz)[:, None]
    pos = xyz + np.where(free, bend * x * x + noise, 0.0)
    return pos.astype(np.float32), np.where(free, swing * x * x, 0.0).astype(np.float32)


def _spacing(case):
    return min(SIZE[0] / case["nx"], SIZE[1] / case["ny"], SIZE[2] / case["nz"]) / _ORDER[case["element"]]


def _parts(case):
    """The scenes of a batch or a pool, as VBD cases; the same for every seed."""
    rng = np.random.default_rng(case["layout"])
    out = []
    for _ in range(case["scenes"]):
        if case["kind"] == "batch":
            cells = (int(rng.integers(8, case["nx_max"] + 1)), int(rng.integers(4, case["nyz_max"] + 1)),
                     int(rng.integers(4, case["nyz_max"] + 1)))
        else:
            target = min(case["median"] * float(np.exp(rng.normal())), 150000.0)
            k = max(1, int(round((target / 32.0) ** (1.0 / 3.0))))
            cells = (max(1, int(round((target / (2 * k + 1) ** 2 - 1.0) / 2.0))), k, k)
        out.append(_vbd("", "p2" if rng.random() < 0.5 else "q2", cells, young=float(10.0 ** rng.uniform(5.0, 7.0)),
                        poisson=float(rng.uniform(0.3, 0.49)), iterations=case["iterations"], dt=case["dt"],
                        substeps=case["substeps"]))
    return out


# -------------------------------------------------------------- prepare / run
_engine = None


def _shared_engine():
    global _engine
    if _engine is None:
        _engine = oe.Engine(0)
    return _engine


def _scene(case, seed):
    xyz, topo = _beam(case["element"], case["nx"], case["ny"], case["nz"], case["curve"])
    args = dict(material=MATERIALS[case["material"]], young=case["young"], poisson=case["poisson"], density=DENSITY,
                distribution=oe.MASS_FEMSHAPE, gravity=(0.0, GRAVITY, 0.0), sub_iterations=case["substeps"])
    if case["kind"] == "vbd":
        args.update(solver=oe.SOLVER_VBD, iterations=case["iterations"], rho=case["rho"], damping=case["damping"])
    elif case["kind"] == "xpbd":
        args.update(solver=oe.SOLVER_XPBD, global_damping=case["damping"])
    else:
        args.update(solver=oe.SOLVER_EXPLICIT, damping=case["damping"])
    s = oe.Scene(_shared_engine(), ELEMENTS[case["element"]], xyz, topo, **args)
    s.fix_plane((1e-6, 0.0, 0.0), (-1.0, 0.0, 0.0))
    s.box_limit((-10.0, -5.0, -10.0), (10.0, 5.0, 10.0))
    pos, last, vel = _initial(case, seed, xyz)
    s.set_state(p=pos, last_p=last, v=vel)
    return s


def _initial(case, seed, xyz):
    pos, vel = _motion(xyz, seed, _spacing(case))
    return pos, (pos - vel * np.float32(case["dt"] / case["substeps"])).astype(np.float32), vel


class _Program:
    """What a program keeps: its scenes and the batch or server over them."""

    def __init__(self, case, seed):
        self.case = case
        self.kind = case["kind"]
        self.holder = None
        engine = _shared_engine()                # before the scenes' threads ask for it
        if self.kind in ("batch", "served"):
            parts = list(enumerate(_parts(case)))
            with ThreadPoolExecutor(8) as ex:
                self.scenes = list(ex.map(lambda p: _scene(p[1], seed * 1000 + p[0]), parts))
            if self.kind == "batch":
                self.holder = oe.Batch(engine, self.scenes)
            else:
                self.holder = oe.Server(engine, max_batch=case["max_batch"], streams=case["streams"])
                self.slots = [self.holder.add_scene(s) for s in self.scenes]
        else:
            self.scenes = [_scene(case, seed)]

    def __del__(self):
        if self.holder is not None:
            self.holder.close()
        for s in self.scenes:
            s.close()


def prepare(case, seed):
    return _Program(case, seed)


def run(state):
    case = state.case
    if state.kind == "batch":
        state.holder.step(case["dt"], case["substeps"])
    elif state.kind == "served":
        for slot in state.slots:
            state.holder.submit(slot, case["dt"], case["substeps"])
        state.holder.drain()
    else:
        s = state.scenes[0]
        s.update(case["dt"])
        if state.kind == "xpbd":
            # an XPBD state is its last two positions
            return {"positions": s.positions(), "last_positions": s.last_positions()}
        return {"positions": s.positions(), "velocities": s.velocities()}
    return {"positions": [s.positions() for s in state.scenes], "velocities": [s.velocities() for s in state.scenes]}


# ----------------------------------------------------------------------- work
_S = {"p1": 4, "q1": 8, "p2": 10, "p3": 20, "q2": 27}
_Q = {"p1": 1, "q1": 8, "p2": 4, "p3": 11, "q2": 27}


def _counts(case):
    p, n = _ORDER[case["element"]], (case["nx"], case["ny"], case["nz"])
    cells = n[0] * n[1] * n[2]
    E = cells * (6 if case["element"] in _TET_NODES else 1)
    if case["element"] == "p3":                 # every lattice node but those inside the tetrahedra's cells
        N = len(_beam("p3", *n)[0])
    else:
        N = (p * n[0] + 1) * (p * n[1] + 1) * (p * n[2] + 1)
    return N, E


def work(case):
    """Bytes: topology, rest positions, masses and the two state arrays in, two
    state arrays out.  Operations: per (element, point) and visited node the
    node's rank-1 change of the gradient, the stress and the node's terms (170
    for a VBD vertex block); XPBD visits an element twice per substep, the
    explicit pass once; plus the vertex solves."""
    if case["kind"] in ("batch", "served"):
        parts = [work(c) for c in _parts(case)]
        return {k: sum(w[k] for w in parts) for k in ("bytes", "flops")}
    N, E = _counts(case)
    S, Q = _S[case["element"]], _Q[case["element"]]
    n = case["substeps"]
    grad = min(18 * S, 144)                     # a point's gradient from the nodes (sum-factorised on hexahedra)
    if case["kind"] == "vbd":
        flops = n * case["iterations"] * (E * S * Q * 170.0 + N * 100.0)
    elif case["kind"] == "xpbd":
        flops = n * (2.0 * E * (Q * (grad + 120) + Q * S * 15 + S * 12) + N * 30.0)
    else:
        flops = n * (E * (Q * (grad + 150) + Q * S * 50) + N * 40.0)
    return {"bytes": 4.0 * S * E + N * (12 + 4 + 24 + 24), "flops": flops}


# ---------------------------------------------------------- 64-bit restatement
_P3_POINTS = [
    0.040490506727590427904, 0.013560701879802881248, 0.77125473269537614396, 0.75250850700965499218,
    0.068099370938206657544, 0.097987203649279111528, 0.067223294893383397919, 0.035183929773598715540,
    0.15636389323939528517, 0.41926631387951301955, 0.047781435559086662956, 0.47961101102565506515,
    0.45076587609127682921, 0.059456616299433828754, 0.056824017127933668103, 0.12941137378891040544,
    0.33019041483746447430, 0.0023910074574393647140, 0.12154199133392780408, 0.30649398842969027834,
    0.56297276014304609149, 0.097204644587583266535, 0.68439041545304002412, 0.11180076739738309399,
    0.029569495206479612381, 0.31790356021339460924, 0.32329398483747895376, 0.43271023904776856339,
    0.35382323920929709127, 0.10962240533194123060, 0.24027666492807261966, 0.12680172591539201621,
    0.32847320672203844660]
_P3_WEIGHTS = [
    0.039251090924839956986, 0.055273369155936898089, 0.055393798871576367671, 0.059933185146559528333,
    0.069469965937635366759, 0.076162715245558357258, 0.079426680068025307113, 0.10646803415549009608,
    0.11023423242849765546, 0.15497611601624608491, 0.19341081204963445073]


def _shape(element):
    """(dN (Q, S, 3), weights (Q,)): Lagrange basis from the Vandermonde matrix."""
    p = _ORDER[element]
    if element in _TET_NODES:
        nodes = np.array(_TET_NODES[element]) / p
        mono = [(a, b, c) for a in range(p + 1) for b in range(p + 1 - a) for c in range(p + 1 - a - b)]
        if element == "p1":
            qp, w = np.full((1, 3), 0.25), np.array([1 / 6])
        elif element == "p2":
            a, b = (5 - math.sqrt(5)) / 20, (5 + 3 * math.sqrt(5)) / 20
            qp, w = np.array([(b, a, a), (a, b, a), (a, a, b), (a, a, a)]), np.full(4, 1 / 24)
        else:
            qp, w = np.array(_P3_POINTS).reshape(11, 3), np.array(_P3_WEIGHTS) / 6
    else:
        nodes = np.array(_HEX8 if element == "q1" else _HEX27, np.float64)
        mono = [(a, b, c) for a in range(p + 1) for b in range(p + 1) for c in range(p + 1)]
        if element == "q1":
            qp, w = np.array(_HEX8) / math.sqrt(3), np.ones(8)
        else:
            qp = np.array(_HEX27) * math.sqrt(0.6)
            w = np.prod(np.where(np.array(_HEX27) == 0, 8 / 9, 5 / 9), axis=1)
    mono = np.array(mono)
    basis = lambda x: np.prod(x[:, None, :] ** mono[None], axis=2)                       # noqa: E731
    coeff = np.linalg.inv(basis(nodes))
    dN = []
    for d in range(3):
        m = mono.copy()
        m[:, d] = np.maximum(m[:, d] - 1, 0)
        dm = np.prod(qp[:, None, :] ** m[None], axis=2) * mono[None, :, d]
        dN.append(dm @ coeff)
    return np.stack(dN, 2), w


def _neighbours(pairs_a, pairs_b, n):
    """Rows of (neighbour, multiplicity) of a multigraph given every ordered pair."""
    key, mult = np.unique(pairs_a.astype(np.int64) * n + pairs_b, return_counts=True)
    a, b = key // n, key % n
    off = np.searchsorted(a, np.arange(n + 1))
    return b, mult, off


def _vertex_colours(topo, n):
    """Saturation-degree colouring: the next vertex is the one of most
    neighbouring colours, then of most uncoloured neighbours, then of the
    highest id; it takes the lowest free colour."""
    S = topo.shape[1]
    a = np.repeat(topo, S, axis=1).ravel()
    b = np.tile(topo, (1, S)).ravel()
    keep = a != b
    nb, mult, off = _neighbours(a[keep], b[keep], n)
    nb, mult, off = nb.tolist(), mult.tolist(), off.tolist()
    deg = [sum(mult[off[v]:off[v + 1]]) for v in range(n)]
    sat, seen, colour = [0] * n, [0] * n, [-1] * n
    heap = [(0, -deg[v], -v) for v in range(n)]
    heapq.heapify(heap)
    push, pop = heapq.heappush, heapq.heappop
    while heap:
        s, d, v = pop(heap)
        v = -v
        if colour[v] >= 0 or -s != sat[v] or -d != deg[v]:
            continue
        used = seen[v]
        c = 0
        while used >> c & 1:
            c += 1
        colour[v] = c
        bit = 1 << c
        for k in range(off[v], off[v + 1]):
            u = nb[k]
            if colour[u] >= 0:
                continue
            if not seen[u] & bit:
                seen[u] |= bit
                sat[u] += 1
            deg[u] -= mult[k]
            push(heap, (-sat[u], -deg[u], -u))
    return np.array(colour)


def _element_colours(topo):
    """Smallest-last colouring of the elements; an edge per shared vertex."""
    E, S = topo.shape
    owner = np.argsort(topo.ravel(), kind="stable") // S
    counts = np.bincount(topo.ravel())
    start = np.concatenate([[0], np.cumsum(counts)])
    a, b = [], []
    for c in np.unique(counts):
        rows = owner[start[:-1][counts == c][:, None] + np.arange(c)[None]]
        a.append(np.repeat(rows, c, axis=1).ravel())
        b.append(np.tile(rows, (1, c)).ravel())
    a, b = np.concatenate(a), np.concatenate(b)
    keep = a != b
    nb, mult, off = _neighbours(a[keep], b[keep], E)
    nb, mult, off = nb.tolist(), mult.tolist(), off.tolist()
    deg = [sum(mult[off[e]:off[e + 1]]) for e in range(E)]
    heap = [(deg[e], e) for e in range(E)]
    heapq.heapify(heap)
    gone, order = [False] * E, []
    while heap:
        d, e = heapq.heappop(heap)
        if gone[e]:
            continue
        gone[e] = True
        order.append(e)
        for k in range(off[e], off[e + 1]):
            u = nb[k]
            if not gone[u]:
                # an edge per shared vertex: every step of the degree is a key
                deg[u] -= mult[k]
                heapq.heappush(heap, (deg[u], u))
    colour = [-1] * E
    for e in reversed(order):
        used = {colour[u] for u in nb[off[e]:off[e + 1]]}
        c = 0
        while c in used:
            c += 1
        colour[e] = c
    return np.array(colour)


class _Exact:
    """One scene in 64 bits; displacements u from the rest positions X."""

    def __init__(self, case, seed):
        dev = "cuda" if torch.cuda.is_available() else "cpu"
        self.case, self.dev = case, dev
        xyz, topo = _beam(case["element"], case["nx"], case["ny"], case["nz"], case["curve"])
        self.np_topo, self.n = topo.astype(np.int64), len(xyz)
        t64 = lambda x: torch.as_tensor(np.asarray(x, np.float64), device=dev)           # noqa: E731
        dN, w = _shape(case["element"])
        self.dN, self.S, self.Q = t64(dN), dN.shape[1], dN.shape[0]
        self.dN_mat = self.dN.permute(1, 0, 2).reshape(self.S, self.Q * 3).contiguous()
        self.X = t64(xyz)
        self.topo = torch.as_tensor(self.np_topo, device=dev)
        J = self.gradient(self.X, self.topo)
        self.V = torch.linalg.det(J).abs() * t64(w)
        self.inv = torch.linalg.inv(J)
        vol = self.V.sum(1)
        mass = torch.zeros(self.n, dtype=torch.float64, device=dev)
        mass.index_add_(0, self.topo.ravel(), (vol * DENSITY / self.S).repeat_interleave(self.S))
        self.m = mass
        young, nu = float(np.float32(case["young"])), float(np.float32(case["poisson"]))
        self.lam = young * nu / ((1 + nu) * (1 - 2 * nu))
        self.mu = young / (2 * (1 + nu))
        self.dt = float(np.float32(np.float32(case["dt"]) / np.float32(case["substeps"])))
        self.g = t64([0.0, float(np.float32(GRAVITY)), 0.0])
        self.fixed = torch.as_tensor(_fixed(xyz), device=dev)
        self.free = torch.ones(self.n, dtype=torch.bool, device=dev)    # the first sweep precedes the first fixation
        pos, last, vel = _initial(case, seed, xyz)
        self.u, self.last, self.v = t64(pos) - self.X, t64(last) - self.X, t64(vel)
        self.lo, self.hi = t64([-10.0, -5.0, -10.0]), t64([10.0, 5.0, 10.0])

    def gradient(self, x, nodes):
        """sum_k x_k (x) dN_k per point: (n, Q, 3, 3)."""
        xs = x[nodes].permute(0, 2, 1).reshape(-1, self.S)
        return (xs @ self.dN_mat).view(-1, 3, self.Q, 3).permute(0, 2, 1, 3)

    @staticmethod
    def mul(A, B):
        return (A.unsqueeze(-1) * B.unsqueeze(-3)).sum(-2)

    def deformation(self, e):
        F = self.mul(self.gradient(self.u, self.topo[e]), self.inv[e])
        return F + torch.eye(3, dtype=torch.float64, device=self.dev)

    @staticmethod
    def cofactor(F):
        a, b, c = F[..., 0], F[..., 1], F[..., 2]
        C = torch.stack([torch.linalg.cross(b, c), torch.linalg.cross(c, a), torch.linalg.cross(a, b)], -1)
        return C, (a * C[..., 0]).sum(-1)

    def node_terms(self, e, dN_r):
        """Force and Hessian block of the node whose derivatives are dN_r (n, Q, 3)."""
        F = self.deformation(e)
        C, J = self.cofactor(F)
        alpha = 1.0 + self.mu / self.lam if self.case["material"] == "stable" else 1.0
        V = self.V[e].unsqueeze(-1)
        g = (self.inv[e] * dN_r.unsqueeze(-1)).sum(-2)
        Fg, c = (F * g.unsqueeze(-2)).sum(-1), (C * g.unsqueeze(-2)).sum(-1)
        f = -(V * (self.mu * Fg + (self.lam * (J - alpha)).unsqueeze(-1) * c)).sum(1)
        gg = (self.mu * V * (g * g).sum(-1, keepdim=True)).sum((1, 2))
        H = (self.lam * V.unsqueeze(-1) * c.unsqueeze(-1) * c.unsqueeze(-2)).sum(1)
        return f, H + gg[:, None, None] * torch.eye(3, dtype=torch.float64, device=self.dev)

    def constraints(self):
        self.u[self.fixed] = 0.0
        self.v[self.fixed] = 0.0
        self.free = ~self.fixed
        x = self.X + self.u
        out = ((x < self.lo) | (x > self.hi)) & self.free[:, None]
        self.u = torch.where(out, torch.minimum(torch.maximum(x, self.lo), self.hi) - self.X, self.u)

    # -- vertex block descent
    def vbd(self):
        case, dt = self.case, self.dt
        colour = _vertex_colours(self.np_topo, self.n)
        of_inc = colour[self.np_topo]
        sweeps = []
        for c in range(colour.max() + 1):
            e, r = np.nonzero(of_inc == c)
            verts, slot = np.unique(self.np_topo[e, r], return_inverse=True)
            sweeps.append([torch.as_tensor(a, device=self.dev) for a in (e, r, slot, verts)])
        rho = float(np.float32(case["rho"]))
        k = float(np.float32(case["damping"])) / dt
        mh2 = self.m / (dt * dt)
        eye = torch.eye(3, dtype=torch.float64, device=self.dev)
        for _ in range(case["substeps"]):
            prev1 = self.u.clone()
            prev2 = getattr(self, "prev2", prev1)
            y = self.u + (self.u - self.last) + self.g * dt * dt
            self.last, self.u = self.u.clone(), y.clone()
            omega = 1.0
            for it in range(case["iterations"]):
                for e, r, slot, verts in sweeps:
                    f, H = self.node_terms(e, self.dN[:, r].permute(1, 0, 2))
                    fv = torch.zeros(len(verts), 3, dtype=torch.float64, device=self.dev).index_add_(0, slot, f)
                    Hv = torch.zeros(len(verts), 3, 3, dtype=torch.float64, device=self.dev).index_add_(0, slot, H)
                    if k > 0.0:
                        fv = fv - k * (Hv * (self.u[verts] - self.last[verts]).unsqueeze(1)).sum(-1)
                        Hv = Hv * (1.0 + k)
                    w = mh2[verts]
                    fv = fv - w[:, None] * (self.u[verts] - y[verts])
                    du = torch.linalg.solve(Hv + w[:, None, None] * eye, fv.unsqueeze(-1)).squeeze(-1)
                    self.u[verts] += du * self.free[verts][:, None]
                self.constraints()
                if rho > 0.0:
                    omega = 2.0 / (2.0 - rho * rho) if it == 1 else 4.0 / (4.0 - rho * rho * omega) if it > 1 else omega
                    if it >= 2:
                        self.u = prev2 + omega * (self.u - prev2)
                    prev2, prev1 = prev1, self.u.clone()
            self.prev2 = prev2
            self.v = (self.u - self.last) / dt

    # -- XPBD
    def xpbd_energy(self, F, m):
        C, J = self.cofactor(F)
        J_, s = J[..., None, None], self.case["material"] == "stable"
        if m == 0:
            rest = 1.0 if s else 1.0 + self.mu / self.lam
            return (J - rest) ** 2, 2.0 * (J_ - rest) * C
        e = (F * F).sum((-1, -2)) - 3.0
        return (e - 2.0 * (J - 1.0), 2.0 * F - 2.0 * C) if s else (e, 2.0 * F)

    def xpbd(self):
        case, dt = self.case, self.dt
        colour = _element_colours(self.np_topo)
        groups = [torch.as_tensor(np.nonzero(colour == c)[0], device=self.dev) for c in range(colour.max() + 1)]
        w = 1.0 / self.m
        damp = float(np.float32(case["damping"]))
        for _ in range(case["substeps"]):
            self.last = self.u.clone()
            self.v = self.v + self.g * dt
            self.u = self.u + self.v * dt
            for e in groups:
                nodes = self.topo[e]
                wn = w[nodes].unsqueeze(-1)
                for m, k in ((0, self.lam), (1, self.mu)):
                    energy, P = self.xpbd_energy(self.deformation(e), m)
                    V = self.V[e]
                    C = (energy * V).sum(1)
                    Ps = self.mul(P, self.inv[e].transpose(-1, -2)) * V[..., None, None]
                    grad = torch.einsum("nqij,qsj->nsi", Ps, self.dN)
                    if self.S == 4:
                        C = C.abs().sqrt()
                        grad = grad * torch.where(C < 1e-12, 0.0, 0.5 / C)[:, None, None]
                        step = -C / ((grad * grad * wn).sum((1, 2)) + 1.0 / (k * dt * dt))
                        move = step[:, None, None] * wn * grad * self.free[nodes].unsqueeze(-1)
                    else:
                        step = -2.0 * C / ((grad * grad * wn).sum((1, 2)) + 4.0 * C / (k * dt * dt))
                        move = torch.where(C < 1e-12, 0.0, step)[:, None, None] * wn * grad
                    self.u.index_add_(0, nodes.ravel(), move.reshape(-1, 3))
            self.constraints()
            self.v = (self.u - self.last) / dt
            if damp > 0.0:
                self.v = self.v * (1.0 - torch.clamp(damp * dt * w, max=1.0))[:, None]

    # -- explicit
    def explicit(self):
        dt, k = self.dt, float(np.float32(self.case["damping"]))
        every = torch.arange(len(self.topo), device=self.dev)
        chunk = max(1, 40_000_000 // (self.Q * self.S * 9))
        for _ in range(self.case["substeps"]):
            f = torch.zeros_like(self.u)
            H = torch.zeros(self.n, 3, 3, dtype=torch.float64, device=self.dev)
            for e in every.split(chunk):
                self.element_forces(e, f, H if k else None)
            if k:
                f = f - k * (H * self.v.unsqueeze(1)).sum(-1)
            self.last = self.u.clone()
            self.v = self.v + (self.g + f / self.m[:, None]) * dt
            self.u = self.u + self.v * dt
            self.constraints()

    def element_forces(self, e, f, H):
        F = self.deformation(e)
        C, J = self.cofactor(F)
        alpha = 1.0 + self.mu / self.lam if self.case["material"] == "stable" else 1.0
        V = self.V[e][..., None, None]
        inv_t = self.inv[e].transpose(-1, -2)
        P = self.mul(V * (self.mu * F + self.lam * (J[..., None, None] - alpha) * C), inv_t)
        nodes = self.topo[e].ravel()
        f.index_add_(0, nodes, -torch.einsum("nqij,qsj->nsi", P, self.dN).reshape(-1, 3))
        if H is not None:
            K, G = self.mul(C, inv_t), self.mul(self.inv[e], inv_t)
            c = torch.einsum("nqij,qsj->nqsi", K, self.dN)
            gg = (torch.einsum("nqij,qsj->nqsi", G, self.dN) * self.dN).sum(-1) * V[..., 0] * self.mu
            h = (self.lam * V.unsqueeze(-1) * c.unsqueeze(-1) * c.unsqueeze(-2)).sum(1)
            eye = torch.eye(3, dtype=torch.float64, device=self.dev)
            H.index_add_(0, nodes, (h + gg.sum(1)[..., None, None] * eye).reshape(-1, 3, 3))

    def out(self, name):
        x = {"positions": self.X + self.u, "last_positions": self.X + self.last, "velocities": self.v}[name]
        return x.cpu().numpy()


def exact(case, seed):
    if case["kind"] in ("batch", "served"):
        # the smaller scenes, while they fit the time
        parts = _parts(case)
        pos, vel, left = [None] * len(parts), [None] * len(parts), 60000
        for i in sorted(range(len(parts)), key=lambda j: _counts(parts[j])[0]):
            left -= _counts(parts[i])[0]
            if left < 0:
                break
            x = _Exact(parts[i], seed * 1000 + i)
            x.vbd()
            pos[i], vel[i] = x.out("positions"), x.out("velocities")
        return {"positions": pos, "velocities": vel}
    x = _Exact(case, seed)
    getattr(x, case["kind"])()
    return {k: x.out(k) for k in (("positions", "last_positions") if case["kind"] == "xpbd" else
                                  ("positions", "velocities"))}
