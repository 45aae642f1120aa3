"""The per-vertex pass between sweeps (constraints, Chebyshev, velocity, next
predictor in one launch): n substeps in one call equal n calls of one substep
bit for bit, for every constraint list that takes another route (none,
fixation, box, both, and two boxes, which run one by one), and a scene with two
equal boxes equals the scene with one."""
import numpy as np
import pytest

import octopusengine_amd as oe

pytestmark = pytest.mark.gpu

DT = 1.0 / 256.0   # dt * n / n is exact
LO, HI = (-10.0, -0.01, -10.0), (10.0, 0.255, 10.0)   # clamps the bent beam
KINDS = {
    "vbd": dict(solver=oe.SOLVER_VBD, iterations=3),
    "vbd-chebyshev": dict(solver=oe.SOLVER_VBD, iterations=4, rho=0.75),
    "vbd-no-iterations": dict(solver=oe.SOLVER_VBD, iterations=0, rho=0.75),
    "xpbd": dict(solver=oe.SOLVER_XPBD, global_damping=1.0),
    "explicit": dict(solver=oe.SOLVER_EXPLICIT, damping=1e-5),
}


def make(engine, kind, constraints):
    xyz, topo = oe.beam_mesh(oe.TETRA10, (7, 2, 3), (1.0, 0.25, 0.25))   # 525 vertices: two blocks and a part
    s = oe.Scene(engine, oe.TETRA10, xyz, topo, material=oe.NEOHOOKE, young=1e5, poisson=0.4, **KINDS[kind])
    for c in constraints:
        if c == "fix":
            s.fix_plane((1e-6, 0.0, 0.0), (-1.0, 0.0, 0.0))
        else:
            s.box_limit(LO, HI)
    x = xyz[:, 0:1]
    p = (xyz + x * x * np.float32([0.0, -0.06, 0.01])).astype(np.float32)
    v = (x * x * np.float32([0.0, -2.0, 0.3])).astype(np.float32)
    s.set_state(p=p, last_p=(p - v * np.float32(DT)).astype(np.float32), v=v)
    return s


def state(s):
    return [s.positions(), s.last_positions(), s.velocities(), s.forces(), s.masks()]


@pytest.mark.parametrize("constraints", [(), ("fix",), ("box",), ("fix", "box"), ("fix", "box", "box")],
                         ids=["none", "fix", "box", "fix+box", "fix+2box"])
@pytest.mark.parametrize("kind", KINDS)
def test_substeps_equal_single_steps(engine, kind, constraints):
    dt = DT / 64 if kind == "explicit" else DT
    many, one = make(engine, kind, constraints), make(engine, kind, constraints)
    many.step(3 * dt, 3)
    many.step(2 * dt, 2)
    for _ in range(5):
        one.step(dt, 1)
    for a, b in zip(state(many), state(one)):
        assert np.array_equal(a, b)
    p = many.positions()
    assert np.isfinite(p).all()
    free = many.masks() != 0
    if "box" in constraints and kind != "vbd-no-iterations":
        clamped = (p[free] <= np.float32(LO)) | (p[free] >= np.float32(HI))
        assert kind == "vbd-chebyshev" or (p[free] >= np.float32(LO) - 1e-6).all()   # the acceleration follows the box
        assert clamped.any()
    if len(constraints) == 3:
        single = make(engine, kind, constraints[:2])
        single.step(3 * dt, 3)
        single.step(2 * dt, 2)
        for a, b in zip(state(many), state(single)):
            assert np.array_equal(a, b)
    for s in (many, one):
        s.close()


def _disjoint_tetrahedra(n):
    """n unit-corner tetrahedra apart from each other: one colour of n elements."""
    ref = np.float32([(0, 0, 0), (0.02, 0, 0), (0, 0.02, 0), (0, 0, 0.02)])
    at = np.stack(np.meshgrid(np.arange(24), np.arange(24), [0.0], indexing="ij"), -1).reshape(-1, 3)[:n]
    xyz = (at[:, None, :] * 0.04 + ref[None]).reshape(-1, 3).astype(np.float32)
    return xyz, np.arange(4 * n, dtype=np.int32).reshape(n, 4)


@pytest.mark.parametrize("material", [oe.NEOHOOKE, oe.STABLE_NEOHOOKE])
@pytest.mark.parametrize("mesh", [(1, 1, 1), (16, 4, 4), (35, 8, 6), (36, 8, 6), "disjoint"], ids=str)
def test_small_linear_xpbd_equals_its_launches(engine, mesh, material):
    """The one-workgroup run of a small linear XPBD scene (up to 2,304 vertices:
    35x8x6 has 2,268, 36x8x6 has 2,331 and is launched colour by colour; 576
    disjoint tetrahedra give one colour of more elements than threads) against
    the launches of the same scene with its box limit added twice."""
    xyz, topo = _disjoint_tetrahedra(576) if mesh == "disjoint" else oe.beam_mesh(oe.TETRA, mesh, (1.0, 0.25, 0.25))
    scenes = []
    for boxes in (1, 2):
        s = oe.Scene(engine, oe.TETRA, xyz, topo, material=material, young=1e6, poisson=0.45, solver=oe.SOLVER_XPBD,
                     global_damping=0.5)
        s.fix_plane((1e-6, 0.0, 0.0), (-1.0, 0.0, 0.0))
        for _ in range(boxes):
            s.box_limit(LO, HI)
        rng = np.random.default_rng(5)
        p = (xyz + rng.uniform(-1e-3, 1e-3, xyz.shape)).astype(np.float32)
        s.set_state(p=p, last_p=p, v=rng.standard_normal(xyz.shape).astype(np.float32))
        for n in (1, 7, 20):
            s.step(1e-3 * n, n)
        scenes.append(s)
    for a, b in zip(state(scenes[0]), state(scenes[1])):
        assert np.array_equal(a, b)
    assert np.isfinite(scenes[0].positions()).all()
    for s in scenes:
        s.close()
