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
