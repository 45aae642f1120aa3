"""A vertex of infinite mass (inverse mass 0) is free, not masked: a box limit
holds it like any other vertex.  A small linear XPBD scene (one workgroup for
the whole call) against the same scene with its box limit added twice (launched
colour by colour), bit for bit."""
import numpy as np
import pytest

import octopusengine_amd as oe

pytestmark = pytest.mark.gpu


def test_box_holds_vertices_of_infinite_mass(engine):
    xyz, topo = oe.beam_mesh(oe.TETRA, (4, 2, 2), (1.0, 0.25, 0.25))
    lo, hi = np.float32([-10.0, -0.02, -10.0]), np.float32([10.0, 5.0, 10.0])
    out = []
    for boxes in (1, 2):
        s = oe.Scene(engine, oe.TETRA, xyz, topo, solver=oe.SOLVER_XPBD, density=float("inf"))
        s.fix_plane((1e-6, 0.0, 0.0), (-1.0, 0.0, 0.0))
        for _ in range(boxes):
            s.box_limit(lo, hi)
        for n in (1, 9):
            s.step(0.02 * n, n)   # falls 2 m without a box
        out.append([s.positions(), s.velocities(), s.masks()])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    free = out[0][2] != 0
    assert free.any() and (out[0][0][free, 1] >= lo[1] - 1e-6).all()
