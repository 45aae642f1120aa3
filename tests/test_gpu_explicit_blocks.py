"""The explicit element pass at the edges of its blocks (64, 32, 25, 11 and 9
elements of 4, 8, 10, 20 and 27 nodes): one element, whole blocks and one or two
elements more, with and without damping, against the per-vertex gather and, on
the largest, with per-point (curved) records.

Velocities after one substep are dt f / m.  Nodes move by 3% of a cell, so strains
are about 0.03 and F is off by at most some 8 roundings of 6e-8: 1.6e-5 of the
strain, times 5 for the part of the volume term (lambda is 9 mu) - 1e-4 of the
largest velocity."""
import numpy as np
import pytest

import octopusengine_amd as oe
from scenes import make_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("curve", [0.0, 0.02], ids=["straight", "curved"])
@pytest.mark.parametrize("damping", [0.0, 1e-2], ids=["undamped", "damped"])
@pytest.mark.parametrize("el,n", [(3, 1), (3, 13), (3, 64), (6, 1), (6, 32), (6, 33), (7, 5), (7, 6), (8, 2), (8, 9),
                                  (8, 11), (9, 1), (9, 9), (9, 10)])
def test_block_edges(engine, el, n, damping, curve):
    kw = dict(size=(0.25 * n, 0.25, 0.25), solver=2, material=2, young=1e6, poisson=0.45, damping=damping,
              noise=0.0075, seed=n, curve=curve)
    v = []
    for tile in ((64, 1, oe.PASS_TASKS), (16, 1, oe.PASS_GATHER)):
        g, _, _, _ = make_pair(engine, el, (n, 1, 1), **kw)
        g.set_tile(*tile)
        assert g.get_tile_ex()["mode"] == tile[2]
        if damping:   # a velocity for the damping term to act on
            g.set_state(v=np.random.default_rng(n).uniform(-0.1, 0.1, g.velocities().shape).astype(np.float32))
        before = g.velocities().astype(np.float64)
        g.step(1e-5, 1)
        v.append(g.velocities().astype(np.float64) - before)
        g.close()
    assert np.abs(v[0]).max() > 1e-4
    assert np.abs(v[0] - v[1]).max() <= 1e-4 * np.abs(v[1]).max()
