"""An XPBD projection moves all nodes of an element by one multiplier times the
gradient of its energy, w_k beta g_k with sum_k g_k = 0, so without gravity it
leaves an element's momentum as it was.

4,000 quadratic tetrahedra that share no vertex (one colour), Stable Neo-Hookean
(at rest undeformed), deformed by up to 1e-3 of their size, one substep.  Two constraints round every stored node value
(10 nodes, 2^-24 of at most twice the largest displacement: 2.4e-6 of it) and
the gradient sums (12 roundings of each of 10 nodes' corrections, at most the
displacement: 7.2e-6); the velocity adds 6e-7.  Bound: 1.1e-5 of the largest
displacement of the element.  Multipliers that differ between nodes by the
rounding of an energy that is nearly zero are over it by a factor of 100."""
import numpy as np
import pytest

import octopusengine_amd as oe
from meshes import P2_EDGES

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("seed", [0, 1])
def test_p2_projection_keeps_momentum(engine, seed):
    size, n, dt = 0.02, 4000, 1e-3
    corner = np.array([(0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1)], np.float64) * size
    ref = np.concatenate([corner, [(corner[i] + corner[j]) / 2 for i, j in P2_EDGES]]).astype(np.float32)
    rest = np.tile(ref, (n, 1))
    s = oe.Scene(engine, oe.TETRA10, rest, np.arange(10 * n, dtype=np.int32).reshape(n, 10), material=oe.STABLE_NEOHOOKE,
                 young=1e6, poisson=0.45, solver=oe.SOLVER_XPBD, distribution=oe.MASS_UNIFORM, gravity=(0.0, 0.0, 0.0))
    u = np.random.default_rng(seed).uniform(-1e-3, 1e-3, rest.shape) * size
    p = (rest + u).astype(np.float32)
    s.set_state(p=p, last_p=p, v=np.zeros_like(p))
    s.step(dt, 1)
    d = s.velocities().astype(np.float64).reshape(n, 10, 3) * dt   # equal masses: momentum over mass
    u = (p.astype(np.float64) - rest).reshape(n, 10, 3)
    u_max = np.abs(u).max((1, 2))
    moved = np.median(np.abs(d).max((1, 2)) / u_max)
    assert 0.1 < moved < 1.0   # the projection moves the nodes, by no more than they were displaced
    off = np.abs(d.sum(1)).max(1) / u_max
    print(f"largest momentum {off.max():.2e} of the displacement, {(off > 1.1e-5).sum()} elements over", flush=True)
    assert off.max() <= 1.1e-5
    s.close()
