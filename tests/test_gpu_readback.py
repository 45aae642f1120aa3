"""Read-back through the pinned halves: exact values at the sizes where the
pass can go wrong (a partial 256-record block, a whole one, one past it, and
more than one and more than two halves of 65,536 vertices)."""
import numpy as np
import pytest

import octopusengine_amd as oe

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells", [(1, 1, 1), (63, 1, 1), (64, 1, 1), (40, 40, 40), (63, 45, 45)])
@pytest.mark.parametrize("solver", [oe.SOLVER_XPBD, oe.SOLVER_VBD])
def test_state_reads_back_as_set(engine, cells, solver):
    if solver == oe.SOLVER_VBD and cells[1] > 40:
        pytest.skip("one large size is enough for the packed records")
    xyz, topo = oe.beam_mesh(oe.HEXA, cells, (1.0, 0.25, 0.25))
    s = oe.Scene(engine, oe.HEXA, xyz, topo, solver=solver)
    rng = np.random.default_rng(3)
    v = rng.standard_normal(xyz.shape).astype(np.float32)
    p = (xyz + rng.uniform(-1e-3, 1e-3, xyz.shape)).astype(np.float32)
    s.set_state(p=p, last_p=xyz, v=v)
    assert np.array_equal(s.velocities(), v)
    assert np.array_equal(s.init_positions(), xyz)
    assert np.array_equal(s.last_positions(), xyz)
    # a displacement is stored to half an ulp of itself (and to half a quantum
    # of 2^-30 m in the packed records), then X + u is rounded once
    u = np.abs(p.astype(np.float64) - xyz)
    bound = np.spacing(np.abs(p)) * 0.5 + np.maximum(u * 2.0 ** -24, 2.0 ** -30)
    assert (np.abs(s.positions().astype(np.float64) - p) <= bound).all()
    if solver == oe.SOLVER_XPBD:   # float displacements: the host's own sum, bit for bit
        d = (p.astype(np.float64) - xyz).astype(np.float32)
        assert np.array_equal(s.positions(), (xyz.astype(np.float64) + d).astype(np.float32))
    s.close()
