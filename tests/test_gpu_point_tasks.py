"""Point tasks (an element's points spread over lanes) where they can go wrong:
partial blocks, a block's last group, curved (per-point) records, vertices of
more elements than a block takes at a time, both sides of the line between the
quadratic tetrahedra's forms.  Against the FP64 oracle, max vertex error <= 1e-5
of the bounding-box diagonal after 2 steps (the bound of one step, doubled)."""
import numpy as np
import pytest

import octopusengine_amd as oe
import pyoracle as O
from meshes import hex_book
from scenes import make_pair, max_err

pytestmark = pytest.mark.gpu


def check(g, o, xyz):
    for _ in range(2):
        g.step(0.005, 1)
        o.step(0.005, 1)
    diag = float(np.linalg.norm(xyz.max(0) - xyz.min(0)))
    err = max_err(g.positions(), o.positions())
    assert err <= 2e-5 * diag, err


@pytest.mark.parametrize("curve", [0.0, 0.02], ids=["straight", "curved"])
@pytest.mark.parametrize("el,cells", [(3, (1, 1, 1)), (3, (9, 4, 3)), (6, (1, 1, 1)), (6, (5, 3, 2)), (6, (9, 5, 7)),
                                      (7, (1, 1, 1)), (7, (5, 2, 3)), (7, (20, 9, 9)), (8, (1, 1, 1)), (8, (3, 2, 1)),
                                      (8, (6, 3, 3))])
def test_beams_match_the_oracle(engine, el, cells, curve):
    g, o, rest, _ = make_pair(engine, el, cells, young=1e6, poisson=0.45, noise=1e-4, seed=2, curve=curve, damping=1e-3)
    assert g.get_tile()[2] == oe.PASS_TASKS
    check(g, o, rest)


def test_vertices_of_many_hexahedra(engine):
    """40 8-node hexahedra around an axis: its vertices take two rounds of 32."""
    xyz, topo = hex_book(40)
    used, topo = np.unique(np.asarray(topo)[:, :8], return_inverse=True)
    xyz, topo = np.ascontiguousarray(xyz[used]), topo.reshape(-1, 8).astype(np.int32)
    fixed = np.nonzero(xyz[:, 2] < 1e-6)[0].astype(np.int32)
    g = oe.Scene(engine, oe.HEXA, xyz, topo, material=3, young=1e5, poisson=0.45, iterations=10)
    o = O.Scene(6, xyz, topo, material=3, young=1e5, poisson=0.45, iterations=10)
    g.fix_vertices(fixed)
    o.fix(fixed)
    assert g.get_tile()[2] == oe.PASS_TASKS
    check(g, o, xyz)


def test_quadratic_forms_agree(engine):
    """Split form (the default of a launch of few incidences) against the
    throughput form (latency_blocks = 0): the same terms, one float ulp of a
    coordinate below 1 m after a step."""
    out = []
    for lat in (512, 0):
        s = oe.make_scene(engine, oe.TETRA10, (8, 4, 3))
        s.set_tile_ex(mode=oe.PASS_TASKS, latency_blocks=lat)
        s.step(0.005, 1)
        out.append(s.positions().astype(np.float64))
        s.close()
    assert np.abs(out[0] - out[1]).max() <= 6e-8
