"""Batches whose scenes are dealt into several groups side by side (a group keeps
at least 4e5 (incidence, quadrature point) pairs per colour pass): the same
positions, bit for bit, as on one stream, eagerly and replayed from a graph with
host reads between.  Groups share nothing, so there is nothing to differ by."""
import numpy as np
import pytest

import octopusengine_amd as oe

pytestmark = pytest.mark.gpu

BIG = (64, 16, 16)      # 98,304 P2 tetrahedra: about 3.6e5 pairs per pass
BATCHES = {
    "three groups of one type": [(oe.TETRA10, BIG, 2)] * 6,
    "two groups and the hexahedra": [(oe.TETRA10, BIG, 2)] * 4 + [(oe.HEXA27, (4, 2, 2), 3)] * 2,
    "other types beside": [(oe.TETRA10, BIG, 1), (oe.HEXA, BIG, 3), (oe.TETRA, BIG, 2), (oe.TETRA10, BIG, 2),
                           (oe.TETRA20, (6, 3, 3), 2), (oe.HEXA27, (12, 6, 6), 2)],
}


@pytest.mark.parametrize("name", list(BATCHES))
def test_groups_give_the_same_steps(engine, name):
    sets, batches = [], []
    for _ in range(3):
        s = [oe.make_scene(engine, el, cells, iterations=it) for el, cells, it in BATCHES[name]]
        sets.append(s)
        batches.append(oe.Batch(engine, s))
    batches[0].set_streams(1)
    batches[2].set_graph(True)
    for i in range(3):
        for b in batches:
            b.step(0.005, 2)
        for one, eager, graph in zip(*sets):
            p = one.positions()
            assert np.array_equal(p, eager.positions()), f"step {i}, eager"
            assert np.array_equal(p, graph.positions()), f"step {i}, graph"
    for b in batches:
        b.close()
    for s in sets:
        for x in s:
            x.close()
