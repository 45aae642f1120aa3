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


@pytest.mark.parametrize("el,cells,n", [(oe.HEXA27, (8, 2, 2), 1), (oe.HEXA27, (16, 4, 4), 33),
                                        (oe.HEXA27, (16, 4, 4), 60), (oe.TETRA10, (8, 2, 2), 1),
                                        (oe.TETRA10, (16, 4, 4), 12), (oe.TETRA10, (16, 4, 4), 40)])
def test_small_batches(engine, el, cells, n):
    """Batches on both sides of the lines between the forms of their passes
    against the throughput form: the same terms in another order, two ulps of a
    coordinate below 1 m after a step; and the same steps on one stream."""
    out = []
    for lat, streams in ((None, 2), (None, 1), (0, 2)):
        s = [oe.make_scene(engine, el, cells) for _ in range(n)]
        b = oe.Batch(engine, s)
        b.set_streams(streams)
        if lat is not None:
            t = b.get_tile_ex(el)
            b.set_tile_ex(el, t["lanes"], t["qpl"], oe.PASS_TASKS, t["inc_per_block"], lat)
        b.step(0.005, 1)
        out.append(np.stack([x.positions().astype(np.float64) for x in s]))
        b.close()
        for x in s:
            x.close()
    assert np.array_equal(out[0], out[1])
    assert np.abs(out[0] - out[2]).max() <= 1.2e-7
