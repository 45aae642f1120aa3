"""Batches and servers of meshes with a vertex of more elements than a task
block holds (256): the element type starts with the gather there, as the single
scene does, and every scene steps like its twin alone; a task layout is refused
with such a scene, and a layout that a server was told is kept."""
import numpy as np
import pytest

import octopusengine_amd as oe
from meshes import hex_book, p1_to_p2, tet_fan
from scenes import max_err

pytestmark = pytest.mark.gpu


def fan(el):
    """A mesh of `el` with a vertex of 600 (or 520) elements."""
    if el == oe.TETRA:
        return tet_fan(300)
    if el == oe.HEXA:
        xyz, topo = hex_book(260)
        used, topo = np.unique(np.asarray(topo)[:, :8], return_inverse=True)
        xyz, topo = np.ascontiguousarray(xyz[used]), topo.reshape(-1, 8)
        # a second layer, so that the axis vertex between has 520 elements
        top = xyz + np.float32([0.0, 0.0, 1.0])
        both, inv = np.unique(np.concatenate([xyz, top]).round(6), axis=0, return_inverse=True)
        inv = inv.reshape(-1)
        return both.astype(np.float32), np.concatenate([inv[topo], inv[topo + len(xyz)]]).astype(np.int32)
    raise ValueError(el)


def make(engine, el, mesh=None):
    if mesh is None:
        return oe.make_scene(engine, el, (6, 2, 2), young=1e5, poisson=0.45)
    s = oe.Scene(engine, el, *mesh, material=3, young=1e5, poisson=0.45, iterations=5)
    s.fix_vertices(np.nonzero(mesh[0][:, 2] < -0.4 if el == oe.TETRA else mesh[0][:, 2] < 1e-6)[0].astype(np.int32))
    return s


@pytest.mark.parametrize("el", [oe.TETRA, oe.HEXA])
@pytest.mark.parametrize("held", ["batch", "server"])
def test_fans_step_like_their_scenes(engine, el, held):
    mesh = fan(el)
    assert np.bincount(mesh[1].reshape(-1)).max() > 256
    shapes = [(el, None), (el, mesh), (oe.TETRA10, None)]
    together, alone = ([make(engine, *s) for s in shapes] for _ in range(2))
    if held == "batch":
        b = oe.Batch(engine, together)
        step = lambda: b.step(0.005, 1)
    else:
        b = oe.Server(engine, max_batch=4, streams=2)
        slots = [b.add_scene(s) for s in together]

        def step():
            for k in slots:
                b.submit(k, 0.005, 1)
            b.drain()
    assert b.get_tile_ex(el)["mode"] == oe.PASS_GATHER
    assert b.get_tile_ex(oe.TETRA10)["mode"] == oe.PASS_TASKS
    for _ in range(2):
        step()
        for s in alone:
            s.step(0.005, 1)
    with pytest.raises(oe.OEError):
        b.set_tile_ex(el, 64, 1, oe.PASS_TASKS, 0, 512)
    for (e, m), x, y in zip(shapes, together, alone):
        err = max_err(x.positions(), y.positions())
        print(f"{held} el={e} fan={m is not None} |together-alone|={err:.2e}", flush=True)
        assert err <= 1e-6
        assert np.isfinite(x.positions()).all()
    b.close()
    for s in together + alone:
        s.close()


def test_server_keeps_a_layout_it_was_told(engine):
    """A server told to run task passes refuses the fan, as it would refuse
    them with the fan in it."""
    srv = oe.Server(engine, max_batch=4, streams=1)
    srv.set_tile_ex(oe.TETRA, 64, 1, oe.PASS_TASKS, 0, 512)
    s = make(engine, oe.TETRA, fan(oe.TETRA))
    with pytest.raises(oe.OEError):
        srv.add_scene(s)
    assert srv.get_tile_ex(oe.TETRA)["mode"] == oe.PASS_TASKS
    s.step(0.005, 1)   # still its own
    srv.close()
    s.close()


def test_a_refused_scene_leaves_the_server_as_it_was(engine):
    """A quadratic fan is refused; scenes added after it keep their own fixed
    vertices when the layout is set anew."""
    cells = (6, 2, 2)
    fixings = [((1e-6, 0.0, 0.0), (-1.0, 0.0, 0.0)), ((1.0 - 1e-6, 0.0, 0.0), (1.0, 0.0, 0.0))]

    def beam(fix):
        s = oe.make_scene(engine, oe.TETRA10, cells, young=1e5, poisson=0.45, fix_x0=False)
        s.fix_plane(*fix)
        return s
    held, alone = ([beam(f) for f in fixings] for _ in range(2))
    refused = oe.Scene(engine, oe.TETRA10, *p1_to_p2(*tet_fan(300)), iterations=2)
    srv = oe.Server(engine, max_batch=4, streams=1)
    slots = [srv.add_scene(held[0])]
    with pytest.raises(oe.OEError):
        srv.add_scene(refused)
    slots.append(srv.add_scene(held[1]))
    assert slots == [0, 1]
    t = srv.get_tile_ex(oe.TETRA10)
    srv.set_tile_ex(oe.TETRA10, t["lanes"], t["qpl"], t["mode"], t["inc_per_block"], t["latency_blocks"])
    for _ in range(2):
        for k in slots:
            srv.submit(k, 0.005, 1)
        srv.drain()
        for s in alone:
            s.step(0.005, 1)
    for x, y in zip(held, alone):
        assert np.array_equal(x.masks(), y.masks())
        assert max_err(x.positions(), y.positions()) <= 1e-6
    refused.step(0.005, 1)
    srv.close()
    for s in held + alone + [refused]:
        s.close()
