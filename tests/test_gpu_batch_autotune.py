"""The batch tuner times the layout that a batch starts with beside its own list
(gathers, cached gradients, block sizes at one latency threshold), so that
tuning cannot end on a layout it timed slower than the start.  Small batches of
quadratic elements start with thresholds that the list does not have."""
import numpy as np
import pytest

import octopusengine_amd as oe

pytestmark = pytest.mark.gpu

LANES, CACHED = 5, 5   # 4 .. 64 lanes, and the same with cached gradients
LISTED = {oe.TETRA: LANES * 1 + CACHED + 3, oe.TETRA10: LANES * 3 + CACHED + 3, oe.HEXA27: LANES * 4 + CACHED + 7}


def test_the_start_is_among_the_candidates(engine):
    oe.autotune_clear()
    scenes = [oe.make_scene(engine, el, (4, 2, 2)) for el in LISTED]
    b = oe.Batch(engine, scenes)
    start = {el: b.get_tile_ex(el) for el in LISTED}
    assert start[oe.TETRA10]["latency_blocks"] != 512 and start[oe.HEXA27]["latency_blocks"] != 512
    b.set_tile(oe.TETRA10, 16, 1, oe.PASS_GATHER)   # what it starts with, not what it was set to
    b.autotune()
    recs = {r["element"]: r for r in oe.autotune_cache() if r["form"] == "batch"}
    for el, n in LISTED.items():
        print(f"element {el}: {recs[el]}", flush=True)
        assert recs[el]["candidates"] == n + (start[el]["latency_blocks"] != 512)
    b.step(0.005, 1)
    assert all(np.isfinite(s.positions()).all() for s in scenes)
    b.close()
    for s in scenes:
        s.close()
    oe.autotune_clear()
