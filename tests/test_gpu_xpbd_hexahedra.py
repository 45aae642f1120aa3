"""XPBD on 8-node hexahedra at the line between its two forms (32 lanes per
element in colours of up to 2,048 elements, 8 lanes past that)."""
import numpy as np
import pytest

import octopusengine_amd as oe
import pyoracle as O
from scenes import max_err

pytestmark = pytest.mark.gpu
MATERIALS = [oe.NEOHOOKE, oe.STABLE_NEOHOOKE]


@pytest.mark.parametrize("material", MATERIALS)
@pytest.mark.parametrize("n", [2047, 2048, 2049, 2055])
def test_copies_of_a_hexahedron_stay_copies(engine, n, material):
    """n hexahedra that share no vertex (one colour of n elements) and start as
    copies of one another: each lane group, in whole blocks and in a last block
    of 1 or 7, gives the same bits."""
    ref, one = oe.beam_mesh(oe.HEXA, (1, 1, 1), (0.1, 0.1, 0.1))
    xyz = np.tile(ref, (n, 1))
    topo = (one + 8 * np.arange(n)[:, None]).astype(np.int32)
    assert np.bincount(oe.host_color_dual(oe.HEXA, topo, len(xyz))[0]).tolist() == [n]
    s = oe.Scene(engine, oe.HEXA, xyz, topo, material=material, young=1e6, poisson=0.45, solver=oe.SOLVER_XPBD)
    p = np.tile((ref + np.random.default_rng(1).uniform(-1e-3, 1e-3, ref.shape)).astype(np.float32), (n, 1))
    s.set_state(p=p, last_p=p, v=np.zeros_like(p))
    s.step(0.01, 10)
    x = s.positions().reshape(n, 8, 3)
    assert np.abs(x[0] - p[:8]).max() > 1e-4
    assert np.array_equal(x, np.broadcast_to(x[0], x.shape))
    s.close()


@pytest.mark.parametrize("material", MATERIALS)
def test_both_forms_match_the_oracle(engine, material):
    """A beam with colours on both sides, against the FP64 oracle: max vertex
    error <= 1e-5 of the bounding-box diagonal after one frame."""
    xyz, topo = oe.beam_mesh(oe.HEXA, (41, 20, 21), (1.0, 0.5, 0.5))
    sizes = np.bincount(oe.host_color_dual(oe.HEXA, topo, len(xyz))[0])
    assert sizes.max() > 2048 > sizes.min()
    kw = dict(material=material, young=1e6, poisson=0.45, solver=oe.SOLVER_XPBD)
    s, o = oe.Scene(engine, oe.HEXA, xyz, topo, **kw), O.Scene(oe.HEXA, xyz, topo, **kw)
    p = (xyz + np.random.default_rng(1).uniform(-1e-3, 1e-3, xyz.shape)).astype(np.float32)
    s.set_state(p=p, last_p=p, v=np.zeros_like(p))
    o.set("p", p.astype(np.float64))
    o.set("last_p", p.astype(np.float64))
    s.step(0.01, 10)
    o.step(0.01, 10)
    moved = np.abs(o.positions() - p).max()
    err = max_err(s.positions(), o.positions())
    print(f"material {material}: colours {sizes.tolist()} moved {moved:.2e} err {err:.2e}", flush=True)
    assert moved > 1e-4
    assert err <= 1e-5 * 1.5 ** 0.5
    s.close()
