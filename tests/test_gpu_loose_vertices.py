"""Vertices that no element uses, in front of a mesh (with uniform masses they
are particles: they fall, and constraints act on them).  They have no partial
sums, so the vertex blocks of the task passes leave them out: packed like any
other, such a slot could sit in a block whose rows of partials are all taken, or
in one without incidences, and its sum would be another slot's row or past the
block's last.

The blocks on the CPU, for meshes that would have such blocks; then those meshes
on the GPU against the FP64 oracle, max vertex error <= 1e-5 of the bounding-box
diagonal a step."""
import subprocess
from pathlib import Path

import numpy as np
import pytest

import octopusengine_amd as oe
import pyoracle as O
from meshes import tet_fan
from octopusengine_amd import _lib as L
from scenes import max_err

HERE = Path(__file__).resolve().parent


def mesh(kind, n_loose):
    """(element, vertices with n_loose unused ones in front, topology)."""
    el, cells = kind
    xyz, topo = tet_fan(128) if cells == "fan" else oe.beam_mesh(el, cells, (1.0, 0.25, 0.25))
    loose = np.random.default_rng(4).uniform([0.5, 0.0, 0.0], [2.0, 0.25, 0.25], (n_loose, 3)).astype(np.float32)
    loose[0] = (0.0, 0.1, 0.1)   # fixed with the x = 0 face
    return el, np.concatenate([loose, xyz]), (topo + n_loose).astype(np.int32)


Q2A, Q2B, FAN = (oe.HEXA27, (2, 2, 2)), (oe.HEXA27, (4, 2, 2)), (oe.TETRA, "fan")
OTHERS = [(oe.TETRA, (5, 2, 2)), (oe.HEXA, (4, 2, 2)), (oe.TETRA10, (4, 2, 2)), (oe.TETRA20, (2, 1, 1))]


@pytest.fixture(scope="module")
def vertex_blocks(tmp_path_factory):
    """The engine's block builder: (incidences of every slot, blocks)."""
    exe = tmp_path_factory.mktemp("blocks") / "vertex_blocks"
    pkg = L.LIB_PATH.parent
    subprocess.run(["g++", "-std=c++17", f"-I{pkg / 'csrc'}", str(HERE / "vertex_blocks.cpp"), str(L.LIB_PATH),
                    f"-Wl,-rpath,{pkg}", "-Wl,--allow-shlib-undefined", "-o", str(exe)], check=True)

    def run(el, topo, n_vertices, max_inc, max_slots):
        text = " ".join(map(str, [el, n_vertices, len(topo), max_inc, max_slots, *topo.reshape(-1)]))
        out = subprocess.run([str(exe)], input=text, capture_output=True, text=True, check=True).stdout.splitlines()
        return np.fromstring(out[0], np.int64, sep=" "), [tuple(map(int, l.split())) for l in out[1:]]
    return run


def packed(valence, max_inc, max_slots):
    """(incidences, empty slots) of the blocks that one colour's slots, by
    falling valence, would fill if none were left out."""
    out, slots, inc, empty = [], 0, 0, 0
    for nb in valence:
        if slots == max_slots or inc + nb > max_inc:
            out.append((inc, empty))
            slots = inc = empty = 0
        slots, inc, empty = slots + 1, inc + nb, empty + (nb == 0)
    return out + [(inc, empty)]


# most incidences and slots of a block: 27-node hexahedra in the latency form, linear tetrahedra
LIMITS = {Q2A: (8, 64), Q2B: (8, 64), FAN: (256, 256)}


@pytest.mark.parametrize("kind,n_loose,full", [(Q2A, 1, True), (Q2A, 140, False), (Q2B, 1, True), (Q2B, 140, False),
                                               (FAN, 1, True), (FAN, 520, False)], ids=str)
def test_blocks_hold_no_empty_slot(vertex_blocks, kind, n_loose, full):
    el, xyz, topo = mesh(kind, n_loose)
    max_inc, max_slots = LIMITS[kind]
    colors, n_colors, _ = oe.host_color_primal(el, topo, len(xyz))
    valence = np.bincount(topo.reshape(-1), minlength=len(xyz))
    would = [b for c in range(n_colors) for b in packed(np.sort(valence[colors == c])[::-1], max_inc, max_slots)]
    assert any(empty and inc == (max_inc if full else 0) for inc, empty in would)   # the mesh is one to look at
    nb, got = vertex_blocks(el, topo, len(xyz), max_inc, max_slots)
    off = np.concatenate([[0], np.cumsum(nb)])
    seen = np.zeros(len(nb), int)
    for first, slots, own, inc in got:
        assert 0 < slots <= max_slots and 0 < inc <= max_inc
        assert own == off[first] and inc == nb[first:first + slots].sum()
        assert (nb[first:first + slots] > 0).all(), (first, slots, nb[first:first + slots])
        seen[first:first + slots] += 1
    assert np.array_equal(seen, (nb > 0).astype(int))


@pytest.mark.gpu
@pytest.mark.parametrize("held", ["scene", "batch"])
@pytest.mark.parametrize("kind,n_loose", [(k, n) for k in (Q2A, Q2B) for n in (1, 140)] +
                         [(FAN, 1), (FAN, 520)] + [(k, 300) for k in OTHERS], ids=str)
def test_loose_vertices_match_the_oracle(engine, kind, n_loose, held):
    el, xyz, topo = mesh(kind, n_loose)
    g = oe.Scene(engine, el, xyz, topo, material=3, young=1e6, poisson=0.45, distribution=oe.MASS_UNIFORM)
    o = O.Scene(el, xyz, topo, material=3, young=1e6, poisson=0.45, femshape=False)
    fixed = np.nonzero(xyz[:, 0] < 1e-6)[0].astype(np.int32)
    g.fix_vertices(fixed)
    o.fix(fixed)
    g.box_limit((-10.0, -5.0, -10.0), (10.0, 5.0, 10.0))
    o.box((-10.0, -5.0, -10.0), (10.0, 5.0, 10.0))
    assert g.get_tile()[2] == oe.PASS_TASKS
    b = oe.Batch(engine, [g]) if held == "batch" else g
    for _ in range(2):
        b.step(0.005, 1)
        o.step(0.005, 1)
    err = max_err(g.positions(), o.positions())
    print(f"{kind} + {n_loose} loose, {held}: err {err:.2e}", flush=True)
    assert err <= 2e-5 * float(np.linalg.norm(xyz.max(0) - xyz.min(0)))
    assert np.abs(g.positions() - xyz)[1:n_loose, 1].min(initial=1.0) > 1e-4   # the free particles fall
    if held == "batch":
        b.close()
    g.close()


@pytest.mark.gpu
@pytest.mark.parametrize("rho", [0.0, 0.8])
@pytest.mark.parametrize("kind", [Q2A, OTHERS[0], OTHERS[2]], ids=str)
def test_loose_vertices_on_a_floor(engine, kind, rho):
    """A box floor in the fall of the loose vertices: the task passes, which
    leave them out, give the bits of the gather, which solves them."""
    el, xyz, topo = mesh(kind, 40)
    xyz[1:40, 1] = np.float32(0.25) * np.random.default_rng(5).uniform(0.0, 0.02, 39).astype(np.float32)
    out = []
    for mode in (oe.PASS_TASKS, oe.PASS_GATHER):
        s = oe.Scene(engine, el, xyz, topo, material=3, young=1e6, poisson=0.45, distribution=oe.MASS_UNIFORM, rho=rho)
        s.fix_vertices(np.nonzero(xyz[:, 0] < 1e-6)[0].astype(np.int32))
        s.box_limit((-10.0, -0.001, -10.0), (10.0, 5.0, 10.0))
        s.set_tile(16, 1, mode)
        s.step(0.03, 6)
        out.append([a[:40] for a in (s.positions(), s.last_positions(), s.velocities())])
        s.close()
    for a, b in zip(*out):
        assert np.array_equal(a, b)
    low = out[0][0][1:, 1] <= -0.001 + 1e-6
    assert low.any() and not low.all()
