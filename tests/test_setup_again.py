"""A committed sim that is given other materials, ids and sources before it
is committed again: the one-sweep step's tables of the first set-up must not
be used, whatever the order of the calls."""

import numpy as np
import pytest

import gmes_amd as g

from test_step1d import line
from test_step2d import plane
from test_step3d import box, media_box

pytestmark = pytest.mark.gpu


def set_up_again(lib, sim, other, aux=None):
    """Gives sim the tables of other: records, ids, an auxiliary grid and the
    sources before the commit."""
    tiles = other._tiles
    lib.set_materials(sim._sim, tiles.record_array(), tiles.coef_array())
    for c in sim._active:
        lib.set_material_ids(sim._sim, c.index, tiles.ids[c])
    for (p, ci, a), vals in tiles.profiles.items():
        lib.set_profile(sim._sim, p, ci, a, vals)
    if aux is not None:
        lib.attach_aux(sim._sim, aux._sim)
    sim.geom_tree, sim._tiles, sim.src_list = other.geom_tree, tiles, other.src_list
    sim.init_source()
    lib.commit(sim._sim)
    for c in sim._active:
        sim.field[c][...] = other.field[c]


CASES = {
    # fewer records than before, more of them, dispersive cells before or after
    "fewer_records": (lambda lib, **k: media_box(lib, (22, 21, 24), wave=False, point=(g.Ez, g.Hx), **k),
                      lambda lib, **k: media_box(lib, (22, 21, 24), wave=False, media=False, point=(g.Ez, g.Hx), **k)),
    "more_records": (lambda lib, **k: box(lib, (22, 21, 24), **k),
                     lambda lib, **k: box(lib, (22, 21, 24), bound=g.Cpml, comps=(g.Ex, g.Hy), **k)),
    "media": (lambda lib, **k: box(lib, (22, 21, 24), **k),
              lambda lib, **k: media_box(lib, (22, 21, 24), wave=False, point=(g.Ez,), **k)),
    "plane": (lambda lib, **k: plane(lib, "tmz", (31, 33), media=True, **k),
              lambda lib, **k: plane(lib, "tmz", (31, 33), bound=g.Cpml, sources=3, **k)),
    "line": (lambda lib, **k: line(lib, "z", 300, media=True, **k),
             lambda lib, **k: line(lib, "z", 300, bound=g.Upml, sources=2, **k)),
}


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("aux", [False, True], ids=["alone", "aux"])
def test_sources_before_the_commit(engine_lib, case, precision, aux):
    first, second = CASES[case]
    a, b = first(engine_lib, precision=precision), second(engine_lib, precision=precision)
    a._advance(3)
    b._advance(3)
    engine_lib.commit(b._sim)  # absorber and dispersive state from the start
    grids = [line(engine_lib, "z", 40, precision=precision) for _ in range(2)] if aux else [None, None]
    if aux:
        engine_lib.attach_aux(b._sim, grids[1]._sim)
    set_up_again(engine_lib, a, b, grids[0])
    for k in (1, 4, 5):
        for s, aux_sim in ((a, grids[0]), (b, grids[1])):
            if aux_sim is not None:
                aux_sim._prepare(k)
            s._advance(k)
        for c in a._active:
            x, y = np.array(a.field[c]), np.array(b.field[c])
            assert np.abs(y).max() > 0
            np.testing.assert_array_equal(x, y)


KINDS = {"box": lambda lib, **k: box(lib, (22, 21, 24), bound=g.Cpml, **k),
         "media": lambda lib, **k: media_box(lib, (22, 21, 24), wave=False, **k),
         "plane": lambda lib, **k: plane(lib, "tez", (31, 33), bound=g.Upml, media=True, **k),
         "line": lambda lib, **k: line(lib, "z", 300, bound=g.Cpml, media=True, **k)}


@pytest.mark.parametrize("kind", sorted(KINDS))
@pytest.mark.parametrize("what", ["commit", "aux"])
@pytest.mark.parametrize("steps", [2, 3])
def test_state_outlives_the_second_buffers(engine_lib, kind, what, steps):
    """After an even or odd number of one-sweep steps the sim is committed
    again, or (a plane or line) gets an auxiliary grid and takes two-kernel
    steps; fields, absorber words, dispersive state and monitors go on."""
    from gmes_amd.monitor import DftBox
    lib = engine_lib
    a, b = (KINDS[kind](lib, precision="fp64") for _ in range(2))
    lib.set_ghost_fusion(b._sim, 0)
    e, h = a._active[0], a._active[-1]
    mons, pids, grids = [], [], []
    for s in (a, b):
        pids.append([lib.add_probe(s._sim, c.index, 2) for c in (e, h)])
        mons.append(DftBox(s, h, (0, 0, 0), s._shape[h], [0.05, 0.1], 1))
        s._advance(steps)
        if what == "commit":
            before = [np.array(s.field[c]) for c in s._active]
            lib.commit(s._sim)
            lib.sync(s._sim)
            for c, x in zip(s._active, before):
                s._dev_newer[c] = True
                np.testing.assert_array_equal(np.array(s.field[c]), x)
        else:
            grids.append(line(lib, "z", 40, precision="fp64"))
            lib.attach_aux(s._sim, grids[-1]._sim)
            s._aux_fdtds.append(grids[-1])
    for k in (1, 4, 2):
        for s in (a, b):
            s._advance(k)
        for c in a._active:
            np.testing.assert_array_equal(np.array(a.field[c]), np.array(b.field[c]))
    np.testing.assert_array_equal(mons[0].values(), mons[1].values())
    for p, q in zip(*pids):
        x, y = lib.read_probe(a._sim, p), lib.read_probe(b._sim, q)
        assert len(x) == steps + 7
        np.testing.assert_array_equal(x, y)
