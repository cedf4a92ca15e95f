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
