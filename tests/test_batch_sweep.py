"""Batched one-sweep steps: members of every kind advanced together against
two-kernel sims stepped alone; every value must agree."""

import numpy as np
import pytest

import gmes_amd as g
from gmes_amd.batch import Batch

from test_step1d import line
from test_step2d import plane
from test_step3d import box, media_box

pytestmark = pytest.mark.gpu


def members(lib, precision, bloch):
    kw = dict(precision=precision, bloch=bloch)
    out = [plane(lib, "tmz", (40, 190), bound=g.Cpml, media=True, **kw), plane(lib, "tez", (31, 300), bound=g.Upml, **kw),
           plane(lib, "tmz", (9, 256), **kw), plane(lib, "tez", (12, 257), sources=3, **kw), line(lib, "z", 300, **kw)]
    if not (precision == "fp64" and bloch is not None):
        out += [box(lib, (14, 12, 13), bound=g.Cpml, **kw), box(lib, (40, 33, 64), bound=g.Cpml, axes="xy", **kw),
                box(lib, (12, 11, 200), bound=g.Upml, **kw), box(lib, (9, 8, 30), **kw),
                box(lib, (10, 12, 13), bound=g.Cpml, over_shell=True, **kw),  # two-kernel steps
                box(lib, (9, 9, 300), bound=g.Cpml, **kw),                    # the same: long rows
                media_box(lib, (22, 21, 24), **kw), media_box(lib, (20, 19, 30), media=False, **kw),
                media_box(lib, (22, 21, 24), wave=False, seam=False, bound=g.Cpml, **kw)]
    return out


@pytest.mark.parametrize("precision,bloch", [("fp32", None), ("fp64", None), ("fp32", (0.3, -0.2, 0.0)),
                                             ("fp64", (0.3, -0.2, 0.0))], ids=["fp32", "fp64", "c64", "c128"])
@pytest.mark.parametrize("graph", [True, False], ids=["graph", "direct"])
def test_members_match_alone(engine_lib, precision, bloch, graph):
    a, b = members(engine_lib, precision, bloch), members(engine_lib, precision, bloch)
    for s in b:
        engine_lib.set_ghost_fusion(s._sim, 0)
    mons = [[engine_lib.add_probe(s._sim, c.index, 3) for c in s._active] for s in a + b]
    batch = Batch(a, graph=graph)

    def agree():
        for q, (x, y) in enumerate(zip(a, b)):
            for c in x._active:
                u, v = np.array(x.field[c]), np.array(y.field[c])
                assert np.abs(v).max() > 0
                np.testing.assert_array_equal(u, v, err_msg="member %d %s" % (q, c.__name__))

    for k in (1, 6, 3, 2, 9):
        batch.advance(k)
        for s in b:
            s._advance(k)
        agree()
    # alone, and back to the batch
    for s in a + b:
        s._advance(3)
    agree()
    batch.advance(5)
    for s in b:
        s._advance(5)
    agree()
    for x, y, px, py in zip(a, b, mons, mons[len(a):]):
        for p, q in zip(px, py):
            u, v = engine_lib.read_probe(x._sim, p), engine_lib.read_probe(y._sim, q)
            assert len(u) == 29
            np.testing.assert_array_equal(u, v)
    batch.close()
