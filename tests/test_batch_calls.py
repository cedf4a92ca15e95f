"""Batched calls of one, two and more steps replay captured steps that start
from either buffer set of the one-sweep members; members are stepped alone,
and take two-kernel steps in between."""

import numpy as np
import pytest

from gmes_amd.batch import Batch

from test_batch_sweep import members

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,bloch", [("fp32", None), ("fp32", (0.3, -0.2, 0.0))], ids=["fp32", "c64"])
def test_calls_of_every_length(engine_lib, precision, bloch):
    lib = engine_lib
    a, b = members(lib, precision, bloch), members(lib, precision, bloch)
    for s in b:
        lib.set_ghost_fusion(s._sim, 0)
    ids = {s: [lib.add_probe(s._sim, c.index, 3) for c in s._active] for s in a + b}
    batch = Batch(a)

    def steps(lengths):
        for k in lengths:
            batch.advance(k)
            for s in b:
                s._advance(k)
        for q, (x, y) in enumerate(zip(a, b)):
            for c in x._active:
                np.testing.assert_array_equal(np.array(x.field[c]), np.array(y.field[c]),
                                              err_msg="member %d %s" % (q, c.__name__))

    steps((1, 1, 1, 2, 3, 1, 2, 1, 4, 1, 5, 2, 3, 3))
    for s in (a[0], b[0], a[5], b[5]):
        s._advance(1)
    steps((1, 2, 3, 4, 1))
    lib.set_ghost_fusion(a[1]._sim, 0)
    steps((3, 1, 2))
    lib.set_ghost_fusion(a[1]._sim, 1)
    steps((1, 3, 2, 2, 1))
    for x, y in zip(a, b):
        for p, q in zip(ids[x], ids[y]):
            u, v = lib.read_probe(x._sim, p), lib.read_probe(y._sim, q)
            assert len(u) in (56, 57)
            np.testing.assert_array_equal(u, v)
    batch.close()
