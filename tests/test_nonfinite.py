"""Infinities, and zeros of either sign, in the fields: one-sweep steps give
the two-kernel step's values, which keep the reference's formulas (a CPML
cell's 0 times infinity is NaN, a Dielectric cell has no such product)."""

import numpy as np
import pytest

import gmes_amd as g

from test_memory import swept
from test_step1d import line
from test_step2d import plane
from test_step3d import box, media_box

pytestmark = pytest.mark.gpu


def fill(sim, seed):
    """Mostly zeros of either sign, some waves, a few infinities."""
    rng = np.random.default_rng(seed)
    for c in sim._active:
        a = sim.field[c]
        for part in ((a.real, a.imag) if np.iscomplexobj(a) else (a,)):
            x = rng.choice([0.0, -0.0, 0.5, 1.0], size=part.shape, p=[0.4, 0.4, 0.1, 0.1]) * rng.choice([1, 2], size=part.shape)
            far = rng.random(part.shape) < 2.0 / 10 ** 3
            part[...] = np.where(far, rng.choice([np.inf, -np.inf], size=part.shape), x)


def same(a, b):
    for c in a._active:
        x, y = np.array(a.field[c]), np.array(b.field[c])
        for u, v in ((x.real, y.real), (x.imag, y.imag)):
            nan = np.isnan(v)
            np.testing.assert_array_equal(np.isnan(u), nan)
            np.testing.assert_array_equal(u[~nan], v[~nan])
            np.testing.assert_array_equal(np.signbit(u[~nan]), np.signbit(v[~nan]))


TYPES = {"fp32": dict(), "fp64": dict(precision="fp64"), "c64": dict(bloch=(0.3, -0.2, 0.1))}
CASES = {"none": lambda lib, **k: box(lib, (14, 12, 13), **k),
         "upml": lambda lib, **k: box(lib, (14, 12, 13), bound=g.Upml, **k),
         "media": lambda lib, **k: media_box(lib, (22, 21, 24), wave=False, **k),
         "wave": lambda lib, **k: media_box(lib, (22, 21, 24), media=False, **k),
         "media_cpml": lambda lib, **k: media_box(lib, (22, 21, 24), wave=False, seam=False, bound=g.Cpml, **k),
         "tmz": lambda lib, **k: plane(lib, "tmz", (41, 67), bound=g.Cpml, media=True, **k),
         "tez": lambda lib, **k: plane(lib, "tez", (41, 67), bound=g.Upml, **k),
         "line": lambda lib, **k: line(lib, "z", 300, bound=g.Cpml, media=True, **k)}
for axes in ("xyz", "x", "z", "xy", "yz"):
    CASES["cpml_" + axes] = lambda lib, axes=axes, **k: box(lib, (17, 16, 70), bound=g.Cpml, axes=axes, **k)
    # blocks of several kinds in one launch
    CASES["split_" + axes] = lambda lib, axes=axes, **k: box(lib, (110, 113, 107), bound=g.Cpml, axes=axes, **k)


@pytest.mark.parametrize("case", sorted(CASES))
@pytest.mark.parametrize("kind", sorted(TYPES))
def test_values_that_are_not_finite(engine_lib, case, kind):
    a, b = (CASES[case](engine_lib, **TYPES[kind]) for _ in range(2))
    engine_lib.set_ghost_fusion(b._sim, 0)
    for s in (a, b):
        assert swept(engine_lib, s) == (s is a)
        fill(s, 3)
    for k in (1, 1, 3):
        a._advance(k)
        b._advance(k)
        same(a, b)
