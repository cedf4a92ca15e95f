"""Which step a sim takes: the tests that compare a sim with a two-kernel one
mean nothing when both take the two-kernel step."""

import pytest

import gmes_amd as g

from test_memory import swept
from test_step3d import box

pytestmark = pytest.mark.gpu

FP64, C64 = dict(precision="fp64"), dict(precision="fp32", bloch=(0.3, -0.2, 0.1))

# rows too long for the bodies of an absorber: a block would own one or two
LONG = [((9, 9, 256), g.Cpml, FP64, True), ((9, 9, 257), g.Cpml, FP64, False), ((9, 9, 257), g.Upml, C64, False),
        ((9, 9, 341), None, FP64, True), ((9, 9, 341), g.Upml, dict(), True), ((9, 9, 342), None, dict(), False),
        ((40, 96, 153), g.Upml, FP64, True), ((40, 96, 154), g.Upml, FP64, False), ((40, 96, 154), g.Cpml, C64, False),
        ((40, 96, 154), g.Cpml, FP64, True), ((40, 110, 256), g.Upml, dict(), True),
        ((40, 110, 257), g.Upml, dict(), False), ((40, 110, 257), g.Cpml, dict(), True)]


@pytest.mark.parametrize("n,bound,kw,sweeps", LONG, ids=lambda v: getattr(v, "__name__", str(v)))
def test_long_rows(engine_lib, n, bound, kw, sweeps):
    sim = box(engine_lib, n, bound=bound, **kw)
    assert swept(engine_lib, sim) == sweeps
    sim.close()


def filled(lib, n, share, precision="fp64", bloch=None):
    """A Drude block over a share of a box without an absorber."""
    s = share ** (1.0 / 3.0)
    geom = [g.DefaultMedium(g.Dielectric()),
            g.Block(g.Drude(eps_inf=2.0, dps=(g.DrudePole(omega=0.5, gamma=0.05),)), center=(0, 0, 0),
                    size=[v * s for v in n])]
    sim = g.FDTD(g.Cartesian(size=n, resolution=1), geom, [], courant_ratio=0.4, verbose=False, precision=precision,
                 bloch=bloch, _engine=lib)
    sim.init()
    return sim


@pytest.mark.parametrize("kw", [FP64, C64], ids=["fp64", "c64"])
def test_media_over_much_of_the_grid(engine_lib, kw):
    for n, share, sweeps in (((80, 80, 80), 1.2, False), ((80, 80, 80), 0.7, True), ((72, 72, 72), 1.2, True)):
        sim = filled(engine_lib, n, share, **kw)
        assert swept(engine_lib, sim) == sweeps
        sim.close()
