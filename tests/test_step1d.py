"""One-sweep 1-D steps (step1d.hip) against the two-kernel step, which the
oracle tests pin: every value must agree.  Lengths at the edges of a block
(255 cells and a rim)."""

import numpy as np
import pytest

import gmes_amd as g

pytestmark = pytest.mark.gpu

MODES = {"x": (g.TEMxFDTD, g.Ey, g.Hz), "y": (g.TEMyFDTD, g.Ez, g.Hx), "z": (g.TEMzFDTD, g.Ex, g.Hy)}


def line(lib, axis, n, precision="fp32", bound=None, bloch=None, media=False, sources=1):
    cls, e, h = MODES[axis]
    size = [n if a == axis else 0 for a in "xyz"]

    def at(v):
        return [v if a == axis else 0 for a in "xyz"]

    def ext(v):
        return [v if a == axis else 4 for a in "xyz"]

    geom = [g.DefaultMedium(g.Dielectric()), g.Block(g.Dielectric(3.0), center=at(n / 8), size=ext(n / 9)),
            g.Block(g.Const(0.25), center=at(-2), size=ext(1.1))]
    if media:
        pole, crit = g.DrudePole(omega=0.5, gamma=0.05), g.CriticalPoint(amp=0.6, phi=-0.4, omega=0.4, gamma=0.05)
        for q, kind in enumerate([g.Drude(eps_inf=2.0, dps=(pole,)),
                                  g.DcpAde(eps_inf=2.0, sigma=0.01, dps=(pole,), cps=(crit,)),
                                  g.DcpPlrc(eps_inf=2.0, sigma=0.01, dps=(pole,), cps=(crit, crit))]):
            geom.append(g.Block(kind, center=at((-0.5 + 0.3 * q) * n), size=ext(n / 6)))
    if bound is not None:
        geom.append(g.Shell(bound(), thickness=3))
    src = [g.PointSource(g.Continuous(freq=0.05, width=5), center=at(q - 1), component=(e, h)[q % 2])
           for q in range(sources)]
    sim = cls(g.Cartesian(size=size, resolution=1), geom, src, courant_ratio=0.5, verbose=False, precision=precision,
              bloch=bloch, _engine=lib)
    sim.init()
    rng = np.random.default_rng(5)
    for c in (e, h):
        a = sim.field[c]
        a[...] = rng.standard_normal(a.shape)
        if bloch is not None:
            a[...] += 1j * rng.standard_normal(a.shape)
    return sim


def run_pair(lib, axis, steps=(1, 4, 7), graph=False, **kw):
    a, b = line(lib, axis, **kw), line(lib, axis, **kw)
    lib.set_ghost_fusion(b._sim, 0)
    if graph:
        lib.set_graph(a._sim, 1)
    for k in steps:
        a._advance(k)
        b._advance(k)
        for c in MODES[axis][1:]:
            x, y = np.array(a.field[c]), np.array(b.field[c])
            assert np.abs(x).max() > 0
            np.testing.assert_array_equal(x, y)
    return a, b


@pytest.mark.parametrize("axis", sorted(MODES))
@pytest.mark.parametrize("n", [9, 254, 255, 256, 511, 801])
@pytest.mark.parametrize("kw", [dict(), dict(precision="fp64"), dict(bloch=(0.3, -0.2, 0.1)),
                                dict(precision="fp64", bloch=(0.3, -0.2, 0.1))], ids=["fp32", "fp64", "c64", "c128"])
@pytest.mark.parametrize("bound", [None, g.Cpml, g.Upml], ids=["none", "cpml", "upml"])
def test_lengths(engine_lib, axis, n, kw, bound):
    run_pair(engine_lib, axis, n=n, bound=bound, **kw)


@pytest.mark.parametrize("axis", sorted(MODES))
@pytest.mark.parametrize("kw", [dict(), dict(precision="fp64", bound=g.Cpml), dict(bloch=(0.3, -0.2, 0.1))],
                         ids=["fp32", "fp64_cpml", "c64"])
@pytest.mark.parametrize("sources", [0, 3])
def test_media_sources_and_graph(engine_lib, axis, kw, sources):
    a, b = run_pair(engine_lib, axis, steps=(5, 2, 1, 8), graph=True, n=40, media=True, sources=sources, **kw)
    snap = a.snapshot()
    a._advance(3)
    want = {c: np.array(a.field[c]) for c in MODES[axis][1:]}
    a.restore(snap)
    engine_lib.set_ghost_fusion(a._sim, 0)
    a._advance(3)
    for c, v in want.items():
        np.testing.assert_array_equal(a.field[c], v)
