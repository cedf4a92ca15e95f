"""One-sweep 2-D steps (step2d.hip) against the two-kernel step.

As in test_step3d.py the two-kernel step with separate ghost copies is the
reference, and every value must agree.  The sizes sit at the edges of the
kernel's tiling: a wave of columns and one more, the widest row of one
block, the narrowest row of several, a last stretch of one column, a single
row per block.
"""

import numpy as np
import pytest

import gmes_amd as g

pytestmark = pytest.mark.gpu

MODES = {"tmz": (g.TMzFDTD, (g.Ez, g.Hx, g.Hy)), "tez": (g.TEzFDTD, (g.Ex, g.Ey, g.Hz))}
SIZES = [(9, 9), (31, 33), (6, 64), (12, 65), (40, 190), (9, 512), (11, 513), (300, 449), (7, 673)]


def plane(lib, mode, n, precision="fp32", bound=None, bloch=None, media=False, sources=1, res=1):
    cls, comps = MODES[mode]
    s = 1.0 / res
    geom = [g.DefaultMedium(g.Dielectric()),
            g.Cylinder(g.Dielectric(3.0), center=(0.3 * s, 0.2 * s, 0), radius=min(n) * s / 4, axis=(0, 0, 1), height=4),
            g.Block(g.Const(0.25), center=(-s, s, 0), size=(1.1 * s, 1.1 * s, 4 * s))]
    if media:
        pole, crit = g.DrudePole(omega=0.5 * res, gamma=0.05 * res), g.CriticalPoint(amp=0.6, phi=-0.4, omega=0.4 * res,
                                                                                       gamma=0.05 * res)
        kinds = [g.Drude(eps_inf=2.0, dps=(pole,)),
                 g.Lorentz(eps_inf=2.0, lps=(g.LorentzPole(amp=1.2, omega=0.4 * res, gamma=0.02 * res),)),
                 g.DcpAde(eps_inf=2.0, sigma=0.01, dps=(pole,), cps=(crit,)),
                 g.DcpPlrc(eps_inf=2.0, sigma=0.01, dps=(pole,), cps=(crit, crit))]
        for q, kind in enumerate(kinds):  # the first ones reach over the periodic edges
            geom.append(g.Block(kind, center=((-n[0] / 2 + q * n[0] / 4) * s, (-n[1] / 2 + q * n[1] / 4) * s, 0),
                                size=(n[0] * s / 5, n[1] * s / 5, 4 * s)))
    if bound is not None:
        geom.append(g.Shell(bound(), thickness=3 * s))
    src = [g.PointSource(g.Continuous(freq=0.05 * res, width=5 * s), center=((q - 1) * s, 0, 0),
                         component=comps[q % 3]) for q in range(sources)]
    sim = cls(g.Cartesian(size=(n[0] * s, n[1] * s, 0), resolution=res), geom, src, courant_ratio=0.5, verbose=False,
              precision=precision, bloch=bloch, _engine=lib)
    sim.init()
    rng = np.random.default_rng(5)
    for c in comps:
        a = sim.field[c]
        a[...] = rng.standard_normal(a.shape)
        if bloch is not None:
            a[...] += 1j * rng.standard_normal(a.shape)
    return sim


def agree(a, b, mode):
    for c in MODES[mode][1]:
        x, y = np.array(a.field[c]), np.array(b.field[c])
        assert np.abs(x).max() > 0
        np.testing.assert_array_equal(x, y)


def run_pair(lib, mode, steps=(1, 4, 7), graph=False, **kw):
    a, b = plane(lib, mode, **kw), plane(lib, mode, **kw)
    lib.set_ghost_fusion(b._sim, 0)
    if graph:
        lib.set_graph(a._sim, 1)
    for k in steps:
        a._advance(k)
        b._advance(k)
        agree(a, b, mode)
    return a, b


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("bound", [None, g.Cpml, g.Upml], ids=["none", "cpml", "upml"])
def test_real(engine_lib, mode, n, precision, bound):
    run_pair(engine_lib, mode, n=n, precision=precision, bound=bound)


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("n", [(9, 9), (12, 65), (9, 512), (11, 513)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("bound", [None, g.Cpml, g.Upml], ids=["none", "cpml", "upml"])
def test_bloch(engine_lib, mode, n, precision, bound):
    run_pair(engine_lib, mode, n=n, precision=precision, bound=bound, bloch=(0.3, -0.2, 0.0))


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("n", [(31, 33), (40, 190), (24, 513)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("kw", [dict(), dict(precision="fp64"), dict(bloch=(0.3, -0.2, 0.0)),
                                dict(precision="fp64", bound=g.Cpml), dict(bound=g.Upml)],
                         ids=["fp32", "fp64", "c64", "fp64_cpml", "fp32_upml"])
def test_dispersive(engine_lib, mode, n, kw):
    a, b = run_pair(engine_lib, mode, n=n, media=True, **kw)
    # on to the two-kernel step and back
    for on in (0, 1):
        engine_lib.set_ghost_fusion(a._sim, on)
        a._advance(3)
        b._advance(3)
        agree(a, b, mode)


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("res", [1, 3], ids=["exact_division", "division"])
def test_fp64_matches_the_oracle(engine_lib, oracle_lib, mode, res):
    a, b = (plane(lib, mode, (20, 23), precision="fp64", res=res, media=True) for lib in (engine_lib, oracle_lib))
    a._advance(12)
    b._advance(12)
    for c in MODES[mode][1]:
        x, y = np.array(a.field[c]), np.array(b.field[c])
        assert np.linalg.norm(x - y) <= 1e-12 * np.linalg.norm(y)


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("sources", [0, 3, 6])
def test_sources_and_graph(engine_lib, mode, sources):
    run_pair(engine_lib, mode, steps=(5, 2, 1, 8, 3), graph=True, n=(15, 22), bound=g.Cpml, sources=sources)


@pytest.mark.parametrize("mode", sorted(MODES))
def test_monitors_see_each_step(engine_lib, mode):
    from gmes_amd.monitor import DftBox
    e, h = (g.Ez, g.Hx) if mode == "tmz" else (g.Ex, g.Hz)
    out = []
    for fuse in (1, 0):
        sim = plane(engine_lib, mode, (10, 12), bound=g.Cpml, media=True)
        engine_lib.set_ghost_fusion(sim._sim, fuse)
        pids = [engine_lib.add_probe(sim._sim, h.index, 0), engine_lib.add_probe(sim._sim, e.index, 30)]
        sh = sim._shape[h]
        mon = DftBox(sim, h, (0, 0, 0), sh, [0.05, 0.1], 1)
        sim._advance(9)
        engine_lib.sync(sim._sim)
        out.append(([engine_lib.read_probe(sim._sim, p) for p in pids], mon.values()))
        sim.close()
    for x, y in zip(out[0][0], out[1][0]):
        assert len(x) == 9
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(out[0][1], out[1][1])


@pytest.mark.parametrize("bound", [g.Cpml, g.Upml], ids=["cpml", "upml"])
def test_snapshot_between_the_steps(engine_lib, bound):
    """A snapshot taken on either buffer set restores the run, and keeps the
    blob's order whatever the device layout: k fastest, 32 words around."""
    a = plane(engine_lib, "tez", (40, 50), bound=bound, media=True)
    for k in (3, 4):
        a._advance(k)
        snap = a.snapshot()
        a._advance(5)
        want = {c: np.array(a.field[c]) for c in MODES["tez"][1]}
        a.restore(snap)
        a._advance(5)
        for c, v in want.items():
            np.testing.assert_array_equal(a.field[c], v)
