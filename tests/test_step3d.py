"""One-sweep 3-D steps (step3d.hip) against the two-kernel step.

A sim with ghost fusion turned off takes the two-kernel step with separate
ghost copies, which the oracle tests pin; the one-sweep step keeps every
formula and operand order, so all six fields, ghost planes included, must
agree in every value.  The sizes sit at the edges of the kernel's tiling:
rows of one block and of none to spare, one row more than a tile, a single
plane or row of cells per block, rows longer than a wave by one.
"""

import numpy as np
import pytest

import gmes_amd as g

pytestmark = pytest.mark.gpu

FP64_TOL = 1e-12


def box(lib, n, precision="fp32", bound=None, bloch=None, comps=(g.Ex,), over_shell=False, res=1, axes="xyz"):
    """A box of n cells with two dielectric objects, an absorber of 3 cells,
    waves everywhere and a source on each of comps."""
    space = g.Cartesian(size=tuple(v / res for v in n), resolution=res)
    s = 1.0 / res
    geom = [g.DefaultMedium(g.Dielectric()),
            g.Sphere(g.Dielectric(3.0), center=(0.3 * s, 0.2 * s, -0.4 * s), radius=min(n) * s / 4),
            g.Block(g.Dielectric(5.0, 1.5), center=(s, -s, s), size=(2.2 * s, 3.1 * s, 4.3 * s)),
            g.Block(g.Const(0.25), center=(-s, s, 0), size=(1.1 * s, 1.1 * s, 1.1 * s))]
    if bound is not None:
        # layers on the named axes: elsewhere the shell lies outside the box
        size = [v * s if a in axes else (v + 8) * s for a, v in zip("xyz", n)]
        faces = {"%s_%s" % (side, a): a in axes for side in ("plus", "minus") for a in "xyz"}
        geom.append(g.Shell(bound(), size=size, thickness=3 * s, **faces))
    if over_shell:  # a medium on top of the absorber: its cells are not CPML
        geom.append(g.Block(g.Dielectric(2.0), center=(-n[0] * s / 2, 0, 0), size=(4 * s, 2 * s, 2 * s)))
    src = [g.PointSource(g.Continuous(freq=0.05 * res, width=5 * s), center=(q * s, 0, 0), component=c)
           for q, c in enumerate(comps)]
    sim = g.FDTD(space, geom, src, courant_ratio=0.5, verbose=False, precision=precision, bloch=bloch, _engine=lib)
    sim.init()
    rng = np.random.default_rng(5)
    for c in g.constant.COMPONENTS:
        a = sim.field[c]
        a[...] = rng.standard_normal(a.shape)
        if bloch is not None:
            a[...] += 1j * rng.standard_normal(a.shape)
    return sim


def agree(a, b):
    for c in g.constant.COMPONENTS:
        x, y = np.array(a.field[c]), np.array(b.field[c])
        assert np.abs(x).max() > 0
        np.testing.assert_array_equal(x, y)


def run_pair(lib, steps=(1, 4, 7), graph=False, **kw):
    a, b = box(lib, **kw), box(lib, **kw)
    lib.set_ghost_fusion(b._sim, 0)
    if graph:
        lib.set_graph(a._sim, 1)
    for k in steps:
        a._advance(k)
        b._advance(k)
        agree(a, b)
    return a, b


SIZES = [(9, 9, 9), (8, 2, 8), (7, 17, 64), (12, 9, 65), (5, 8, 341), (33, 8, 85), (8, 70, 16)]


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("bound", [None, g.Cpml, g.Upml], ids=["none", "cpml", "upml"])
def test_fp32(engine_lib, n, bound):
    run_pair(engine_lib, n=n, bound=bound if min(n) >= 8 else None)


@pytest.mark.parametrize("n", SIZES + [(10, 11, 256), (9, 9, 257)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("kw", [dict(precision="fp64"), dict(bloch=(0.3, -0.2, 0.1))], ids=["fp64", "c64"])
@pytest.mark.parametrize("bound", [None, g.Cpml, g.Upml], ids=["none", "cpml", "upml"])
def test_eight_byte_words(engine_lib, n, kw, bound):
    run_pair(engine_lib, n=n, bound=bound if min(n) >= 8 else None, **kw)


AXES = ["x", "y", "z", "xy", "xz", "yz"]


@pytest.mark.parametrize("axes", AXES)
@pytest.mark.parametrize("kw", [dict(), dict(precision="fp64", res=3), dict(bloch=(0.3, -0.2, 0.1))],
                         ids=["fp32", "fp64", "c64"])
def test_layers_on_some_axes(engine_lib, axes, kw):
    """No live absorber words along the other axes."""
    run_pair(engine_lib, n=(13, 12, 15), bound=g.Cpml, axes=axes, **kw)


# from 5 MB a component the launch has blocks of several kinds
@pytest.mark.parametrize("n,kw", [((110, 113, 107), dict()), ((80, 91, 93), dict(precision="fp64")),
                                  ((91, 80, 93), dict(bloch=(0.3, -0.2, 0.1)))], ids=["fp32", "fp64", "c64"])
@pytest.mark.parametrize("axes", ["xyz"] + AXES)
def test_blocks_of_several_kinds(engine_lib, n, kw, axes):
    run_pair(engine_lib, n=n, steps=(1, 4), bound=g.Cpml, axes=axes, **kw)


@pytest.mark.parametrize("res", [1, 3], ids=["exact_division", "division"])
def test_fp64_matches_the_oracle(engine_lib, oracle_lib, res):
    a, b = (box(lib, n=(10, 11, 13), precision="fp64", res=res) for lib in (engine_lib, oracle_lib))
    a._advance(12)
    b._advance(12)
    for c in g.constant.COMPONENTS:
        x, y = np.array(a.field[c]), np.array(b.field[c])
        assert np.linalg.norm(x - y) <= FP64_TOL * np.linalg.norm(y)


@pytest.mark.parametrize("comps", [(), (g.Jz, g.Hy), (g.Ex, g.My, g.Ez, g.Hx)], ids=["none", "two", "four"])
def test_sources(engine_lib, comps):
    run_pair(engine_lib, n=(12, 11, 14), bound=g.Cpml, comps=comps)


def test_graph_of_two_steps(engine_lib):
    """Odd and even counts, so that the graph starts on either buffer set,
    with host reads and writes between."""
    a, b = run_pair(engine_lib, steps=(5, 2, 1, 8, 3), graph=True, n=(12, 11, 14), bound=g.Cpml)
    a.ez[3, 3, 3] = b.ez[3, 3, 3] = 2.0
    a._advance(6)
    b._advance(6)
    agree(a, b)


def test_switching_between_the_steps(engine_lib):
    """A sim that goes back and forth between the two kinds of step."""
    a, b = run_pair(engine_lib, n=(12, 11, 14), bound=g.Upml, steps=(3,))
    for on in (0, 1, 0, 1):
        engine_lib.set_ghost_fusion(a._sim, on)
        a._advance(3)
        b._advance(3)
        agree(a, b)
    snap = a.snapshot()
    a._advance(5)
    want = {c: np.array(a.field[c]) for c in g.constant.COMPONENTS}
    a.restore(snap)
    a._advance(5)
    for c, v in want.items():
        np.testing.assert_array_equal(a.field[c], v)


def test_object_over_the_absorber(engine_lib):
    """Dielectric cells where the CPML has live state: the two-kernel step."""
    run_pair(engine_lib, n=(14, 12, 13), bound=g.Cpml, over_shell=True)


def test_monitors_see_each_step(engine_lib, tmp_path):
    """Probes on ghost planes and inside, and a DFT box over a ghost plane,
    read the values of every step."""
    from gmes_amd.monitor import DftBox
    out = []
    for fuse in (1, 0):
        sim = box(engine_lib, n=(10, 9, 12), bound=g.Cpml)
        engine_lib.set_ghost_fusion(sim._sim, fuse)
        sh = sim._shape[g.Hz]
        pids = [engine_lib.add_probe(sim._sim, g.Hz.index, 3 * sh[2] + 4),  # i = 0: a ghost cell of Hz
                engine_lib.add_probe(sim._sim, g.Ez.index, 555)]
        mon = DftBox(sim, g.Hx, (0, 0, 0), (10, 10, 13), [0.05, 0.1], 1)
        sim._advance(9)
        engine_lib.sync(sim._sim)
        out.append(([engine_lib.read_probe(sim._sim, p) for p in pids], mon.values()))
        sim.close()
    for x, y in zip(out[0][0], out[1][0]):
        assert len(x) == 9
        np.testing.assert_array_equal(x, y)
    np.testing.assert_array_equal(out[0][1], out[1][1])


def media_box(lib, n, precision="fp32", bloch=None, media=True, wave=True, bound=None, point=(), seam=True):
    """Dispersive objects (over the periodic edges with seam), a plane wave
    through a total-field box, point sources."""
    geom = [g.DefaultMedium(g.Dielectric())]
    if media:
        pole, crit = g.DrudePole(omega=0.5, gamma=0.05), g.CriticalPoint(amp=0.6, phi=-0.4, omega=0.4, gamma=0.05)
        kinds = [g.Drude(eps_inf=2.0, dps=(pole,)),
                 g.Lorentz(eps_inf=2.0, lps=(g.LorentzPole(amp=1.2, omega=0.4, gamma=0.02),)),
                 g.DcpAde(eps_inf=2.0, sigma=0.01, dps=(pole,), cps=(crit,)),
                 g.DcpPlrc(eps_inf=2.0, sigma=0.01, dps=(pole,), cps=(crit, crit))]
        for q, kind in enumerate(kinds):
            c = [(-0.5 if seam and q == 0 else 0.2 * q - 0.3) * v for v in n]
            geom.append(g.Block(kind, center=c, size=[v / 5 for v in n]))
        geom.append(g.Block(g.Const(0.25), center=(0.1 * n[0], 0, 0), size=(1.1, 1.1, 1.1)))
    if bound is not None:
        geom.append(g.Shell(bound(), thickness=2))
    wf = g.Continuous(freq=0.05, width=5)
    src = [g.PointSource(wf, center=(q, 1, 2), component=c) for q, c in enumerate(point)]
    if wave:
        src.append(g.TotalFieldScatteredField(wf, center=(0, 0, 0), size=(2 * n[0], 2 * n[1], n[2] - 7.3),
                                              direction=(0, 0, -1), polarization=(1, 0, 0)))
    sim = g.FDTD(g.Cartesian(size=n, resolution=1), geom, src, courant_ratio=0.5, verbose=False, precision=precision,
                 bloch=bloch, _engine=lib)
    sim.init()
    rng = np.random.default_rng(5)
    for c in g.constant.COMPONENTS:
        a = sim.field[c]
        a[...] = rng.standard_normal(a.shape)
        if bloch is not None:
            a[...] += 1j * rng.standard_normal(a.shape)
    return sim


@pytest.mark.parametrize("kw", [dict(), dict(precision="fp64"), dict(bloch=(0.3, -0.2, 0.0))], ids=["fp32", "fp64", "c64"])
@pytest.mark.parametrize("what", [dict(wave=False), dict(media=False), dict(), dict(wave=False, seam=False, bound=g.Cpml),
                                  dict(wave=False, seam=False, bound=g.Upml), dict(wave=False, point=(g.Ez, g.Hx, g.Ey)),
                                  dict(media=False, bound=g.Cpml)],
                         ids=["media", "wave", "both", "media_cpml", "media_upml", "media_points", "wave_cpml"])
@pytest.mark.parametrize("graph", [False, True], ids=["direct", "graph"])
def test_cells_finished_after_the_sweep(engine_lib, kw, what, graph):
    """Dispersive cells and sources on many cells, and the H cells next to
    them, the periodic images included; in the last case some of those have
    absorber state (the two-kernel step)."""
    n = (22, 21, 24)
    a, b = media_box(engine_lib, n, **kw, **what), media_box(engine_lib, n, **kw, **what)
    engine_lib.set_ghost_fusion(b._sim, 0)
    if graph:
        engine_lib.set_graph(a._sim, 1)
    for k in (1, 4, 7):
        a._advance(k)
        b._advance(k)
        agree(a, b)
    snap = a.snapshot()
    a._advance(3)
    want = {c: np.array(a.field[c]) for c in g.constant.COMPONENTS}
    a.restore(snap)
    a._advance(3)
    for c, v in want.items():
        np.testing.assert_array_equal(a.field[c], v)


def test_finished_cells_match_the_oracle(engine_lib, oracle_lib):
    a, b = (media_box(lib, (16, 15, 20), precision="fp64") for lib in (engine_lib, oracle_lib))
    a._advance(12)
    b._advance(12)
    for c in g.constant.COMPONENTS:
        x, y = np.array(a.field[c]), np.array(b.field[c])
        assert np.linalg.norm(x - y) <= FP64_TOL * np.linalg.norm(y)


@pytest.mark.parametrize("precision,media", [("fp32", 9), ("fp64", 7), ("fp32", 3)])
def test_many_media(engine_lib, precision, media):
    """Entry ids of 32 bits: more distinct triples of E and of H cells than 16
    hold together (and, with 3 media, fewer)."""
    rng = np.random.default_rng(8)
    n = (14, 13, 15)
    kinds = [g.Dielectric(1.0 + 0.3 * q, 1.0 + 0.1 * q) for q in range(media)]
    geom = [g.DefaultMedium(g.Dielectric())]
    for _ in range(900):
        c = [rng.uniform(-v / 2, v / 2) for v in n]
        geom.append(g.Block(kinds[rng.integers(media)], center=c, size=rng.uniform(0.8, 2.6, 3)))
    src = [g.PointSource(g.Continuous(freq=0.05, width=5), center=(0, 0, 0), component=c) for c in (g.Ex, g.Hy)]
    sims = []
    for fuse in (1, 0):
        sim = g.FDTD(g.Cartesian(size=n, resolution=1), geom, src, courant_ratio=0.4, verbose=False,
                     precision=precision, _engine=engine_lib)
        sim.init()
        r = np.random.default_rng(5)
        for c in g.constant.COMPONENTS:
            sim.field[c][...] = r.standard_normal(sim.field[c].shape)
        engine_lib.set_ghost_fusion(sim._sim, fuse)
        sims.append(sim)
    for k in (1, 6):
        for sim in sims:
            sim._advance(k)
        agree(*sims)
