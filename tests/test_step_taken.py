"""Which step a sim takes: the tests that compare a sim with a two-kernel one
mean nothing when both take the two-kernel step."""

import numpy as np
import pytest

import gmes_amd as g
from gmes_amd.batch import Batch

import test_step1d as t1
import test_step2d as t2
import test_step3d as t3
from test_batch_sweep import members
from test_memory import swept
from test_step1d import line
from test_step2d import plane
from test_step3d import box, media_box

pytestmark = pytest.mark.gpu


def takes(lib, sim, sweeps):
    assert swept(lib, sim) == sweeps
    sim.close()


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


BOUNDS = [None, g.Cpml, g.Upml]
KINDS3 = {"fp32": dict(), "fp64": FP64, "c64": C64}


@pytest.mark.parametrize("kind", sorted(KINDS3))
def test_boxes(engine_lib, kind):
    """The boxes of test_step3d.py."""
    kw = KINDS3[kind]
    for n in t3.SIZES + ([] if kind == "fp32" else [(10, 11, 256), (9, 9, 257)]):
        for bound in BOUNDS if min(n) >= 8 else [None]:
            takes(engine_lib, box(engine_lib, n, bound=bound, **kw), bound is None or kind == "fp32" or n[2] <= 256)
    for axes in t3.AXES:
        takes(engine_lib, box(engine_lib, (13, 12, 15), bound=g.Cpml, axes=axes, **kw), True)
    for n in ((110, 113, 107), (80, 91, 93)):
        takes(engine_lib, box(engine_lib, n, bound=g.Cpml, axes="xz", **kw), True)
    for comps in ((), (g.Jz, g.Hy), (g.Ex, g.My, g.Ez, g.Hx)):
        takes(engine_lib, box(engine_lib, (12, 11, 14), bound=g.Cpml, comps=comps, **kw), True)
    takes(engine_lib, box(engine_lib, (14, 12, 13), bound=g.Cpml, over_shell=True, **kw), False)


MEDIA = {"media": (dict(wave=False), True), "wave": (dict(media=False), True), "both": (dict(), False),
         "both_apart": (dict(seam=False, n=(22, 21, 42)), True),
         "media_cpml": (dict(wave=False, seam=False, bound=g.Cpml), True),
         "media_upml": (dict(wave=False, seam=False, bound=g.Upml), True),
         "media_points": (dict(wave=False, point=(g.Ez, g.Hx, g.Ey)), False),
         "wave_cpml": (dict(media=False, bound=g.Cpml), False)}


@pytest.mark.parametrize("kind", sorted(KINDS3))
@pytest.mark.parametrize("what", sorted(MEDIA))
def test_media_boxes(engine_lib, kind, what):
    """Those of test_cells_finished_after_the_sweep.  With both, a face of the
    total-field box crosses a dispersive object, the points are inside one, and
    in the last case the H cells next to the faces have absorber state: two-kernel
    steps."""
    kw, sweeps = MEDIA[what]
    kw = dict(dict(n=(22, 21, 24)), **kw)
    takes(engine_lib, media_box(engine_lib, **dict(kw, **KINDS3[kind])), sweeps)


def test_planes_and_lines(engine_lib):
    for mode in sorted(t2.MODES):
        for kw in (dict(), FP64, C64, dict(C64, **FP64)):
            for n in t2.SIZES:
                for bound in BOUNDS:
                    takes(engine_lib, plane(engine_lib, mode, n, bound=bound, **kw), True)
            takes(engine_lib, plane(engine_lib, mode, (31, 33), media=True, sources=6, **kw), True)
    for axis in sorted(t1.MODES):
        for kw in (dict(), FP64, C64, dict(C64, **FP64)):
            for bound in BOUNDS:
                takes(engine_lib, line(engine_lib, axis, 256, bound=bound, media=True, sources=3, **kw), True)


@pytest.mark.parametrize("precision,bloch", [("fp32", None), ("fp64", None), ("fp32", (0.3, -0.2, 0.0))],
                         ids=["fp32", "fp64", "c64"])
def test_batch_members(engine_lib, precision, bloch):
    """Those of test_batch_sweep.py: alone, and the ones that sweep in a batch."""
    sims = members(engine_lib, precision, bloch)
    # an object over the absorber; rows too long for 8-byte words; a face through a dispersive object
    two = [9, 11] if (precision, bloch) == ("fp32", None) else [9, 10, 11]
    if (precision, bloch) == ("fp32", None):
        assert swept(engine_lib, sims[10])
    assert [q for q, s in enumerate(sims) if not swept(engine_lib, s)] == two
    # (its rows do not fit the batch's blocks)
    batch = Batch([s for q, s in enumerate(sims) if q not in two + [10]])
    batch.profile(True)
    batch.advance(3)
    launches = batch.read_profile()[1]
    assert launches[0] and launches[2] and not launches[1] and not launches[3]
    batch.close()


def bits(n):
    b = 1
    while (1 << b) < n + 16:  # and 16 cells with sources
        b += 1
    return b


@pytest.mark.parametrize("media,wide", [(9, True), (7, True), (3, False)])
def test_width_of_entry_ids(engine_lib, media, wide):
    """The boxes of test_many_media: distinct triples of E and of H records of
    a thread's cells that do not, or do, fit 16 bits together."""
    rng = np.random.default_rng(8)
    n = (14, 13, 15)
    kinds = [g.Dielectric(1.0 + 0.3 * q, 1.0 + 0.1 * q) for q in range(media)]
    geom = [g.DefaultMedium(g.Dielectric())]
    for _ in range(900):
        c = [rng.uniform(-v / 2, v / 2) for v in n]
        geom.append(g.Block(kinds[rng.integers(media)], center=c, size=rng.uniform(0.8, 2.6, 3)))
    sim = g.FDTD(g.Cartesian(size=n, resolution=1), geom, [], courant_ratio=0.4, verbose=False, precision="fp32",
                 _engine=engine_lib)
    sim.init()
    ids = {c: np.asarray(sim._tiles.ids[c]).reshape(sim._shape[c]) for c in g.constant.COMPONENTS}
    count = []
    for first in (0, 3):
        cells = []
        for t in range(3):
            up = [first == 3 and a != t for a in range(3)]  # H cells sit one up across their own axis
            x = ids[g.constant.COMPONENTS[first + t]]
            cells.append(x[tuple(slice(u, u + m) for u, m in zip(up, n))].ravel())
        count.append(len(np.unique(np.stack(cells), axis=1).T))
    assert (sum(bits(v) for v in count) > 16) == wide
    takes(engine_lib, sim, True)


@pytest.mark.parametrize("kind", sorted(KINDS3))
@pytest.mark.parametrize("graph", [False, True], ids=["direct", "graph"])
@pytest.mark.parametrize("wave", [False, True], ids=["points", "wave"])
def test_media_and_sources(engine_lib, kind, graph, wave):
    """Dispersive cells and sources that keep clear of them, point sources or
    the faces of a total-field box, all finished after the sweep."""
    a, b = (media_box(engine_lib, (22, 21, 42), seam=False, wave=wave, **KINDS3[kind]) for _ in range(2))
    if not wave:
        for s in (a, b):
            s.src_list = [g.PointSource(g.Continuous(freq=0.05, width=5), center=(10, q - 9, 17), component=c)
                          for q, c in enumerate((g.Ez, g.Hx, g.Ey))]
            s.init_source()
    engine_lib.set_ghost_fusion(b._sim, 0)
    assert swept(engine_lib, a) and not swept(engine_lib, b)
    if graph:
        engine_lib.set_graph(a._sim, 1)
    for k in (1, 4, 7):
        a._advance(k)
        b._advance(k)
        t3.agree(a, b)
    snap = a.snapshot()
    a._advance(3)
    want = {c: np.array(a.field[c]) for c in g.constant.COMPONENTS}
    a.restore(snap)
    a._advance(3)
    for c, v in want.items():
        np.testing.assert_array_equal(a.field[c], v)


@pytest.mark.parametrize("kind", sorted(KINDS3))
@pytest.mark.parametrize("n", [(1, 8, 8), (2, 2, 2), (8, 9, 1), (1, 2, 1), (3, 1200, 1), (1, 40, 70), (2, 3, 341), (70, 2, 1)],
                         ids=lambda n: "x".join(map(str, n)))
def test_thin_boxes(engine_lib, kind, n):
    """Boxes of one or two cells along an axis."""
    a, b = (box(engine_lib, n, **KINDS3[kind]) for _ in range(2))
    engine_lib.set_ghost_fusion(b._sim, 0)
    assert swept(engine_lib, a) and not swept(engine_lib, b)
    for k in (1, 4):
        a._advance(k)
        b._advance(k)
        t3.agree(a, b)
