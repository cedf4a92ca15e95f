"""One-sweep steps when device memory runs out: whatever the two-kernel step
has room for is still accepted, with the same results.

Each case runs in a process of its own, where memory_shim.c counts and limits
the engine's device allocations.
"""

import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
for path in (ROOT, HERE):
    if path not in sys.path:
        sys.path.insert(0, path)

CASES = {}


def case(f):
    CASES[f.__name__] = f
    return f


@pytest.mark.gpu
@pytest.mark.parametrize("name", ["source_lists", "commit", "many_sims", "half_full", "set_up_at_once"])
def test_limited_memory(engine_lib, tmp_path, name):
    shim = str(tmp_path / "memory_shim.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", shim, os.path.join(HERE, "memory_shim.c"), "-lpthread"],
                   check=True)
    out = subprocess.run([sys.executable, os.path.abspath(__file__), shim, name], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, timeout=100)
    assert out.returncode == 0, out.stdout.decode()


def builders():
    import gmes_amd as g
    from test_step1d import line
    from test_step2d import plane
    from test_step3d import box, media_box
    return [lambda lib: box(lib, (22, 21, 24), bound=g.Cpml), lambda lib: media_box(lib, (22, 21, 24)),
            lambda lib: box(lib, (22, 21, 24), precision="fp64", bound=g.Upml),
            lambda lib: plane(lib, "tez", (41, 67), bound=g.Cpml, media=True),
            lambda lib: line(lib, "z", 300, bound=g.Cpml, media=True)]


def fields(sim):
    return [np.array(sim.field[c]) for c in sim._active]


def agree(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


@case
def commit(lib, shim):
    """Memory taken by others between the look at it and the allocation."""
    for build in builders():
        start = shim.shim_used()
        shim.shim_peak(1)
        sim = build(lib)
        sim._advance(5)
        want = fields(sim)
        sim.close()
        most = shim.shim_peak(1) - start
        # on a device this small nothing is held twice: the two-kernel step
        shim.shim_limit(start + int(1.1 * most), 1)
        sim = build(lib)
        sim._advance(5)
        agree(fields(sim), want)
        sim.close()
        least = shim.shim_peak(1) - start
        assert least < most
        for q in range(13):
            shim.shim_limit(start + least + (most - least) * q // 12 - (q == 12), 0)
            sim = build(lib)
            sim._advance(5)
            agree(fields(sim), want)
            sim.close()
        shim.shim_limit(0, 0)


@case
def many_sims(lib, shim):
    """A device that holds every sim once, but not twice: sims made later find
    the room that the second buffers of earlier ones hold, while those are
    being stepped."""
    import threading

    import gmes_amd as g
    from gmes_amd.batch import Batch
    from test_step3d import box, media_box

    def made():
        return box(lib, (40, 41, 42), bound=g.Cpml), media_box(lib, (44, 41, 42))

    start = shim.shim_used()
    pair = made()
    twice = shim.shim_used() - start
    for s in pair:
        lib.set_graph(s._sim, 1)
        s._advance(5)
    want = [fields(s) for s in pair]
    for s in pair:
        s.close()
    shim.shim_limit(start + int(1.2 * twice), 1)
    pair = made()
    once = shim.shim_used() - start
    for s in pair:
        s.close()
    assert once < 0.8 * twice
    shim.shim_limit(start + int(7.3 * once) + (4 << 20), 1)
    batch = Batch([s for _ in range(2) for s in made()])
    done = 3
    batch.advance(done)
    swept = [lib.footprint(s._sim) for s in batch.sims]
    errors, sims = [], []

    def work():
        try:
            mine = made()
            for s in mine:
                lib.set_graph(s._sim, 1)
                s._advance(4)
            sims.extend(mine)
        except Exception as e:
            errors.append(e)

    threads = [threading.Thread(target=work) for _ in range(5)]
    for t in threads:
        t.start()
    while any(t.is_alive() for t in threads):
        k = 1 + done % 6
        batch.advance(k)
        done += k
    for t in threads:
        t.join()
    assert not errors, errors
    assert [lib.footprint(s._sim) for s in batch.sims] < swept
    for s in sims:
        s._advance(1)
    for q, s in enumerate(sims):
        agree(fields(s), want[q % 2])
    for s in sims:
        s.close()
    shim.shim_limit(0, 0)
    alone = made()
    for s in alone:
        s._advance(done)
    for q, s in enumerate(batch.sims):
        agree(fields(s), fields(alone[q % 2]))
    batch.close()


@case
def source_lists(lib, shim):
    """No room for the lists of cells finished after the sweep, nor for the
    scratch memory they are made in."""
    from test_step3d import media_box
    for kw in (dict(wave=False), dict(media=False)):  # dispersive cells; a total-field box
        a, b = (media_box(lib, (22, 21, 24), **kw) for _ in range(2))
        lib.set_ghost_fusion(b._sim, 0)
        full, used = lib.footprint(a._sim), shim.shim_used()
        for room in (1024, 20000, 40000, 60000, None):
            shim.shim_limit(shim.shim_used() + room if room else 0, 0)
            a.init_source()
            if room == 1024:
                # neither fits: what the lists held is free, and leaves the
                # footprint (which counts the few bytes of no sources twice)
                assert shim.shim_used() < used - 4096
                if "media" not in kw:
                    assert 0 <= used - shim.shim_used() - (full - lib.footprint(a._sim)) < 1024
            shim.shim_limit(0, 0)
            for s in (a, b):
                s._advance(4)
            agree(fields(a), fields(b))


def swept(lib, sim):
    """Whether a step of sim is a one-sweep step (it launches no H kernel)."""
    lib.profile(sim._sim, 1)
    sim._advance(2)
    lib.sync(sim._sim)
    launches = lib.read_profile(sim._sim)[1]
    lib.profile(sim._sim, 0)
    return launches[1] == 0


@case
def half_full(lib, shim):
    """Small sims take one-sweep steps however full the device is; large ones
    do not when they would fill more than half of it."""
    import gmes_amd as g
    from test_step1d import line
    from test_step2d import plane
    from test_step3d import box
    shim.shim_limit(shim.shim_used() + (16 << 20), 1)
    large = [box(lib, (40, 41, 42), bound=g.Cpml) for _ in range(2)]
    assert not swept(lib, large[1])
    shim.shim_limit(shim.shim_used() + (10 << 20), 1)
    small = [line(lib, "z", 300, bound=g.Cpml, media=True), plane(lib, "tmz", (20, 24))]
    assert all(swept(lib, s) for s in small)


@case
def set_up_at_once(lib, shim):
    """Sims committed by several threads together do not take the same room."""
    import threading

    import gmes_amd as g
    from test_step3d import box
    start = shim.shim_used()
    sim = box(lib, (40, 41, 42), bound=g.Cpml)
    twice = shim.shim_used() - start
    shim.shim_limit(shim.shim_used() + 1, 1)
    lib.commit(sim._sim)
    once = shim.shim_used() - start
    shim.shim_limit(shim.shim_used() + 4 * once, 1)
    sims = [sim] + [box(lib, (40, 41, 42), bound=g.Cpml) for _ in range(3)]
    assert not any(swept(lib, s) for s in sims)
    shim.shim_limit(start + 2 * (4 * once + 5 * (twice - once) // 4), 1)
    shim.shim_wait(50000)
    threads = [threading.Thread(target=lib.commit, args=(s._sim,)) for s in sims]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    shim.shim_wait(0)
    assert sum(swept(lib, s) for s in sims) == 1


def main(path, name):
    from gmes_amd import _abi
    shim = ctypes.CDLL(path, ctypes.RTLD_GLOBAL)
    for f in (shim.shim_used, shim.shim_peak):
        f.restype = ctypes.c_size_t
    shim.shim_limit.argtypes = [ctypes.c_size_t, ctypes.c_int]
    hip = ctypes.CDLL("libamdhip64.so.7")
    shim.shim_init(*(ctypes.cast(getattr(hip, f), ctypes.c_void_p) for f in ("hipMalloc", "hipFree", "hipMemGetInfo")))
    lib = _abi.engine()
    CASES[name](lib, shim)
    assert shim.shim_peak(0) > 0, "the engine's allocations do not pass through the shim"
    print("ok", flush=True)


if __name__ == "__main__":
    main(sys.argv[1], sys.argv[2])
