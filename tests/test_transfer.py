"""Field reads and writes around the size from which they go through pinned
buffers in pieces, with lengths that leave remainders in the last part and
piece, from several threads at once."""

import threading

import numpy as np
import pytest

import gmes_amd as g

pytestmark = pytest.mark.gpu


def sim_of(lib, n, precision):
    sim = g.FDTD(g.Cartesian(size=n, resolution=1), [g.DefaultMedium(g.Dielectric())], [], courant_ratio=0.5,
                 verbose=False, precision=precision, _engine=lib)
    sim.init()
    return sim


def round_trip(lib, sim, seed):
    rng = np.random.default_rng(seed)
    for c in (g.Ex, g.Hz):
        shape, dtype = sim.field[c].shape, sim.field[c].dtype
        want = rng.standard_normal(shape).astype(dtype)
        lib.write_field(sim._sim, c.index, want)
        got = np.empty(shape, dtype)
        lib.read_field(sim._sim, c.index, got)
        np.testing.assert_array_equal(got, want)


@pytest.mark.parametrize("n,precision", [((32, 255, 255), "fp32"), ((32, 256, 256), "fp32"), ((33, 257, 259), "fp32"),
                                         ((100, 101, 103), "fp64"), ((160, 160, 161), "fp64"), ((9, 1000, 300), "fp32")])
def test_round_trip(engine_lib, n, precision):
    sim = sim_of(engine_lib, n, precision)
    round_trip(engine_lib, sim, 1)
    sim.close()


def test_more_threads_than_buffers(engine_lib):
    sims = [sim_of(engine_lib, (48, 220, 210), "fp32") for _ in range(7)]
    errors = []

    def work(q):
        try:
            for r in range(3):
                round_trip(engine_lib, sims[q], 10 * q + r)
        except Exception as e:  # reported by the main thread
            errors.append(e)

    threads = [threading.Thread(target=work, args=(q,)) for q in range(len(sims))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for s in sims:
        s.close()
    assert not errors
