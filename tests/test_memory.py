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
@pytest.mark.parametrize("name", ["source_lists"])
def test_limited_memory(engine_lib, tmp_path, name):
    shim = str(tmp_path / "memory_shim.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", shim, os.path.join(HERE, "memory_shim.c"), "-lpthread"],
                   check=True)
    out = subprocess.run([sys.executable, os.path.abspath(__file__), shim, name], stdout=subprocess.PIPE,
                         stderr=subprocess.STDOUT, timeout=100)
    assert out.returncode == 0, out.stdout.decode()


def fields(sim):
    return [np.array(sim.field[c]) for c in sim._active]


def agree(a, b):
    for x, y in zip(a, b):
        np.testing.assert_array_equal(x, y)


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
