"""The device bytes a served slab is admitted by cover what it holds, the
second buffers of its one-sweep steps included."""

import pytest

from gmes_amd import workloads

from test_memory import swept


@pytest.mark.gpu
@pytest.mark.parametrize("side", [64, 112, 150])
def test_slab_estimate_covers_the_sim(engine_lib, side):
    sim, flux = workloads.pc_slab(side, 0.3)
    sim._advance(3)
    assert swept(engine_lib, sim)
    flux.flux()
    held = engine_lib.footprint(sim._sim) + sum(engine_lib.footprint(a._sim) for a in sim._aux_fdtds)
    assert held <= workloads.pc_slab_footprint(side)
    sim.close()
