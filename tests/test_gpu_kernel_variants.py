"""The occupancy choices of mfg_set_kernel_variant beyond the built kernels
run the nearest one with that kernel's launch. Needs an MI355X."""
import numpy as np
import pytest

from molflow_sources_amd import geometry

pytestmark = pytest.mark.gpu


def low_flux_tube():
    m = geometry.tube_model()
    m.settings.low_flux_mode, m.settings.low_flux_cutoff = 1, 1e-3
    return m


@pytest.mark.parametrize("model,waves,runs_as", [
    (geometry.tube_model, 1, 2), (geometry.tube_model, 5, 4), (low_flux_tube, 1, 2),
    (lambda: geometry.time_dependent_tube("1e-3,2e-3,9.2e-3", window=2e-3), 5, 3)])
def test_choice_outside_the_built_range_fills_the_chip_like_the_nearest(model, waves, runs_as):
    from molflow_sources_amd.simulation import GpuSimulation
    sim = GpuSimulation(0)
    sim.load(model())
    sim.rebuild_accel()
    sim.set_carry(True)
    parked, hits = [], []
    for w in (waves, runs_as):
        sim.set_kernel_variant(w)
        sim.reset(seed=3)
        sim.run(1_000_000)          # more than the lanes: what is parked is about one particle a lane
        parked.append(sim.in_flight())
        sim.drain()
        hits.append(sim.read().facets["nb_mc_hit"])
        sim.set_carry(True)
    sim.close()
    # parked lanes differ by the few that each wave had free when it looked
    assert abs(parked[0] - parked[1]) < 0.05 * parked[1]
    assert np.array_equal(hits[0], hits[1])
