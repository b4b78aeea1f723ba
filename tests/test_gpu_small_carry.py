"""Small runs that keep particles in flight: a run ends when the queue is
empty and parks what is left, however few particles there are, and the runs
and the drain together count what one run counts. Needs an MI355X."""
import numpy as np
import pytest

from molflow_sources_amd import geometry

pytestmark = pytest.mark.gpu


def low_flux_tube():
    m = geometry.tube_model()
    m.facets["sticking"][3:200] = 0.2
    m.settings.low_flux_mode, m.settings.low_flux_cutoff = 1, 1e-4
    return m


MODELS = {
    "tube": geometry.tube_model,
    "low flux": low_flux_tube,
    "moments": lambda: geometry.time_dependent_tube("1e-3,2e-3,9.2e-3", window=2e-3),
}


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("n", [100, 1000, 20_000])
@pytest.mark.parametrize("name", sorted(MODELS))
def test_small_runs_park_their_particles(name, n, graph):
    from molflow_sources_amd.simulation import GpuSimulation
    sim = GpuSimulation(0)
    sim.load(MODELS[name]())
    sim.rebuild_accel()
    sim.enable_graph(graph)
    k = 4
    sim.reset(seed=31)
    sim.run(k * n)
    one = sim.read()
    sim.reset(seed=31)
    sim.set_carry(True)
    parked = []
    for _ in range(k):
        assert sim.run(n).desorbed == n
        parked.append(sim.in_flight())
    # a wave of 64 ends with its first free lane, after a tenth of a
    # particle's events or so: most of a run's particles are still in flight
    assert all(p > n // 2 for p in parked)
    sim.drain()
    two = sim.read()
    sim.close()
    for fld in ("nb_mc_hit", "nb_desorbed"):
        assert np.array_equal(one.facets[fld], two.facets[fld])
    for fld in ("nb_hit_equiv", "nb_abs_equiv", "sum_1_per_ort_velocity", "sum_v_ort"):
        assert np.allclose(one.facets[fld], two.facets[fld], rtol=1e-9, atol=1e-9)


def test_small_runs_of_variants_park_their_particles():
    from molflow_sources_amd.simulation import GpuSimulation
    ms = geometry.variant_models(5, 2000, 4000, seed=7)
    sim = GpuSimulation(0)
    sim.load_variants(ms)
    sim.rebuild_accel()
    n = np.array([10, 200, 35, 64, 1], dtype=np.uint64)
    seeds = np.arange(5, dtype=np.uint64)
    sim.reset(seed=1)
    sim.run_variants(3 * n, seeds)
    one = [sim.read(variant=v).facets["nb_mc_hit"] for v in range(5)]
    sim.reset(seed=1)
    sim.set_carry(True)
    for _ in range(3):
        sim.run_variants(n, seeds)
        assert sim.in_flight() > int(n.sum()) // 2
    sim.drain()
    assert all(np.array_equal(a, sim.read(variant=v).facets["nb_mc_hit"]) for v, a in enumerate(one))
    sim.close()
