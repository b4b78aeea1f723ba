"""A tree rebuild that is refused leaves the context with the tree it had:
first hits and tallies stay the oracle's. Needs an MI355X."""
import numpy as np
import pytest

from molflow_sources_amd.model import Model, default_facets
from oracle.mfcpu import CpuModel

pytestmark = pytest.mark.gpu


def nested_triangles(n=100, ratio=1.2):
    """n parallel 2-sided triangles about the (1,1,1) axis, each `ratio`
    times smaller and nearer to the corner than the one before: the builder
    splits off the largest few at a time, so with one facet a leaf the 8-wide
    tree is 11 levels deep (8 are accepted), with 16 it is 2."""
    s = 10.0 * ratio ** -np.arange(n, dtype=float)
    tri = np.array([[1.0, 0.5, 0.5], [0.5, 1.0, 0.5], [0.5, 0.5, 1.0]])
    F = default_facets(n)
    F["is_2sided"], F["sticking"] = 1, 0.5
    F["desorb_type"][0], F["outgassing"][0] = 2, 1.0
    return Model((s[:, None, None] * tri).reshape(-1, 3), np.arange(3 * n).reshape(n, 3).tolist(), F, name="nested")


@pytest.mark.parametrize("n_rays", [1, 8, 64, 3000])
def test_refused_rebuild_keeps_the_tree_in_use(n_rays):
    from molflow_sources_amd.simulation import GpuSimulation, MolflowGpuError
    m = nested_triangles()
    cpu = CpuModel(m)
    rng = np.random.default_rng(3)
    o = np.full((n_rays, 3), 12.0) + rng.uniform(-0.5, 0.5, (n_rays, 3))
    d = -o / np.linalg.norm(o, axis=1)[:, None]
    d[::2] *= -1.0
    o[::2] = rng.uniform(0.0, 1e-6, (len(o[::2]), 3))
    last = rng.integers(-1, m.n_facets, n_rays).astype(np.int32)
    ref = cpu.intersect(o, d, last, brute=True)
    sim = GpuSimulation(0)
    sim.load(m)
    sim.rebuild_accel(8, 16)
    with pytest.raises(MolflowGpuError, match="deep"):
        sim.rebuild_accel(8, 1)
    got = sim.intersect(o, d, last)
    assert np.array_equal(got[0], ref[0])
    assert (ref[0] >= 0).any()
    n = 40 * n_rays
    sim.reset(seed=5)
    sim.run(n)
    t, c = sim.read(), CpuModel(m).run(n, seed=5)
    # a trajectory may part by FP64 rounding of the math library
    a, b = t.facets["nb_mc_hit"].astype(np.int64), c.facets["nb_mc_hit"].astype(np.int64)
    assert t.desorbed == n and np.abs(a - b).sum() <= 2 + 2e-4 * b.sum()
    # a rebuild that is accepted after it counts the same
    sim.rebuild_accel(8, 2)
    assert np.array_equal(sim.intersect(o, d, last)[0], ref[0])
    sim.close()


def test_context_without_a_tree_stays_without_one():
    from molflow_sources_amd.simulation import GpuSimulation, MolflowGpuError
    sim = GpuSimulation(0)
    sim.load(nested_triangles())
    with pytest.raises(MolflowGpuError, match="deep"):
        sim.rebuild_accel(8, 1)
    with pytest.raises(MolflowGpuError, match="not built"):
        sim.run(10)
    sim.close()
