"""The wave's shared ray walk: batches at the edges of a wave and models
whose boxes nearly all overlap, so that a node step hits most of its
children and the task stack and the facet list run into their capacities.
First hits against the oracle's brute force, bit for bit. Needs an MI355X."""
import numpy as np
import pytest

from helpers import random_rays
from molflow_sources_amd import geometry
from molflow_sources_amd.model import Model, default_facets
from oracle.mfcpu import CpuModel

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def sim():
    from molflow_sources_amd.simulation import GpuSimulation
    s = GpuSimulation(0)
    yield s
    s.close()


def triangle_soup(n, seed=3):
    """n large random 2-sided triangles through the middle of a 10 cm cube."""
    rng = np.random.default_rng(seed)
    V = rng.uniform(0.0, 10.0, (3 * n, 3))
    F = default_facets(n)
    F["is_2sided"] = 1
    F["sticking"] = 0.5
    F["desorb_type"][0], F["outgassing"][0] = 2, 1.0
    return Model(V, np.arange(3 * n).reshape(n, 3).tolist(), F, name="soup")


@pytest.mark.parametrize("width,leaf", [(8, 1), (8, 2), (8, 3), (8, 16), (4, 2)])
@pytest.mark.parametrize("n_rays", [1, 63, 65, 140_000])
def test_overlapping_boxes_first_hits(sim, width, leaf, n_rays):
    m = triangle_soup(1500)
    sim.load(m)
    sim.rebuild_accel(width, leaf)
    o, d = random_rays(n_rays, [-1] * 3, [11] * 3, seed=5)
    last = np.random.default_rng(6).integers(-1, m.n_facets, n_rays).astype(np.int32)
    got = sim.intersect(o, d, last)
    ref = CpuModel(m).intersect(o, d, last, brute=True)
    assert np.array_equal(got[0], ref[0]), f"{int((got[0] != ref[0]).sum())} first-hit facets differ"
    hit = ref[0] >= 0
    for a, b in zip(got[1:], ref[1:]):
        assert np.allclose(a[hit], b[hit], rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("n_facets", [1, 2, 8, 9, 12, 64, 1500])
@pytest.mark.parametrize("n_rays", [1, 2, 3])
def test_few_rays_first_hits(sim, n_facets, n_rays):
    """Waves of one and two rays, which start at the children of the root,
    and of three, on trees whose root is a leaf's parent only, has leaves
    beside inner children, and has inner children only."""
    m = triangle_soup(n_facets)
    cpu = CpuModel(m)
    sim.load(m)
    o, d = random_rays(40 * n_rays, [-1] * 3, [11] * 3, seed=7)
    last = np.random.default_rng(8).integers(-1, m.n_facets, len(o)).astype(np.int32)
    ref = cpu.intersect(o, d, last, brute=True)
    for width, leaf in ((8, 1), (4, 2)):
        sim.rebuild_accel(width, leaf)
        for i in range(0, len(o), n_rays):
            got = sim.intersect(o[i:i + n_rays], d[i:i + n_rays], last[i:i + n_rays])
            assert np.array_equal(got[0], ref[0][i:i + n_rays]), f"rays from {i}"
            assert np.allclose(got[1], np.where(got[0] >= 0, ref[1][i:i + n_rays], got[1]), rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("n_des", [1, 64, 1025, 8192, 8193, 200_001])
def test_lane_quota_same_seed_tallies(sim, n_des):
    """Runs of fewer particles than waves, of a few per wave of one block per
    CU, just beyond that, and of more than lanes (lane quota 1, 1, 2, 8, 3,
    64) count what the oracle counts."""
    m = geometry.tube_model(1.0, 3.0, 16, 6)
    sim.load(m)
    sim.rebuild_accel()
    sim.reset(seed=9)
    sim.run(n_des)
    t, c = sim.read(), CpuModel(m).run(n_des, seed=9)
    assert t.desorbed == n_des
    a, b = t.facets[0]["nb_mc_hit"].astype(np.int64), c.facets[0]["nb_mc_hit"].astype(np.int64)
    # a few long trajectories may part by FP64 rounding of the math library
    assert np.abs(a - b).sum() <= 2e-4 * b.sum()


def test_parked_lean_particles_resume_in_the_full_kernel(sim):
    """Particles parked by the kernel without a clock and resumed by the one
    with it (event tracing switches kernels) end as in one run."""
    m = geometry.tube_model(1.0, 6.0, 16, 8)
    n = 200_000
    sim.load(m)
    sim.rebuild_accel()
    sim.set_carry(False)
    sim.reset(seed=4)
    sim.run(n)
    one = sim.read()
    sim.reset(seed=4)
    sim.set_carry(True)
    sim.run(n)
    parked = sim.in_flight()
    sim.set_trace(8, 16)
    sim.drain()
    sim.set_trace(0, 0)
    two = sim.read()
    assert parked > 1000
    for fld in ("nb_mc_hit", "nb_desorbed"):
        assert np.array_equal(one.facets[fld], two.facets[fld])
    for fld in ("nb_abs_equiv", "sum_1_per_ort_velocity", "sum_v_ort", "sum_1_per_velocity"):
        assert np.allclose(one.facets[fld], two.facets[fld], rtol=1e-9, atol=0)
    assert one.glob[0]["nb_mc_hit"] == two.glob[0]["nb_mc_hit"]
    assert np.isclose(one.glob[0]["dist_traveled_total"], two.glob[0]["dist_traveled_total"], rtol=1e-12)


@pytest.mark.parametrize("moments,sheets", [(3, 1), (150, 1), (12, 7), (0, 6)])
def test_moment_and_profile_sums_kept_in_lds(sim, moments, sheets):
    """Counters and profiles of hot facets with all, some or one of their
    slots summed in LDS, more profiles than are kept there (more than 4), and
    rays that cross more transparent sheets than the walk notes (more than
    4), against the oracle on the same seed."""
    from molflow_sources_amd import _abi as A
    m = geometry.time_dependent_tube("0.1e-3,0.2e-3,%g" % (0.2e-3 * (max(moments, 1) - 0.4)), window=0.2e-3)
    if moments == 0:
        m.moments = []
        m.settings.calc_constant_flow = 1
        m.facets["outgassing_param"][0] = -1
    V, F = [m.vertices], [m.facets]
    nv = len(m.vertices)
    for k in range(sheets - 1):
        z = 1.0 + 8.0 * k / max(1, sheets - 2)
        V.append(np.array([[-0.6, -0.6, z], [0.6, -0.6, z], [0.6, 0.6, z], [-0.6, 0.6, z]]))
        m.polygons.append([nv, nv + 1, nv + 2, nv + 3])
        nv += 4
        f = default_facets(1)
        f["opacity"], f["is_2sided"], f["profile_type"] = 0.25 * (k % 2), 1, A.PROFILE_V
        F.append(f)
    m.vertices, m.facets = np.concatenate(V), np.concatenate(F)
    n = 30_000
    sim.load(m)
    sim.rebuild_accel()
    sim.reset(seed=11)
    sim.run(n)
    t, c = sim.read(), CpuModel(m).run(n, seed=11)
    assert t.n_slots == 1 + moments
    assert t.desorbed == n
    # a few long trajectories may part by FP64 rounding of the math library
    for a, b in ((t.facets["nb_mc_hit"], c.facets["nb_mc_hit"]), (t.facets["nb_desorbed"], c.facets["nb_desorbed"])):
        a, b = a.astype(np.int64), b.astype(np.int64)
        assert np.abs(a - b).sum() <= 1e-3 * b.sum()
    for a, b in [(t.facets[k], c.facets[k]) for k in ("nb_hit_equiv", "nb_abs_equiv", "sum_v_ort", "sum_1_per_ort_velocity")] + \
                [(t.profiles[k], c.profiles[k]) for k in ("count_equiv", "sum_v_ort", "sum_1_per_ort_velocity")]:
        assert b.sum() > 0
        assert np.abs(a - b).sum() <= 2e-3 * b.sum()
