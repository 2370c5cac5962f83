"""GPU test of pass A on both sides of its dispatch by the boundary's share: a
boundary counts more while its own sums are to be formed (the first step) than
once they are kept, so that the steps of one scene may go different ways (a quad
of lanes per particle, or one).  Every step matches a grouped one, which takes
one lane always, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dimension, precision, fluid block, inner tank, wall layers): quads from the
# first step, from the second on, and never
CASES = [(3, 4, [20] * 3, [60, 40, 40], 2), (3, 4, [40] * 3, [200, 130, 130], 2), (3, 4, [53] * 3, [60, 56, 56], 2),
         (3, 8, [20] * 3, [60, 40, 40], 2), (3, 8, [40] * 3, [100, 80, 80], 2), (3, 8, [46] * 3, [60, 56, 56], 2),
         (2, 4, [200, 200], [600, 400], 40), (2, 8, [200, 200], [600, 400], 20), (2, 8, [200, 200], [600, 400], 60)]


@pytest.mark.parametrize("case", range(len(CASES)))
def test_steps_on_both_sides_match_one_lane(case):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.batch import SceneBatch
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    dim, precision, block, inner, layers = CASES[case]
    scn = tank(0.01, inner, layers, [([0] * dim, block, [1])], [1000], [0, -9.81, 0][:dim], 0.01)
    cfg = solver_config("DFSPH", cs=100)
    a, b = (simulation_from_dicts(cfg, scn, precision=precision, cfl=False) for _ in range(2))
    print(f"[case] {dim}D precision {precision}: {a.fluid.part_num} + {a.bound.part_num}", flush=True)
    rng = np.random.default_rng(1)
    x = a.fluid.to_numpy("pos")
    x = (x + rng.uniform(-1e-3, 1e-3, x.shape)).astype(a.fluid.np_dtype)
    for sim in (a, b):
        sim.fluid.from_numpy("pos", x)
    batch = SceneBatch([b])
    for step in range(3):
        a.sph_step()
        batch.step()
        for f in ("W", "sph_density", "alpha", "alpha_1", "pos", "vel"):
            assert np.array_equal(a.fluid.to_numpy(f), b.fluid.to_numpy(f)), (step, f)
        for f in ("W", "sph_density", "alpha", "alpha_2"):
            assert np.array_equal(a.bound.to_numpy(f), b.bound.to_numpy(f)), (step, f)
        if step == 1:  # the boundary's sums are formed again
            for sim in (a, b):
                sim.bound.invalidate_static_sums()
