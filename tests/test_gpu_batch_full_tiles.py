"""GPU test of a batch of more than 2,048 fluid tiles (524,288 particles), where
a block of the grouped sweeps takes a whole tile in several rounds: every scene
matches its own sph_step() bit for bit, in FP32 and FP64, with surface tension
(one phase, and a mixture) beside a scene without it, with one block per tile
and with a small number of blocks that each go through many."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

EDGE = 58  # three scenes of 58^3 particles: 2,289 tiles


def scenes():
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    out = []
    for phases, solver, gamma in ((1, "DFSPH", 0.07), (2, "VFSPH", 0.07), (1, "DFSPH", 0.0)):
        vf, rho = ([1], [1000]) if phases == 1 else ([1, 0], [1000, 500])
        scn = tank(0.01, [EDGE + 6, EDGE + 2, EDGE + 2], 2, [([0, 0, 0], [EDGE] * 3, vf)], rho, [0, -9.81, 0], 0.01)
        out.append((solver_config(solver, cs=100, gamma=gamma), scn))
    return out


def make(precision):
    from tichi_sph_amd import simulation_from_dicts
    rng = np.random.default_rng(2)
    sims = [simulation_from_dicts(c, s, precision=precision, cfl=False) for c, s in scenes()]
    for sim in sims:
        f = sim.fluid
        x = f.to_numpy("pos")
        f.from_numpy("pos", (x + rng.uniform(-1e-3, 1e-3, x.shape)).astype(f.np_dtype))
        f.from_numpy("vel", rng.normal(0, 0.2, x.shape).astype(f.np_dtype))
    return sims


@pytest.mark.parametrize("precision", [4, 8])
def test_whole_tiles_in_rounds_match_single_scenes(precision):
    from tichi_sph_amd.batch import SceneBatch
    print(f"[case] 3 x {EDGE}^3, precision {precision}", flush=True)
    ref = make(precision)
    assert sum(-(-s.fluid.part_num // 256) for s in ref) > 2048
    batches = [SceneBatch(make(precision)) for _ in range(2)]
    for g in batches[1].grid:
        batches[1].grid[g] = 101
    for step in range(2):
        want = [sim.sph_step(stats=True) for sim in ref]
        for batch in batches:
            di, ii = batch.step()
            for k, (sim, st) in enumerate(zip(batch.sims, want)):
                assert (int(di[k]), int(ii[k])) == (st.div_iter, st.incom_iter), (step, k)
                assert sim.control().compression == st.compression, (step, k)
                for f in ("pos", "vel", "acce_adv", "psi_adv"):
                    assert np.array_equal(sim.fluid.to_numpy(f), ref[k].fluid.to_numpy(f)), (step, k, f)
