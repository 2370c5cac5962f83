"""GPU test of surface tension in a batch: by one lane per particle (2D scenes of
more than 73,728 particles together, where a scene's own step takes four), by four
lanes, and the velocity update alone, in one launch.  Every scene matches its own
sph_step() bit for bit, with one block per tile and with few blocks that each go
through many, and with neighbour lists that overflow."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (dim, particles along an edge of each scene): below the 2D line, above it, 3D
CASES = [(2, (50, 7, 41)), (2, (161, 155, 161, 7)), (3, (19, 6, 23))]


def make(dim, edges, precision, full):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    rng = np.random.default_rng(3)
    sims = []
    for q, e in enumerate(edges):
        gamma = 0.0 if q % 3 == 1 else 0.07
        scn = tank(0.01, [e + 6] + [e + 2] * (dim - 1), 2, [([0] * dim, [e] * dim, [1])], [1000],
                   [0, -9.81, 0][:dim], 0.01)
        sim = simulation_from_dicts(solver_config("DFSPH", cs=100, gamma=gamma), scn, precision=precision,
                                    cfl=False, list_cap_f=64 if full else (9 if dim == 2 else 30))
        f = sim.fluid
        x = f.to_numpy("pos")
        f.from_numpy("pos", (x + rng.uniform(-1e-3, 1e-3, x.shape)).astype(f.np_dtype))
        f.from_numpy("vel", rng.normal(0, 0.2, x.shape).astype(f.np_dtype))
        sims.append(sim)
    return sims


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("dim,edges", CASES)
@pytest.mark.parametrize("full", [True, False])
def test_grouped_tension_matches_single_scenes(dim, edges, precision, full):
    from tichi_sph_amd.batch import SceneBatch
    print(f"[case] {dim}D {edges} precision {precision} full lists {full}", flush=True)
    ref = make(dim, edges, precision, full)
    batches = [SceneBatch(make(dim, edges, precision, full)) for _ in range(2)]
    for g in batches[1].grid:
        batches[1].grid[g] = 37
    for step in range(2):
        want = [sim.sph_step(stats=True) for sim in ref]
        over = [int((sim.fluid.to_numpy("nbr_nf") > sim.fluid.list_cap_f).sum()) for sim in ref]
        assert full == (sum(over) == 0)
        for batch in batches:
            di, ii = batch.step()
            for k, (sim, st) in enumerate(zip(batch.sims, want)):
                assert (int(di[k]), int(ii[k])) == (st.div_iter, st.incom_iter), (step, k)
                for f in ("pos", "vel", "vel_adv", "acce_adv", "psi_adv"):
                    assert np.array_equal(sim.fluid.to_numpy(f), ref[k].fluid.to_numpy(f)), (step, k, f)
