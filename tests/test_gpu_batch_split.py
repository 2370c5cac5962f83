"""GPU test of a batch's solver sweeps on both sides of the tile counts from which
they take whole tiles instead of split ones (the update 512 in FP64 and 896 in FP32,
psi 3072 in FP64), in 2D and 3D: every scene matches its own sph_step() bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (precision, dim, particles along an edge of each scene, tiles of 256 particles)
CASES = [(8, 3, (20,) * 15 + (19,), 507), (8, 3, (20,) * 16, 512), (8, 2, (90,) * 16, 512),
         (4, 3, (20,) * 27 + (19,), 891), (4, 3, (20,) * 28, 896), (4, 2, (90,) * 28, 896),
         (8, 2, (626, 627), 3067), (8, 2, (627, 628), 3077)]


def make(dim, edges, precision):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    rng = np.random.default_rng(4)
    sims = []
    for e in edges:
        scn = tank(0.01, [e + 6] + [e + 2] * (dim - 1), 2, [([0] * dim, [e] * dim, [1])], [1000],
                   [0, -9.81, 0][:dim], 0.01)
        sim = simulation_from_dicts(solver_config("DFSPH", cs=100, gamma=0.0), scn, precision=precision, cfl=False)
        f = sim.fluid
        x = f.to_numpy("pos")
        f.from_numpy("pos", (x + rng.uniform(-1e-3, 1e-3, x.shape)).astype(f.np_dtype))
        f.from_numpy("vel", rng.normal(0, 0.2, x.shape).astype(f.np_dtype))
        sims.append(sim)
    return sims


@pytest.mark.parametrize("precision,dim,edges,tiles", CASES)
def test_sweeps_match_on_both_sides_of_the_lines(precision, dim, edges, tiles):
    from tichi_sph_amd.batch import SceneBatch
    print(f"[case] {dim}D {tiles} tiles precision {precision}", flush=True)
    ref, batch = make(dim, edges, precision), SceneBatch(make(dim, edges, precision))
    assert batch.info.tiles[0] == tiles
    want = [sim.sph_step(stats=True) for sim in ref]
    di, ii = batch.step()
    for k, (sim, st) in enumerate(zip(batch.sims, want)):
        assert (int(di[k]), int(ii[k])) == (st.div_iter, st.incom_iter), k
        assert sim.control().compression == st.compression, k
        for f in ("pos", "vel", "acce_adv", "psi_adv"):
            assert np.array_equal(sim.fluid.to_numpy(f), ref[k].fluid.to_numpy(f)), (k, f)
