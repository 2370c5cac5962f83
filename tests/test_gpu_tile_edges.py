"""GPU tests of the list sweeps at the edges of their blocks: a block of the
cooperative sweeps covers 64 (psi, advection) or 128 (update) particles and a
grouped launch's tile 256, so scenes of one particle, of one less and one more
than a block, and of a few blocks are stepped and compared with the oracle
(the single-step bar of 1e-5 of max(|value|, RMS)), and batched with each
other bit for bit."""
import numpy as np
import pytest

import oracle as O
from test_gpu_parity import TOL, rel_err

pytestmark = pytest.mark.gpu

# edges of the fluid block in particles
BLOCKS = [(1, 1, 1), (9, 7, 1), (4, 4, 4), (13, 5, 1), (127, 1, 1), (43, 3, 1), (17, 5, 3), (16, 4, 4), (257, 1, 1),
          (9, 0, 0), (8, 8, 0), (257, 1, 0)]


def scene(block):
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    d = 3 if block[2] else 2
    block = list(block[:2]) if d == 2 else list(block)
    block[1] = max(block[1], 1)
    inner = [n + 4 for n in block]
    scn = tank(0.02 if d == 2 else 0.01, inner, 3 if d == 2 else 2, [([0] * d, block, [1])], [1000],
               [0, -9.81, 0][:d], 0.01)
    scn["fluid"]["objs"][0]["vel"] = [0.3, -0.2, 0.1][:d]
    return scn, solver_config("DFSPH", cs=50 if d == 2 else 100)


@pytest.mark.parametrize("block", BLOCKS, ids=lambda b: "x".join(map(str, b)))
def test_step_at_block_edges_matches_oracle(block):
    from tichi_sph_amd import simulation_from_dicts
    scn, cfg = scene(block)
    print(f"[case] block {block}", flush=True)
    sim = simulation_from_dicts(cfg, scn)
    o = O.Oracle(cfg, scn, 4)
    o.init_scenario()
    for step in range(2):
        s = sim.sph_step(stats=True)
        st = o.step(O.STEP_CFL)
        assert (s.div_iter, s.incom_iter) == (st.div_iter, st.incom_iter), step
        for f in ("pos", "vel", "sph_density", "alpha"):
            e = rel_err(sim.fluid.to_numpy(f), o.get(0, f))
            assert e <= TOL, (step, f, e)


def test_batch_at_block_edges_is_bit_identical():
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.batch import SceneBatch
    dicts = [scene(b) for b in BLOCKS]
    ref = [simulation_from_dicts(c, s, cfl=False) for s, c in dicts]
    batch = SceneBatch([simulation_from_dicts(c, s, cfl=False) for s, c in dicts])
    for step in range(2):
        di, ii = batch.step()
        for k, sim in enumerate(ref):
            st = sim.sph_step(stats=True)
            assert (int(di[k]), int(ii[k])) == (st.div_iter, st.incom_iter), (step, BLOCKS[k])
            assert st.compression == batch.sims[k].control().compression, (step, BLOCKS[k])
            for f in ("pos", "vel"):
                assert np.array_equal(batch.sims[k].fluid.to_numpy(f), sim.fluid.to_numpy(f)), (step, BLOCKS[k], f)
