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


def _lists(sim):
    """The fluid and boundary lists' counts and entries, slot by slot."""
    f = sim.fluid
    n, cap = f.part_num, f.t["pos"].shape[0]
    out = []
    for rows, count, limit in (("nbr_f", "nbr_nf", f.list_cap_f), ("nbr_b", "nbr_nb", f.list_cap_b)):
        cnt = f.t[count][:n].cpu().numpy()
        lst = f.t[rows].cpu().numpy().reshape(limit, cap)[:, :n]
        out += [cnt, np.where(np.arange(limit)[:, None] < np.minimum(cnt, limit)[None, :], lst, -1)]
    return out


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("caps", [(64, 48), (9, 3)], ids=["lists", "overflow"])
def test_pass_a_by_quads_is_that_by_single_lanes(dim, precision, caps):
    """A small scene's own step runs pass A with a quad of lanes per particle,
    a grouped step with one: every field and list entry is the same, bit for
    bit, also where lists overflow, and around particles outside the grid, at
    one position, or crowded into one cell (more than a list in LDS holds)."""
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.batch import SceneBatch
    scn, cfg = scene((33, 29, 0) if dim == 2 else (11, 13, 9))
    rng = np.random.default_rng(7)
    sims = []
    for _ in range(2):
        sim = simulation_from_dicts(cfg, scn, precision=precision, cfl=False, list_cap_f=caps[0], list_cap_b=caps[1])
        sims.append(sim)
    x = sims[0].fluid.to_numpy("pos")
    x = x + rng.uniform(-0.2, 0.2, x.shape) * sims[0].config.part_size[1]
    x[5] = x[4]
    x[6] = -1.0
    x[7] = 1e9
    x[40:140] = x[30] + rng.uniform(-0.1, 0.1, (100, dim)) * sims[0].config.part_size[1]
    for sim in sims:
        sim.fluid.from_numpy("pos", x.astype(sim.fluid.np_dtype))
    batch = SceneBatch([sims[1]])
    sims[0].sph_step()
    batch.step()
    names = ("W", "sph_density", "sph_compression", "alpha", "alpha_1", "alpha_2", "vol", "pos", "vel")
    for name in names:
        assert np.array_equal(sims[0].fluid.to_numpy(name), sims[1].fluid.to_numpy(name), equal_nan=True), name
    for name in names[:4] + ("alpha_2",):
        assert np.array_equal(sims[0].bound.to_numpy(name), sims[1].bound.to_numpy(name), equal_nan=True), name
    for a, b in zip(_lists(sims[0]), _lists(sims[1])):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("block", BLOCKS, ids=lambda b: "x".join(map(str, b)))
def test_reference_kernels_at_block_edges_match_oracle(block, precision):
    """The sph.py kernels one by one (a quad of lanes per particle in the pair
    kernels) against the oracle, bit for bit, with surface tension."""
    from tichi_sph_amd import simulation_from_dicts
    scn, cfg = scene(block)
    cfg["solver_surface_tension_gamma"] = 0.07
    print(f"[case] block {block} precision {precision}", flush=True)
    sim = simulation_from_dicts(cfg, scn, precision=precision)
    o = O.Oracle(cfg, scn, precision)
    o.init_scenario()
    d_it, i_it, _, _, _ = sim.sph_step_reference()
    st = o.step(O.STEP_CFL)
    assert (d_it, i_it) == (st.div_iter, st.incom_iter)
    for obj, fl, names in ((0, sim.fluid, ("pos", "vel", "sph_density", "alpha", "psi_adv", "acce_adv", "normal")),
                           (1, sim.bound, ("W", "sph_density", "alpha"))):
        for f in names:
            assert np.array_equal(fl.to_numpy(f), o.get(obj, f).reshape(fl.to_numpy(f).shape)), (obj, f)
