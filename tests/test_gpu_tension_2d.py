"""GPU tests of 2D scenes with surface tension on both sides of the size from
which one lane takes a particle instead of a quad (73,728 particles forward,
98,304 reverse): the step against the oracle (the single-step bar of 1e-5 of
max(|value|, RMS)), every scene of a batch against its own step bit for bit, and
the gradients of a block alone and twice in one tank (FP64, the order of sums of
some 60 terms, 1e-14, through the solves; 1e-9 of the largest component)."""
import numpy as np
import pytest
import torch

import oracle as O
from test_gpu_parity import TOL, rel_err

pytestmark = pytest.mark.gpu


def scene(w, h, tank_w=None, blocks=1, shift=0):
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(0.02, [tank_w or w + 20, h + 10], 3, [([4 + shift * k, 4], [w, h], [1]) for k in range(blocks)], [1000],
               [0, -9.81], 0.01)
    return solver_config("DFSPH", cs=50, gamma=0.07), scn


def stir(sim, seed):
    f = sim.fluid
    x = f.to_numpy("pos")
    rng = np.random.default_rng(seed)
    f.from_numpy("pos", (x + rng.uniform(-2e-3, 2e-3, x.shape)).astype(f.np_dtype))
    f.from_numpy("vel", rng.normal(0, 0.2, x.shape).astype(f.np_dtype))


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("w,h", [(271, 272), (272, 273)])
def test_step_matches_oracle(w, h, precision):
    from tichi_sph_amd import simulation_from_dicts
    cfg, scn = scene(w, h)
    print(f"[case] {w} x {h} = {w * h}", flush=True)
    sim = simulation_from_dicts(cfg, scn, precision=precision)
    stir(sim, 1)
    o = O.Oracle(cfg, scn, precision)
    o.init_scenario()
    for f in ("pos", "vel"):
        o.set(0, f, sim.fluid.to_numpy(f))
    s, st = sim.sph_step(stats=True), o.step(O.STEP_CFL)
    assert (s.div_iter, s.incom_iter) == (st.div_iter, st.incom_iter)
    # (the accelerations of an FP32 oracle are themselves 7e-6 from those in FP64)
    for f in ("pos", "vel", "acce_adv")[:2 if precision == 4 else 3]:
        assert rel_err(sim.fluid.to_numpy(f), o.get(0, f)) <= TOL, f


@pytest.mark.parametrize("precision", [4, 8])
def test_batch_is_the_single_scenes(precision):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.batch import SceneBatch
    dicts = [scene(271, 272), scene(272, 273), scene(40, 31), scene(300, 301)]
    print(f"[case] precision {precision}", flush=True)

    def make():
        sims = [simulation_from_dicts(c, s, precision=precision, cfl=False) for c, s in dicts]
        for k, sim in enumerate(sims):
            stir(sim, k)
        return sims
    ref, batch = make(), SceneBatch(make())
    for step in range(2):
        di, ii = batch.step()
        for k, sim in enumerate(ref):
            st = sim.sph_step(stats=True)
            assert (int(di[k]), int(ii[k])) == (st.div_iter, st.incom_iter), (step, k)
            for f in ("pos", "vel", "acce_adv"):
                assert np.array_equal(batch.sims[k].fluid.to_numpy(f), sim.fluid.to_numpy(f)), (step, k, f)


def gradient(blocks, w=250, h=240, gap=256):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.adjoint import DiffRunner, rollout
    cfg, scn = scene(w, h, tank_w=2 * gap + 20, blocks=blocks, shift=gap)
    sim = simulation_from_dicts(cfg, scn, precision=8, cfl=False)
    n = w * h
    assert sim.fluid.part_num == blocks * n
    x = np.round(sim.fluid.to_numpy("pos")[:n] * 2.0 ** 20) * 2.0 ** -20
    sim.fluid.from_numpy("pos", np.concatenate([x + [5.25 * k, 0] for k in range(blocks)]))
    v = np.random.default_rng(5).normal(0, 0.1, (n, 2))
    v0 = torch.tensor(np.tile(v, (blocks, 1)), device=sim.device, requires_grad=True)
    mu, gamma = (torch.tensor(a, dtype=torch.float64, device=sim.device, requires_grad=True) for a in (0.05, 0.07))
    _, vel = rollout(DiffRunner(sim), v0, mu, gamma, 2)
    (vel ** 2).sum().backward()
    return v0.grad.cpu().numpy().reshape(blocks, n, 2), float(mu.grad), float(gamma.grad)


def test_two_distant_blocks_have_the_single_blocks_gradient():
    print("[case] 60,000 particles once and twice, FP64", flush=True)
    (one,), mu1, gamma1 = gradient(1)
    two, mu2, gamma2 = gradient(2)
    scale = np.abs(one).max()
    assert scale > 0
    for g in two:
        assert np.abs(g - one).max() <= 1e-9 * scale
    assert abs(mu2 - 2 * mu1) <= 1e-9 * abs(mu2) and abs(gamma2 - 2 * gamma1) <= 1e-9 * abs(gamma2)
