"""GPU test of the reverse sweeps on both sides of their dispatch (four lanes
per particle up to 49,152 FP64 particles, two above): a block of 27,000
particles stepped and reversed alone, and twice in one tank, far apart.  The
loss sum |v|^2 and the pair sums do not couple the blocks.  Their coordinates
are multiples of 2^-20 m, so the pair distances are bit-equal, and each of the
two has the single one's gradient up to the order of its FP64 sums (1e-15);
1e-9 of the largest component leaves room for their way through the solves."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EDGE = 30
SHIFT = 27 / 64  # of the second block, 42 particles and a little


def gradient(starts):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.adjoint import DiffRunner, rollout
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(0.01, [84, 42, 42], 2, [(list(s), [EDGE] * 3, [1]) for s in starts], [1000], [0, -9.81, 0], 0.01)
    cfg = solver_config("DFSPH", cs=100)
    sim = simulation_from_dicts(cfg, scn, precision=8, cfl=False)
    n = sim.fluid.part_num
    assert n == len(starts) * EDGE ** 3
    x = np.round(sim.fluid.to_numpy("pos")[:EDGE ** 3] * 2.0 ** 20) * 2.0 ** -20
    sim.fluid.from_numpy("pos", np.concatenate([x + [SHIFT * k, 0, 0] for k in range(len(starts))]))
    r = DiffRunner(sim)
    v = np.random.default_rng(5).normal(0, 0.1, (EDGE ** 3, 3))
    v0 = torch.tensor(np.tile(v, (len(starts), 1)), device=sim.device, requires_grad=True)
    mu = torch.tensor(0.05, dtype=torch.float64, device=sim.device, requires_grad=True)
    _, vel = rollout(r, v0, mu, 0.0, 2)
    (vel ** 2).sum().backward()
    return v0.grad.cpu().numpy().reshape(len(starts), EDGE ** 3, 3), float(mu.grad)


def test_two_distant_blocks_have_the_single_blocks_gradient():
    print(f"[case] {EDGE}^3 particles once and twice", flush=True)
    (one,), mu1 = gradient([(6, 6, 6)])
    two, mu2 = gradient([(6, 6, 6), (48, 6, 6)])
    scale = np.abs(one).max()
    assert scale > 0
    for g in two:
        assert np.abs(g - one).max() <= 1e-9 * scale
    assert abs(mu2 - 2 * mu1) <= 1e-9 * abs(mu2)
