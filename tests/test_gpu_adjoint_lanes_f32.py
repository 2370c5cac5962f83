"""GPU test of the FP32 reverse Jacobi sweeps on both sides of their dispatch
(four lanes per particle up to 262,144 particles, two above): a block of 140,608
particles stepped and reversed alone, and twice in one tank.  The blocks lie a
whole number of cells apart and all lengths are multiples of 2^-20 m, so the
forward pass of each is that of the single one bit for bit, clamps included, and
the gradients differ by the order of the FP32 sums alone: some 60 terms a sum
(60 * 2^-24 = 4e-6 of their size), through one step (positions of a second would
round apart) of two solves of two iterations; 1e-4 of the largest component
leaves a factor of 3 on top of eight such sums in a row."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

EDGE, GPS = 52, 1 / 64
SHIFT = 60 * GPS  # of the second block: 30 cells of two particle sizes


def gradient(starts):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.adjoint import DiffRunner, rollout
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(GPS, [126, 64, 64], 2, [(list(s), [EDGE] * 3, [1]) for s in starts], [1000], [0, -9.75, 0], GPS)
    cfg = solver_config("DFSPH", cs=100)
    sim = simulation_from_dicts(cfg, scn, precision=4, cfl=False)
    n = sim.fluid.part_num
    assert n == len(starts) * EDGE ** 3
    x = np.round(sim.fluid.to_numpy("pos")[:EDGE ** 3].astype(np.float64) * 2.0 ** 20) * 2.0 ** -20
    sim.fluid.from_numpy("pos", np.concatenate([x + [SHIFT * k, 0, 0] for k in range(len(starts))]))
    r = DiffRunner(sim)
    r.force = [(2, 2)]  # the mean errors differ by their own order of sums
    v = np.random.default_rng(5).normal(0, 0.1, (EDGE ** 3, 3)).astype(np.float32)
    v0 = torch.tensor(np.tile(v, (len(starts), 1)), device=sim.device, requires_grad=True)
    xs, vel = rollout(r, v0, 0.05, 0.0, 1)
    (vel.double() ** 2).sum().backward()
    out = vel.detach().cpu().numpy().reshape(len(starts), EDGE ** 3, 3)
    return v0.grad.cpu().numpy().reshape(len(starts), EDGE ** 3, 3).astype(np.float64), out


def test_two_distant_blocks_have_the_single_blocks_gradient_in_fp32():
    print(f"[case] {EDGE}^3 particles once and twice, FP32", flush=True)
    (one,), (vel,) = gradient([(6, 6, 6)])
    two, vels = gradient([(6, 6, 6), (66, 6, 6)])
    scale = np.abs(one).max()
    assert scale > 0
    for g, v in zip(two, vels):
        assert np.array_equal(v, vel)
        assert np.abs(g - one).max() <= 1e-4 * scale
    print(f"  largest difference {max(np.abs(g - one).max() for g in two) / scale:.2e}", flush=True)
    assert any((g != one).any() for g in two)  # the two sides do sum in another order
