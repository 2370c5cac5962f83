"""GPU tests of the surface-tension walks, forward and reverse: a candidate that
the 0.99 gate leaves out takes no part, whatever its normal or its velocity
gradient holds.  Four particles in a row: a pair within h of each other, past h
of it (in a neighbouring cell) one below the gate, and next to that the last."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

H = 0.02  # two particle sizes


def row(solver, phases, **kw):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(0.01, [14, 9, 9], 2, [([3, 4, 4], [4, 1, 1], [1, 0][:phases])], [1000, 500][:phases], [0, -9.81, 0], 0.01)
    sim = simulation_from_dicts(solver_config(solver, cs=100, gamma=0.07), scn, cfl=False, **kw)
    f = sim.fluid
    assert f.part_num == 4
    x = f.to_numpy("pos")
    x[:] = x[0]
    x[:, 0] += [0, 0.75 * H, 1.95 * H, 2.7 * H]
    f.from_numpy("pos", x)
    vf = f.to_numpy("volume_frac")
    vf[2:] = 0.5
    f.from_numpy("volume_frac", vf)
    return sim


@pytest.mark.parametrize("precision", [4, 8])
def test_a_gated_candidates_normal_is_not_read(precision):
    got = []
    for bad in (False, True):
        sim = row("VFSPH", 2, precision=precision)
        if bad:
            rv = sim.fluid.to_numpy("rest_volume")
            rv[3] = np.inf  # over its compression a NaN, and so is its neighbour's normal
            sim.fluid.from_numpy("rest_volume", rv)
        sim.sph_step()
        normal = sim.fluid.to_numpy("normal")
        assert np.isnan(normal[2]).any() == bad
        got.append([sim.fluid.to_numpy(f)[:2] for f in ("acce_adv", "vel", "pos")])
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("precision", [4, 8])
def test_a_gated_candidates_gradient_is_not_read(precision):
    from tichi_sph_amd.adjoint import DiffRunner, rollout
    got = []
    for bad in (False, True):
        r = DiffRunner(row("DFSPH", 1, precision=precision))
        dt = torch.float32 if precision == 4 else torch.float64
        v0 = torch.zeros(4, 3, dtype=dt, device="cuda", requires_grad=True)
        weight = torch.arange(12, dtype=dt, device="cuda").reshape(4, 3)
        if bad:
            weight[2] = np.nan
        gamma = torch.tensor(0.07, dtype=dt, device="cuda", requires_grad=True)
        x, v = rollout(r, v0, 0.05, gamma, 2)
        torch.autograd.backward((x, v), (torch.zeros_like(x), weight))
        grad = v0.grad.cpu().numpy()
        assert np.isnan(grad[2]).all() == bad
        got.append(np.append(grad[:2], gamma.grad.item()))
    assert np.isfinite(got[0]).all() and np.array_equal(got[0], got[1])
