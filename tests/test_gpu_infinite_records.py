"""GPU tests of the sweeps on records that hold an infinity: the last trip over a
list reads its last neighbour again for the lanes and slots that are left over,
and what those bring must be left out, not multiplied by zero (0 * inf is a NaN).
Pass A by quads of lanes against single lanes (a grouped step) bit for bit, and
one pair whose second particle is infinite in one quantity: the psi sweep and the
gradient of the first are infinite, as the one term of their sums is."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def scene(dim, block, solver="DFSPH", mu=0.05, **kw):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(0.01, [b + 6 for b in block], 2, [([3] * dim, block, [1])], [1000], [0, -9.81, 0][:dim], mu)
    return simulation_from_dicts(solver_config(solver, cs=100), scn, cfl=False, **kw)


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("dim,obj", [(2, "fluid"), (3, "fluid"), (3, "bound")])
def test_pass_a_sums_an_infinite_mass(dim, obj, precision):
    from tichi_sph_amd.batch import SceneBatch
    sims = [scene(dim, [9, 8, 7][:dim], precision=precision) for _ in range(2)]
    rng = np.random.default_rng(3)
    x = sims[0].fluid.to_numpy("pos")
    x = (x + rng.uniform(-2e-3, 2e-3, x.shape)).astype(sims[0].fluid.np_dtype)
    x -= x.min(0) - 1e-3  # at the walls
    for sim in sims:
        sim.fluid.from_numpy("pos", x)
        o = getattr(sim, obj)
        for field in ("mass", "rest_volume"):
            a = o.to_numpy(field)
            # (of the boundary those nearest to the fluid block)
            near = np.argsort(np.linalg.norm(o.to_numpy("pos") - x.mean(0), axis=1))
            a[near[[0, 5] if field == "mass" else [3]]] = np.inf
            o.from_numpy(field, a)
    batch = SceneBatch([sims[1]])
    sims[0].sph_step()
    batch.step()
    for name in ("W", "sph_density", "sph_compression"):
        for f in ("fluid", "bound"):
            a, b = (getattr(s, f).to_numpy(name) for s in sims)
            assert np.array_equal(a, b, equal_nan=True), (f, name)
    density = sims[0].fluid.to_numpy("sph_density")
    assert np.isinf(density).sum() > 5 and not np.isnan(density).any()


def pair(precision):
    """Two particles apart by 0.6 h, moving apart."""
    sim = scene(3, [2, 1, 1], precision=precision)
    x = sim.fluid.to_numpy("pos")
    x[1] = x[0] + 0.012 * np.array([0.6, 0.64, 0.48], dtype=x.dtype)
    sim.fluid.from_numpy("pos", x)
    return sim


@pytest.mark.parametrize("precision", [4, 8])
def test_psi_of_an_infinite_neighbour(precision):
    from tichi_sph_amd import _lib
    sim = pair(precision)
    m, v = sim.fluid.to_numpy("mass"), sim.fluid.to_numpy("vel")
    m[1] = np.inf
    v[0] = [0.6, 0.64, 0.48]  # towards the other one
    sim.fluid.from_numpy("mass", m)
    sim.fluid.from_numpy("vel", v)
    sim._sort_bound()
    P, (ws, wsb), st = ctypes.byref(sim.params), sim._ws(), sim.stream_ptr()
    f, b, c = ctypes.byref(sim.fluid.struct()), ctypes.byref(sim.bound.struct()), sim.ctrl_ptr()
    lib = sim.lib
    _lib.check(lib.tsph_sort_object(P, f, c, 0, ws, wsb, st), "sort")
    sim.fluid.adopt_swaps()
    f = ctypes.byref(sim.fluid.struct())
    _lib.check(lib.tsph_density_alpha(P, f, b, c, ws, wsb, st), "density_alpha")
    _lib.check(lib.tsph_solver_begin(P, c, 0, st), "solver_begin")
    _lib.check(lib.tsph_solver_psi(P, f, b, c, 0, ws, wsb, st), "solver_psi")
    assert sim.fluid.to_numpy("psi_adv")[0] == np.inf


@pytest.mark.parametrize("precision", [4, 8])
def test_gradient_of_an_infinite_neighbour(precision):
    from tichi_sph_amd.adjoint import DiffRunner, rollout
    sim = pair(precision)
    dt = sim.fluid.dtype
    away = torch.tensor([[-0.6, -0.64, -0.48], [0.6, 0.64, 0.48]], dtype=dt, device="cuda", requires_grad=True)
    x, v = rollout(DiffRunner(sim), away, 0.05, 0.0, 1)
    weight = torch.ones_like(v)
    weight[1, 0] = np.inf
    torch.autograd.backward((x, v), (torch.zeros_like(x), weight))
    assert torch.isinf(away.grad[0]).all(), away.grad
