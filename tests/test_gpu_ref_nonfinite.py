"""GPU test of the sph.py kernels on fields that hold infinities, NaN, zeros to
divide by, and values whose products leave the type: bit for bit the oracle's
results, NaN for NaN.  The reference adds every candidate of the neighbouring
cells, also beyond h, where the kernel is zero: an infinity there makes the sum
a NaN (0 * inf), which no sum over the pairs in range alone would show."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

GRID = [("clear_node", 0), ("encode", 0), ("encode", 1), ("mem_shift", 0), ("fill_node", 0), ("fill_node", 1)]
IN = ("vel", "vel_adv", "mass", "rest_volume", "rest_density", "sph_density", "sph_compression", "alpha", "psi_adv",
      "pressure", "volume_frac")
ACC = ("W", "sph_density", "sph_compression", "alpha_1", "alpha_2", "acce_adv", "psi_adv", "vel_adv", "volume_frac_tmp")
OUT = ACC + ("normal", "drift_vel")
PAIR = ["SPH_prepare_attr", "SPH_prepare_alpha_1", "SPH_prepare_alpha_2", "SPH_advection_viscosity_acc",
        "SPH_advection_surface_tension_acc", "WC_pressure_acce", "IPPE_adv_psi", "IPPE_update_vel_adv",
        "SPH_FBM_diffuse", "SPH_FBM_convect"]
BAD = [("vel", np.nan), ("vel", np.inf), ("vel_adv", -np.inf), ("vel_adv", np.nan), ("mass", np.inf), ("mass", 0.0),
       ("rest_volume", np.nan), ("rest_volume", np.inf), ("sph_density", 0.0), ("sph_compression", 0.0),
       ("sph_density", -1.0), ("alpha", 0.0), ("alpha", np.nan), ("psi_adv", np.inf), ("pressure", np.inf),
       ("volume_frac", np.nan), ("rest_density", 0.0), ("mass", 3e38), ("psi_adv", 3e38)]


def build(dim, precision, solver, gamma):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    block = [6, 5, 5] if dim == 3 else [13, 9]
    scn = tank(0.01, [b + 2 for b in block], 2, [([0] * dim, block, [0.995, 0.005])], [1000, 500],
               [0, -9.81, 0][:dim], 0.01)
    cfg = solver_config(solver, cs=100, fbm_d=1e-4, gamma=gamma)
    o = O.Oracle(cfg, scn, precision)
    o.init_scenario()
    return simulation_from_dicts(cfg, scn, precision=precision, fbm=True), o


@pytest.mark.parametrize("dim,precision,solver,gamma", [
    (3, 4, "DFSPH", 0.07), (3, 4, "VFSPH", 0.0), (2, 4, "DFSPH", 0.0), (3, 8, "VFSPH", 0.07)])
def test_nonfinite_fields_spread_as_in_the_oracle(dim, precision, solver, gamma):
    from tichi_sph_amd import sph as K
    sim, o = build(dim, precision, solver, gamma)
    print(f"[case] {dim}D {solver} precision {precision} gamma {gamma}", flush=True)
    objs, ng = (sim.fluid, sim.bound), sim.ngrid
    rng = np.random.default_rng(5)
    x = objs[0].to_numpy("pos")
    x = (x + rng.uniform(-0.2, 0.2, x.shape) * sim.config.part_size[1]).astype(objs[0].np_dtype)
    objs[0].from_numpy("pos", x)
    o.set(0, "pos", x)
    for name, arg in GRID:
        o.kernel(name, arg)
    ng.clear_node()
    for ob in objs:
        ng.encode(ob)
    ng.mem_shift()
    for ob in objs:
        ng.fill_node(ob)

    base = {}
    for k, ob in enumerate(objs):
        for f in IN + ACC:
            shape = o.get(k, f).shape
            lo, hi = (-1, 1) if f in ("vel", "vel_adv", "acce_adv", "alpha_1") else \
                (0.991, 1) if f == "volume_frac" else (0.5, 2)
            base[k, f] = rng.uniform(lo, hi, shape).astype(ob.np_dtype)

    def put(k, f, a):
        objs[k].from_numpy(f, a.reshape(objs[k].to_numpy(f).shape))
        o.set(k, f, a)

    sim.set_dt(1e-3)
    o.scalar("dt", value=1e-3)
    spread = 0
    for f, v in [(None, None)] + BAD:
        for k, ob in enumerate(objs):
            for name in IN + ACC:
                put(k, name, base[k, name])
        for k in (0, 1):
            if f is None:
                continue
            a = base[k, f].copy()
            rows = rng.choice(len(a), 2, replace=False)
            a[rows] = v
            put(k, f, a)
        state = {(k, name): o.get(k, name).copy() for k in (0, 1) for name in IN + ACC}
        for name in PAIR:
            for nk in (0, 1):
                for (k, g), a in state.items():
                    put(k, g, a)
                getattr(K, name)(ng, objs[0], objs[nk])
                o.kernel(name, 0, nk)
                for g in OUT:
                    got, want = objs[0].to_numpy(g), o.get(0, g)
                    assert np.array_equal(got, want.reshape(got.shape), equal_nan=True), (f, v, name, nk, g)
                    spread += int(np.isnan(want).sum())
    assert spread > 0
