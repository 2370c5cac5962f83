"""GPU test of the sph.py kernels on an Ngrid whose cells' ranges lie in
arbitrary order, as the reference's mem_shift (sph_obj.py:308-314) leaves them
under several threads: every kernel gives bit for bit what it gives on the same
cells in ascending order, for a grid that is out of order everywhere and one
that is in its upper half only (a walk then meets both kinds of row)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

PAIR = ["SPH_prepare_attr", "SPH_prepare_alpha_1", "SPH_prepare_alpha_2", "SPH_advection_viscosity_acc",
        "SPH_advection_surface_tension_acc", "WC_pressure_acce", "IPPE_adv_psi", "IPPE_update_vel_adv",
        "SPH_FBM_diffuse", "SPH_FBM_convect"]
OUT = ("W", "sph_compression", "sph_density", "alpha_1", "alpha_2", "acce_adv", "acce", "normal", "psi_adv",
       "vel_adv", "volume_frac_tmp", "drift_vel", "fbm_zeta")


def scene(dim, rng_cells):
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    block = [9, 8, 7] if dim == 3 else [24, 17]
    scn = tank(0.01, [b + 3 for b in block], 2, [([0] * dim, block, [0.7, 0.3])], [1000, 500],
               [0, -9.81, 0][:dim], 0.01)
    cfg = solver_config("VFSPH", cs=100, fbm_d=1e-4, gamma=0.07)
    if rng_cells == 2:  # cells of one particle size, two to each side
        cfg["solver_neighb_range"] = 2
        cfg["solver_neighb_grid_size_TO_global_part_size"] = 1
    return cfg, scn


def fill(obj, rng):
    """Values of every field that a pair kernel reads."""
    n = obj.part_num

    def put(name, lo, hi):
        t = obj.t[name][:n]
        t.copy_(torch.as_tensor(rng.uniform(lo, hi, tuple(t.shape)), dtype=t.dtype))

    for name in ("vel", "vel_adv", "acce_adv", "normal", "alpha_1"):
        put(name, -1, 1)
    for name in ("mass", "rest_volume", "sph_density", "sph_compression", "alpha", "psi_adv", "pressure", "W", "alpha_2"):
        put(name, 0.5, 2)
    put("volume_frac", 0.991, 1.0)


def scramble(ngrid, first, rng):
    """Moves the ranges of the cells from `first` on into random order."""
    cnt, start = ngrid.node_part_count.cpu().numpy(), ngrid.node_part_shift.cpu().numpy()
    pin, uin = ngrid.part_pid_in_node.cpu().numpy(), ngrid.part_uid_in_node.cpu().numpy()
    order = np.concatenate([np.arange(first), first + rng.permutation(len(cnt) - first)])
    new = np.zeros_like(start)
    new[order] = np.concatenate([[0], np.cumsum(cnt[order])[:-1]])
    p2, u2 = pin.copy(), uin.copy()
    for c in np.nonzero(cnt)[0]:
        p2[new[c]:new[c] + cnt[c]] = pin[start[c]:start[c] + cnt[c]]
        u2[new[c]:new[c] + cnt[c]] = uin[start[c]:start[c] + cnt[c]]
    for t, a in ((ngrid.node_part_shift, new), (ngrid.part_pid_in_node, p2), (ngrid.part_uid_in_node, u2)):
        t.copy_(torch.as_tensor(a))
    return bool((np.diff(new[cnt > 0]) < 0).any())


@pytest.mark.parametrize("half", [False, True], ids=["all", "half"])
@pytest.mark.parametrize("dim,reach,precision", [(2, 1, 4), (3, 1, 4), (3, 1, 8), (3, 2, 4)])
def test_kernels_do_not_need_cells_in_order(dim, reach, precision, half):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd import sph as K
    cfg, scn = scene(dim, reach)
    print(f"[case] {dim}D, range {reach}, precision {precision}, half {half}", flush=True)
    sim = simulation_from_dicts(cfg, scn, precision=precision, fbm=True)
    rng = np.random.default_rng(11)
    fl, bd, ng = sim.fluid, sim.bound, sim.ngrid
    x = fl.to_numpy("pos")
    fl.from_numpy("pos", x + rng.uniform(-0.2, 0.2, x.shape) * sim.config.part_size[1])
    ng.clear_node()
    for o in (fl, bd):
        ng.encode(o)
    ng.mem_shift()
    for o in (fl, bd):
        ng.fill_node(o)
        fill(o, rng)
    start = {(o, name): o.t[name].clone() for o in (fl, bd) for name in OUT}

    def run(name, obj, nobj):
        for (o, f), t in start.items():
            o.t[f].copy_(t)
        getattr(K, name)(ng, obj, nobj)
        return {f: obj.t[f].cpu().numpy() for f in OUT}

    calls = [(name, fl, nobj) for name in PAIR for nobj in (fl, bd)] + [("SPH_prepare_attr", bd, fl)]
    want = [run(*c) for c in calls]
    assert scramble(ng, sim.params.node_num // 2 if half else 0, rng)
    for c, w in zip(calls, want):
        got = run(*c)
        for f in OUT:
            assert np.array_equal(got[f], w[f], equal_nan=True), (c[0], c[2].uid, f)
    assert any(not np.array_equal(w["W"], start[(fl, "W")].cpu().numpy()) for w in want)
