"""GPU tests of tsph_step over more steps than a wrong guess holds back (16): the
iterations that the solves need rise and fall from step to step, so that kernels
launched ahead of a solve's end go, return, are launched again, and are launched
ahead anew with another guess, up to the cap on iterations.  A Simulation with a
timer issues the same calls one by one; both take the same iterations and rounds
to the same state, bit for bit."""
import numpy as np
import pytest

from conftest import load_scene

pytestmark = pytest.mark.gpu

STEPS = 44


def pair(name, **kw):
    from tichi_sph_amd import EventTimer, simulation_from_dicts
    cb, sb = load_scene(name)
    a, b = (simulation_from_dicts(cb, sb, **kw) for _ in range(2))
    v = np.random.default_rng(3).normal(0, 0.2, a.fluid.to_numpy("vel").shape).astype(a.fluid.np_dtype)
    for sim in (a, b):
        sim.fluid.from_numpy("vel", v)
    b.timer = EventTimer()
    return a, b


def limit(sim, iters, cap):
    """Solves that run `iters` iterations (0: as their thresholds have it), at
    most cap + 1."""
    p = sim.params
    p.iter_max = sim.config.iter_threshold_max = cap
    p.iter_min = iters[0] or sim.config.iter_threshold_min
    p.divergence_threshold = p.compression_threshold = 1e9 if iters[0] else 1e-3
    if iters[0] and iters[1] > iters[0]:  # the density solve goes on to the cap
        p.compression_threshold = 0.0


# per step: (iterations of the divergence solve, of the density solve), cap
RISE_FALL = [((2 + (t // 5) % 4, 0), 100) for t in range(STEPS)]
LATE_DENSITY = [((2, 6 if t % 19 < 2 else 0), 5) for t in range(STEPS)]
AT_CAP = [((6, 6), 5) for t in range(STEPS)]
FREE = [((0, 0), 100) for t in range(STEPS)]


@pytest.mark.parametrize("hold", [True, False], ids=["held", "always"])
@pytest.mark.parametrize("plan", [RISE_FALL, LATE_DENSITY, AT_CAP, FREE],
                         ids=["rise_fall", "late_density", "cap", "free"])
@pytest.mark.parametrize("name,kw", [("dambreak_3d_8k", {}), ("two_phase_3d_4k", {"fbm": True}),
                                     ("dambreak_2d_8k", {"wcsph": True})], ids=["3d", "fbm", "wcsph"])
def test_many_steps_are_the_call_by_call_steps(name, kw, plan, hold):
    a, b = pair(name, **kw)
    print(f"[case] {name}, hold {hold}", flush=True)
    held = ahead = 0
    for step, (iters, cap) in enumerate(plan):
        for sim in (a, b):
            limit(sim, iters, cap)
        if not hold:
            a._step.hold = 0  # every step launches ahead, also after a miss
        ahead += a._step.hold == 0
        sa, sb_ = a.sph_step(stats=True), b.sph_step(stats=True)
        held += a._step.hold == 16
        assert (sa.div_iter, sa.incom_iter, sa.fbm_rounds) == (sb_.div_iter, sb_.incom_iter, sb_.fbm_rounds), step
        assert (sa.dt, sa.compression, sa.kinetic_energy) == (sb_.dt, sb_.compression, sb_.kinetic_energy), step
        assert a.pred == b.pred and a._step.fbm_rounds == sa.fbm_rounds, step
        if iters[0]:
            assert sa.div_iter == iters[0] and sa.incom_iter == max(iters), step
        for f in ("pos", "vel", "vel_adv", "mass", "volume_frac", "sph_density", "neighb_cell_seq"):
            assert np.array_equal(a.fluid.to_numpy(f), b.fluid.to_numpy(f)), (step, f)
    assert ahead > (STEPS - 1 if not hold else 2)
    if plan is RISE_FALL:
        assert held >= 2  # a guess fell short, and again after its hold
