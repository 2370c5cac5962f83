"""tsph_step: its argument checks and struct layout (CPU), and the step it
drives against the same step issued call by call (GPU): a Simulation with a
timer issues the calls from Python, one without runs tsph_step, and both take
the same iterations and rounds to the same state, bit for bit."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

from conftest import ROOT, load_scene


def test_step_struct_layout_matches_header(tmp_path):
    from tichi_sph_amd import _lib
    fields = [n for n, _ in _lib.TsphStep._fields_]
    src = ["#include <stdio.h>", "#include <stddef.h>", f'#include "{os.path.join(ROOT, "include", "tichi_sph.h")}"',
           'int main(void){printf("%zu", sizeof(TsphStep));']
    src += [f'printf(" %zu", offsetof(TsphStep, {f}));' for f in fields] + ["return 0;}"]
    c = tmp_path / "layout.c"
    c.write_text("\n".join(src))
    subprocess.check_call(["gcc", "-std=c11", str(c), "-o", str(tmp_path / "layout")])
    got = [int(v) for v in subprocess.check_output([str(tmp_path / "layout")]).split()]
    assert got == [ctypes.sizeof(_lib.TsphStep)] + [getattr(_lib.TsphStep, f).offset for f in fields]


def test_step_without_a_signal_is_refused():
    from tichi_sph_amd import _lib, simulation_from_dicts
    cb, sb = load_scene("dambreak_2d_8k")
    sim = simulation_from_dicts(cb, sb, device="cpu")
    step = _lib.TsphStep()
    for arg in (None, ctypes.byref(step)):
        rc = sim.lib.tsph_step(ctypes.byref(sim.params), ctypes.byref(sim.fluid.struct()),
                               ctypes.byref(sim.bound.struct()), None, arg, None, 0, None)
        assert rc == -1 and b"null step or signal" in sim.lib.tsph_last_error()
    with pytest.raises(_lib.TsphError, match="host-only"):
        sim.sph_step()


@pytest.mark.gpu
@pytest.mark.parametrize("name,kw,edit", [
    ("dambreak_2d_8k", {}, {}),
    ("dambreak_3d_8k", {"cfl": False, "precision": 8}, {}),
    ("dambreak_3d_8k", {"wcsph": True}, {}),
    ("two_phase_3d_4k", {"fbm": True}, {}),
    # an unreachable threshold: every solve runs past its prediction to its cap
    ("dambreak_2d_8k", {}, {"solver_compression_threshold": 0.0, "solver_divergence_threshold": 0.0,
                            "solver_iter_threshold_max": 7}),
    # only the density solve runs past its prediction: the tail is launched again
    ("dambreak_3d_8k", {}, {"solver_compression_threshold": 0.0, "solver_iter_threshold_max": 7}),
    # the same under an FBM round and a tail launched ahead
    ("two_phase_3d_4k", {"fbm": True}, {"solver_compression_threshold": 0.0, "solver_iter_threshold_max": 7}),
    # no iteration at all: the solves signal from their begin
    ("dambreak_3d_8k", {}, {"solver_iter_threshold_min": 0}),
], ids=["2d", "3d_f64", "wcsph", "fbm", "cap", "late", "late_fbm", "none"])
def test_native_step_is_the_call_by_call_step(name, kw, edit):
    from tichi_sph_amd import EventTimer, simulation_from_dicts
    cb, sb = load_scene(name)
    cb.update(edit)
    a, b = (simulation_from_dicts(cb, sb, **kw) for _ in range(2))
    v = np.random.default_rng(3).normal(0, 0.2, a.fluid.to_numpy("vel").shape).astype(a.fluid.np_dtype)
    for sim in (a, b):
        sim.fluid.from_numpy("vel", v)
    b.timer = EventTimer()
    for step in range(4):
        sa, sb_ = a.sph_step(stats=True), b.sph_step(stats=True)
        assert (sa.div_iter, sa.incom_iter, sa.fbm_rounds) == (sb_.div_iter, sb_.incom_iter, sb_.fbm_rounds), step
        assert (sa.dt, sa.compression, sa.kinetic_energy) == (sb_.dt, sb_.compression, sb_.kinetic_energy)
        assert a.pred == b.pred
        assert a._step.fbm_rounds == sa.fbm_rounds
        for f in ("pos", "vel", "vel_adv", "mass", "volume_frac", "sph_density", "neighb_cell_seq"):
            assert np.array_equal(a.fluid.to_numpy(f), b.fluid.to_numpy(f)), (step, f)
