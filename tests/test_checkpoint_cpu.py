"""CPU test of DiffRunner.checkpoint and restore on a host-only Simulation:
they only copy the scene's state, which needs no GPU (every compute call
refuses)."""
import numpy as np
import pytest
import torch

from conftest import load_scene


@pytest.mark.parametrize("precision", [4, 8])
def test_checkpoint_and_restore_host_only(precision):
    from tichi_sph_amd import _lib, simulation_from_dicts
    from tichi_sph_amd.adjoint import DiffRunner
    sim = simulation_from_dicts(*load_scene("dambreak_2d_8k"), device="cpu", precision=precision, cfl=False)
    r = DiffRunner(sim)
    names = ("pos", "vel", "mass", "rest_density", "rest_volume", "volume_frac")
    before = {name: sim.fluid.to_numpy(name).copy() for name in names}
    r.step_index = 3
    st = r.checkpoint()
    ctrl = sim.ctrl.clone()
    for name in names:
        sim.fluid.from_numpy(name, before[name] + 1)
    sim.set_dt(0.5)
    r.step_index = 7
    assert not np.array_equal(sim.fluid.to_numpy("pos"), before["pos"])  # the checkpoint holds copies
    r.restore(st)
    for name in names:
        assert np.array_equal(sim.fluid.to_numpy(name), before[name]), name
    assert torch.equal(sim.ctrl, ctrl) and r.step_index == 3
    with pytest.raises(_lib.TsphError, match="host-only"):
        r.step()
