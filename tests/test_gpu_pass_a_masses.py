"""GPU test of pass A around particles without mass or of infinite mass: a
particle at one position with another, or with itself, adds no term to alpha_2
(sph.py:95 asks for r > 0), so alpha_2 is a number where no such particle lies at
a distance, and a quad of lanes per particle (a small scene's own step) gives it
bit for bit as one lane does (a grouped step)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [4, 8])
@pytest.mark.parametrize("solver,mass", [("VFSPH", 0.0), ("VFSPH", np.nan), ("DFSPH", np.inf)])
def test_alpha_2_of_coincident_particles(solver, mass, precision):
    from tichi_sph_amd import simulation_from_dicts
    from tichi_sph_amd.batch import SceneBatch
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(0.01, [20, 9, 9], 2, [([2, 3, 3], [2, 1, 1], [1]), ([9, 3, 3], [3, 2, 1], [1])], [1000],
               [0, -9.81, 0], 0.01)
    sims = [simulation_from_dicts(solver_config(solver, cs=100), scn, precision=precision, cfl=False)
            for _ in range(2)]
    for sim in sims:
        x, m = sim.fluid.to_numpy("pos"), sim.fluid.to_numpy("mass")
        x[1] = x[0]   # two at one position, no other near
        m[:2] = mass
        sim.fluid.from_numpy("pos", x)
        sim.fluid.from_numpy("mass", m)
    batch = SceneBatch([sims[1]])
    sims[0].sph_step()
    batch.step()
    a2 = [sim.fluid.to_numpy("alpha_2") for sim in sims]
    assert np.array_equal(a2[0], a2[1], equal_nan=True)
    assert np.isfinite(a2[0]).all() and (a2[0][:2] == 0).all() and (a2[0][2:] > 0).all()
