"""GPU test of the cell tables at the edges of the scan: a table of up to 32
tiles of 4,096 counts is scanned by one launch in which every block adds up the
tiles before its own, a longer one by two launches.  Grids just below, at and
above a tile, and on both sides of 32 tiles: cell_start is the exclusive prefix
of cell_count (whole numbers, exact) with and without the time step's
reduction, and the time step is the one of the fastest particle (one FP32
rounding of a square root and a quotient)."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# inner size of a 2D tank in particles -> tiles of its cell table (+ invalid bucket)
GRIDS = [(10, 10, 1), (115, 111, 1), (118, 118, 2), (713, 713, 32), (713, 715, 33)]


@pytest.mark.parametrize("w,h,tiles", GRIDS)
@pytest.mark.parametrize("cfl", [0, 1])
def test_cell_tables_at_scan_edges(w, h, tiles, cfl):
    from tichi_sph_amd import _lib, simulation_from_dicts
    from tichi_sph_amd.scenarios.make_scenarios import solver_config, tank
    scn = tank(0.02, [w, h], 3, [([0, 0], [9, 7], [1])], [1000], [0, -9.81], 0.01)
    sim = simulation_from_dicts(solver_config("DFSPH", cs=50), scn)
    n = sim.fluid.part_num
    length = sim.params.node_num + 1
    print(f"[case] {w}x{h}: {length} counts, cfl {cfl}", flush=True)
    assert -(-length // 4096) == tiles
    vel = np.random.default_rng(w).normal(0, 30.0, (n, 2)).astype(np.float32)
    sim.fluid.from_numpy("vel", vel)
    ws, wsb = sim._ws()
    for obj, c in ((sim.bound, 0), (sim.fluid, cfl)):
        rc = sim.lib.tsph_sort_object(ctypes.byref(sim.params), ctypes.byref(obj.struct()), sim.ctrl_ptr(), c, ws,
                                      wsb, sim.stream_ptr())
        _lib.check(rc, "sort")
        obj.adopt_swaps()
        start = obj.t["cell_start"].cpu().numpy()[:length + 1]
        cell = obj.t["cell"][:obj.part_num].cpu().numpy()
        count = np.bincount(cell, minlength=length)
        assert np.array_equal(start, np.concatenate([[0], np.cumsum(count)]))
    if cfl:
        speed = np.sqrt((vel.astype(np.float64) ** 2).sum(1)).max()
        want = min(sim.params.part_size[1] / sim.params.cs, sim.params.cfl_factor * sim.params.part_size[1] / speed)
        assert abs(sim.control().dt - want) <= 4 * 2.0 ** -24 * want
