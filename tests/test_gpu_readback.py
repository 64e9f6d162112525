"""Read-backs of positions, velocities and forces: packed by the device into
pinned host memory, one stage for every read."""
import numpy as np
import pytest

import rainmd_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters,edge,solute", [(389, 2.2816, True), (2048, 3.95, False), (8000, 6.21, True)])
def test_read_back_is_the_state(waters, edge, solute):
    """3N ends inside a workgroup, at its edge (6144 atoms: 72 x 256 numbers)
    and past the size a pageable copy is staged at; every read in turn, the
    wider after the narrower."""
    system = R.System.solvated(waters, edge, 11, include_solute=solute)
    n3 = 3 * system.atom_count
    print("atoms", system.atom_count, flush=True)
    sim = R.GpuSimulation(system, seed=3)
    rng = np.random.default_rng(5)
    x = system.positions.astype(np.float32)
    v = rng.normal(size=n3).astype(np.float32)
    sim.set_state(x.astype(np.float64), v.astype(np.float64))
    assert np.array_equal(sim.read_positions(), x)
    _, f64 = sim.evaluate(energies=False)
    state = sim.read_state()
    assert np.array_equal(state["positions"], x)
    assert np.array_equal(state["velocities"], v)
    assert np.any(f64)
    # the fixed-point sum scaled once, then rounded once
    assert np.array_equal(state["forces"], f64.reshape(-1).astype(np.float32))
    assert np.array_equal(f64 * 2.0 ** 32, np.rint(f64 * 2.0 ** 32))
    assert np.array_equal(sim.read_positions(), x)
    sim.release()
