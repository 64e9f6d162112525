"""What the minimiser hands back: the energy and largest force of the point it
ends at, its constraints, and the base point again where every trial fails."""
import numpy as np
import pytest

import rainmd_amd as R

from helpers import ALPHA_24, fixture_system

pytestmark = pytest.mark.gpu


def _sim(constraints):
    system, _ = fixture_system("ala-wat", dict(constraints=constraints, rigid_water=constraints != "none", cutoff=1.0))
    sim = R.GpuSimulation(system, alpha=ALPHA_24, grid=[24, 24, 24], seed=3)
    sim.set_state(sim.read_positions().astype(np.float64), R.maxwell_boltzmann(system, 300.0, 3))
    return system, sim


# no clusters, water triangles with stars, and clusters that are no stars
@pytest.mark.parametrize("constraints", ["none", "HBonds", "AllBonds"])
def test_end_point(constraints):
    system, sim = _sim(constraints)
    result = sim.minimise(max_iterations=25, force_tolerance=10.0)
    state = sim.read_state()
    energies, forces = sim.evaluate()
    print(constraints, result, energies["potential"])
    assert not result["converged"]
    # the same sums, in the order of the list's rows
    assert abs(energies["potential"] - result["potential"]) <= 1e-12 * abs(energies["potential"])
    norms = np.linalg.norm(np.asarray(forces, dtype=np.float64).reshape(-1, 3), axis=1)
    assert abs(result["max_force"] - norms.max()) <= 1e-6 * norms.max()  # one rounding to FP32 on each side
    assert not state["velocities"].any()
    p = state["positions"].reshape(-1, 3).astype(np.float64)
    d = np.linalg.norm(p[system.constraint_a] - p[system.constraint_b], axis=1)
    if d.size:
        assert np.max(np.abs(d / system.constraint_distance - 1.0)) < 1e-5


@pytest.mark.parametrize("constraints", ["none", "HBonds", "AllBonds"])
def test_stalled_minimisation_leaves_the_base_point(constraints):
    # every atom moves 0.1 nm along its force in each of the 14 trials, so all
    # raise the energy of a relaxed state
    _, sim = _sim(constraints)
    sim.minimise(max_iterations=10, force_tolerance=10.0)
    sim.evaluate()
    before = sim.read_state()
    result = sim.minimise(max_iterations=5, force_tolerance=10.0, max_step=1e7, max_displacement=0.1)
    after = sim.read_state()
    print(constraints, result)
    assert result["stalled"] and result["rejected"] == 14 and result["iterations"] == 1
    for name in ("positions", "forces"):
        assert np.array_equal(before[name], after[name]), name
