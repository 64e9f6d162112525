"""Direct space, bonded terms and PME planes that go by cells, in one launch:
bit for bit the run and the energies of the separate launches."""
import numpy as np
import pytest

import rainmd_amd as R
from helpers import fixture_system

pytestmark = pytest.mark.gpu


# 70 is the largest square plane that leaves the joined launch within 64 KB of
# LDS (an even K: (2 K + K (K / 2 + 1) + K^2) 8 + 4096 bytes), 72 the first past it
@pytest.mark.parametrize("shape,options", [
    ((1500, 3.56), {}),
    ((1500, 3.56), dict(lanes_per_atom=64, search_mode=2)),   # more than one pass: apart on both sides
    ((1500, 3.56), dict(grid=[45, 70, 70], barostat_interval=10, pressure=1.0)),
    ((1500, 3.56), dict(grid=[45, 72, 72])),
    ("octahedron", dict(grid=[5, 27, 25], lanes_per_atom=32)),  # the support covers the axis
])
def test_joined_run_is_the_separate_launches(shape, options):
    if shape == "octahedron":
        system, _ = fixture_system("ala-oct", dict(cutoff=0.6))
    else:
        system = R.System.solvated(shape[0], shape[1], 21, cutoff=0.6)
    out = []
    for joined in (True, False):
        sim = R.GpuSimulation(system, seed=4, temperature=600.0, pme_bins=1, **options)
        sim.set_concurrent_forces(joined)
        sim.minimise(max_iterations=60, force_tolerance=2000.0)
        sim.set_state(sim.read_positions().astype(np.float64), R.maxwell_boltzmann(system, 600.0, 8))
        sim.run(40, 20)
        energies, _ = sim.evaluate()
        out.append((sim.read_state(), energies, sim.diagnostics()["rebuilds"]))
        sim.release()
    (a, ea, ra), (b, eb, rb) = out
    print(shape, options, "rebuilds", ra, rb, ea["potential"], eb["potential"], flush=True)
    assert ra == rb
    for name in ("positions", "velocities", "forces"):
        assert np.array_equal(a[name], b[name]), name
    assert ea == eb
