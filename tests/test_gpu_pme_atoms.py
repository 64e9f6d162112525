"""Where the PME spread finds its atoms, and the slab pipeline's tile shapes.

A plane (or a slab of one) scans the slots of the cells its support can come
from, given that no atom has moved further than half the skin since the list's
rebuild. The charges are summed in integers, so a run whose planes go by cells
is bit for bit the run whose planes scan every atom, whatever has moved since
the rebuild; an atom missed or taken twice would show in every position."""
import numpy as np
import pytest

import oracle as O
import rainmd_amd as R
from helpers import fixture_system, rel, rel_rms

pytestmark = pytest.mark.gpu

FORCE_BAR = 1e-4


def _moving(shape, **options):
    if shape == "octahedron":
        system, _ = fixture_system("ala-oct", dict(cutoff=0.6))
    else:
        waters, edge = shape
        system = R.System.solvated(waters, edge, 21, cutoff=0.6)
    sim = R.GpuSimulation(system, seed=4, temperature=600.0, **options)
    sim.minimise(max_iterations=100, force_tolerance=2000.0)
    sim.set_state(sim.read_positions().astype(np.float64), R.maxwell_boltzmann(system, 600.0, 8))
    return system, sim


@pytest.mark.parametrize("shape,options", [
    ((1500, 3.56), {}),                              # rectangular, several cells per axis
    ((1500, 3.56), dict(grid=[45, 28, 21], skin=0.5)),   # uneven grid, wide margin
    ((1500, 3.56), dict(grid=[5, 32, 20], cell_reach=1)),  # the support covers the axis
    ("octahedron", {}),                              # sheared
    ("octahedron", dict(grid=[35, 20, 27], skin=0.3)),
])
def test_planes_by_cells_run_as_planes_that_scan(shape, options):
    states = {}
    for mode in ("auto", "planes-scan"):
        _, sim = _moving(shape, pme_bins=1, **options)
        sim.set_pme_pipeline(mode)
        sim.run(60, 20)
        d = sim.diagnostics()
        states[mode] = sim.read_state()
        print(shape, options, mode, "cells", d["cell_counts"], "rebuilds", d["rebuilds"], flush=True)
        sim.release()
    for name in ("positions", "velocities", "forces"):
        assert np.array_equal(states["auto"][name], states["planes-scan"][name]), name


@pytest.mark.parametrize("shape,options", [
    ((1500, 3.56), dict(grid=[36, 35, 32])),   # a last slab of three rows
    ("octahedron", dict(grid=[28, 27, 25])),   # one partial slab, odd sizes
])
def test_slabs_follow_planes(shape, options):
    states = {}
    for mode in ("lines", "planes-scan"):
        _, sim = _moving(shape, **options)
        sim.set_pme_pipeline(mode)
        sim.run(20, 20)
        states[mode] = sim.read_state()
        sim.release()
    # FP32 rounding of the transforms (about 5e-7 of the reciprocal force),
    # grown over 20 steps; one missing atom is above 1e-3
    worst = rel_rms(states["lines"]["velocities"], states["planes-scan"]["velocities"])
    print(shape, options, "velocities", worst)
    assert worst < 2e-5


GRIDS = [(6, 5, 7), (300, 21, 25), (20, 600, 14), (14, 20, 768), (18, 36, 200), (21, 64, 180), (700, 16, 20)]


@pytest.mark.parametrize("grid", GRIDS)
def test_slab_transform_matches_numpy(grid):
    """Every tile width (16, 8 and 4 lines) on every axis, with partial tiles."""
    system = R.System.solvated(389, 2.2816, 101)
    sim = R.GpuSimulation(system, grid=list(grid))
    sim.set_pme_pipeline("lines")
    rng = np.random.default_rng(1)
    real = rng.uniform(-1, 1, size=grid).astype(np.float32)
    got = sim.debug_fft_forward(real)
    want = np.conj(np.fft.rfftn(real.astype(np.float64)))
    err = np.abs(got - want).max() / np.abs(want).max()
    print(grid, err)
    sim.release()
    assert err < 20 * np.sqrt(3 * np.log2(max(grid))) * 2.0 ** -24  # FP32 butterflies, three axes


@pytest.mark.parametrize("grid", [(24, 300, 25), (27, 20, 768), (30, 35, 200)])
def test_slab_forces_match_the_oracle(grid):
    system = R.System.solvated(389, 2.2816, 101)
    sim = R.GpuSimulation(system, grid=list(grid))
    sim.set_pme_pipeline("lines")
    gpu, forces = sim.evaluate(terms=R._lib.TERM_RECIPROCAL)
    ref, ref_forces = O.Oracle(system).potential(sim.read_positions().astype(np.float64),
                                                 alpha=sim.diagnostics()["pme_alpha"], grid=list(grid), terms=8)
    d = rel_rms(forces, ref_forces)
    print(grid, gpu["coulomb_reciprocal"], ref["reciprocal"], "forces", d)
    sim.release()
    assert rel(gpu["coulomb_reciprocal"], ref["reciprocal"]) < 1e-6
    assert d < FORCE_BAR


def test_planes_by_cells_through_volume_moves():
    """A volume move keeps the cell list and may plan other cell counts before
    it is rebuilt: the planes go by the counts it was built with. (4.73 nm at
    a 0.9 nm cutoff: the moves cross from one count per axis to the next.)"""
    edge, waters, seed = next((e, w, s) for e, w, s in R.replica_workload(32) if w > 3500)
    system = R.System.solvated(waters, edge, seed, cutoff=0.9)
    start = R.GpuSimulation(system, temperature=300.0, seed=seed)
    start.minimise(max_iterations=60, force_tolerance=1000.0)
    x = start.read_positions().astype(np.float64)
    start.release()
    states = {}
    for mode in ("auto", "planes-scan"):
        sim = R.GpuSimulation(system, temperature=300.0, seed=seed, pressure=1.0, barostat_interval=5, pme_bins=1)
        sim.set_pme_pipeline(mode)
        sim.set_state(x, R.maxwell_boltzmann(system, 300.0, seed))
        counts = set()
        for _ in range(12):
            sim.run(10, 5)
            counts.add(tuple(sim.diagnostics()["cell_counts"]))
        d = sim.diagnostics()
        states[mode] = sim.read_state()
        print(mode, "cells", counts, "moves", d["barostat_attempts"], "rebuilds", d["rebuilds"], flush=True)
        sim.release()
    for name in ("positions", "velocities", "forces"):
        assert np.array_equal(states["auto"][name], states["planes-scan"][name]), name
