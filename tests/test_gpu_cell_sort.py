"""The cell list of a system too large for one workgroup: each cell's atoms
once, in index order, from few crowded cells to many short ones."""
import numpy as np
import pytest

import rainmd_amd as R

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("options", [
    dict(cutoff=2.5, cell_reach=1),   # 8 cells of about 2050 atoms
    dict(cutoff=1.2, cell_reach=1),   # 27 of about 600
    dict(cutoff=0.9, cell_reach=2),   # 512 of about 32
    dict(cutoff=0.6, cell_reach=3),   # 4096 of about 4, some empty
])
def test_cells_in_index_order(options):
    options = dict(options)
    system = R.System.solvated(5457, 5.48, 21, cutoff=options.pop("cutoff"))  # 16,393 atoms: a last workgroup of 9
    sim = R.GpuSimulation(system, seed=4, **options)
    sim.evaluate(terms=R._lib.TERM_DIRECT, forces=False)
    cell_of, start, atoms = sim.read_cells()
    n, length = sim.atom_count, np.diff(start)
    print(options, "atoms", n, "cells", length.size, "longest", length.max())
    assert start[0] == 0 and start[-1] == n
    assert np.array_equal(np.bincount(cell_of, minlength=length.size), length)
    assert np.array_equal(atoms, np.lexsort((np.arange(n), cell_of)))
    sim.release()
