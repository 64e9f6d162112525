"""The by-cell list search with several waves sharing a cell's atoms."""
import numpy as np
import pytest

import oracle as O
import rainmd_amd as R
from helpers import fixture_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,cutoff,skin", [
    ((700, 2.76), 0.6, 0.1),     # 11 cells per axis: six waves, fewer atoms in some cells than waves
    ((3000, 4.48), 0.6, 0.3),
    ((3000, 4.48), 1.1, 0.4),    # crowded cells: eight waves of three and more atoms
    ("octahedron", 0.6, 0.15),   # sheared
])
def test_lists_of_shared_cells(shape, cutoff, skin):
    """The lists equal those of one wave per atom entry for entry, and as
    sets the FP32 emulation's pairs."""
    if shape == "octahedron":
        system, _ = fixture_system("ala-oct", dict(cutoff=cutoff))
    else:
        system = R.System.solvated(*shape, 31, cutoff=cutoff)
    lists = {}
    for mode in (1, 2):
        sim = R.GpuSimulation(system, skin=skin, search_mode=mode, cell_reach=3)
        sim.evaluate()
        d = sim.diagnostics()
        lists[mode] = sim.read_neighbours()
        pos = sim.read_positions()
        print(shape, cutoff, "mode", mode, "by cell", d["search_by_cell"], "cells", d["cell_counts"], flush=True)
        sim.release()
        assert d["search_by_cell"] == (mode == 2)
    assert np.array_equal(lists[1][0], lists[2][0])
    assert np.array_equal(lists[1][1], lists[2][1])
    counts, entries = lists[2]
    ref_counts, ref = O.pairs_f32(pos, system.box, system.cutoff + d["skin"], system.exclusion_start,
                                  system.exclusion_partners)
    assert np.array_equal(counts, ref_counts)
    for i in range(system.atom_count):
        assert np.array_equal(np.sort(entries[i, :counts[i]]), ref[i, :ref_counts[i]]), i
