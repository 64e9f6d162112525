"""The neighbour list with and without its entries' types: the same LJ
parameters under more type indices than the direct space keeps in LDS."""
import os

import numpy as np
import pytest

import rainmd_amd as R

pytestmark = pytest.mark.gpu


def _sections(text):
    order, sections = [], {}
    for chunk in text.split("%FLAG ")[1:]:
        head, rest = chunk.split("\n", 1)
        name = head.strip()
        fmt, body = rest.split("\n", 1)
        order.append(name)
        sections[name] = [fmt, body]
    return text.split("%FLAG ")[0], order, sections


def _ints(body):
    return [int(x) for x in body.split()]


def _floats(body):
    lines = body.split("\n")
    return [float(line[k:k + 16]) for line in lines for k in range(0, len(line.rstrip()), 16)]


def _write(values, per, form):
    return "".join("".join(form % v for v in values[k:k + per]) + "\n" for k in range(0, len(values), per)) or "\n"


def _retyped(types):
    """ala-wat with its atoms dealt over `types` type indices, each a copy of
    the atom's own type."""
    with open(os.path.join(R.simulation.DATA, "ala-wat.prmtop")) as f:
        head, order, sections = _sections(f.read())
    pointers = _ints(sections["POINTERS"][1])
    old = _ints(sections["ATOM_TYPE_INDEX"][1])
    n_old = pointers[1]
    index = _ints(sections["NONBONDED_PARM_INDEX"][1])
    A, B = (_floats(sections["LENNARD_JONES_%sCOEF" % c][1]) for c in "AB")
    source = list(range(1, n_old + 1))  # new type -> old type
    copies = {t: [t] for t in source}
    rarest = sorted(source, key=lambda t: old.count(t))
    while len(source) < types:  # copies of the types that many atoms share
        t = rarest[-1 - (len(source) % 2)]
        source.append(t)
        copies[t].append(len(source))
    seen = dict.fromkeys(copies, 0)
    new = []
    for t in old:
        new.append(copies[t][seen[t] % len(copies[t])])
        seen[t] += 1
    pairs, a, b = [0] * (types * types), [], []
    for i in range(types):
        for j in range(i + 1):
            k = index[(source[i] - 1) * n_old + source[j] - 1]
            assert k > 0
            a.append(A[k - 1])
            b.append(B[k - 1])
            pairs[i * types + j] = pairs[j * types + i] = len(a)
    pointers[1] = types
    sections["POINTERS"][1] = _write(pointers, 10, "%8d")
    sections["ATOM_TYPE_INDEX"][1] = _write(new, 10, "%8d")
    sections["NONBONDED_PARM_INDEX"][1] = _write(pairs, 10, "%8d")
    sections["LENNARD_JONES_ACOEF"][1] = _write(a, 5, "%16.8E")
    sections["LENNARD_JONES_BCOEF"][1] = _write(b, 5, "%16.8E")
    return head + "".join("%%FLAG %s\n%s\n%s" % (name, *sections[name]) for name in order)


def _run(text, **options):
    system = R.System.build(R.Topology(text), R.Coordinates.load("ala-wat.inpcrd"), cutoff=0.9)
    sim = R.GpuSimulation(system, seed=5, **options)
    sim.minimise(max_iterations=40, force_tolerance=1000.0)
    sim.set_state(sim.read_positions().astype(np.float64), R.maxwell_boltzmann(system, 300.0, 5))
    sim.run(30, 10)
    energies, forces = sim.evaluate()
    out = system.type_count, sim.read_state(), energies["potential"], forces, sim.read_neighbours()
    sim.release()
    return out


@pytest.mark.parametrize("options", [{}, dict(search_mode=2, lanes_per_atom=16)])
@pytest.mark.parametrize("types", [90, 91, 130])
def test_types_beyond_the_lds_table(types, options):
    with open(os.path.join(R.simulation.DATA, "ala-wat.prmtop")) as f:
        few = _run(f.read(), **options)
    many = _run(_retyped(types), **options)
    print("types", few[0], many[0], "potential", few[2], many[2])
    assert many[0] == types
    for name in ("positions", "velocities", "forces"):
        assert np.array_equal(few[1][name], many[1][name]), name
    assert np.array_equal(few[3], many[3])
    # the dispersion tail sums over types in another order
    assert abs(few[2] - many[2]) <= 1e-12 * abs(few[2])
    for a, b in zip(few[4], many[4]):
        assert np.array_equal(a, b)
