"""A list whose rows have grown: the force bits do not depend on what the
engine held before, so a run restored into a new engine follows the saved
one bit for bit."""
import dataclasses

import numpy as np
import pytest

from mdir_amd import systems as S

pytestmark = pytest.mark.gpu


def slab(spacing):
    """4,000 atoms as a slab of nine layers in a 9.28 nm box: at 0.17 nm a
    group's row needs more entries than a box of this mean density is given,
    and the capacity is doubled; at 0.28 nm it is not."""
    k = np.arange(4000)
    x = np.stack([k % 21, k // 21 % 22, k // 462], 1) * spacing
    x += np.random.default_rng(4).uniform(-0.01, 0.01, x.shape)
    n = len(x)
    return S.System(positions=x + 0.5, masses=np.full(n, 40.0), charges=np.zeros(n),
                    types=np.zeros(n, np.int32), sigma=np.full((1, 1), 0.15),
                    epsilon=np.full((1, 1), 0.05), box=np.full(3, 9.28), cutoff=0.6)


def test_bits_do_not_depend_on_an_earlier_growth():
    from mdir_amd.simulation import Simulation
    print("case: 4,000 atoms, forces and a restored run after the rows grew", flush=True)
    s = slab(0.28)
    fresh = Simulation(s, skin=0.1)
    F, e = fresh.forces()
    grown = Simulation(slab(0.17), skin=0.1)
    grown.forces()
    assert grown.stats()["row_cap"] > fresh.stats()["row_cap"]
    grown.positions = s.positions
    F1, e1 = grown.forces()
    assert np.abs(F).max() > 0.1
    assert np.array_equal(F, F1) and np.array_equal(e, e1)
    assert grown.stats()["row_cap"] > fresh.stats()["row_cap"]

    grown.velocities = S.initial_velocities(s, 3, 50.0)
    grown.run(10, 0.002, graph=5)
    cont = Simulation.from_checkpoint(dataclasses.replace(s), grown.state(), skin=0.1)
    assert cont.stats()["row_cap"] < grown.stats()["row_cap"]
    for sim in (grown, cont):
        sim.run(20, 0.002, graph=10)
    assert np.array_equal(grown.positions, cont.positions)
    assert np.array_equal(grown.velocities, cont.velocities)
    for sim in (fresh, grown, cont):
        sim.close()
