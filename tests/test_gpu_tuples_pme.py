"""The bonded tuples as the first blocks of the PME bins (their words by
atom) and alone (by place): the same force words and energies, for every
order and brick shape of the bins."""
import numpy as np
import pytest

from mdir_amd import runtime as rt
from test_gpu_bonded import dipeptide

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bricks", [8, 4, 2, 1])
@pytest.mark.parametrize("order", [4, 6, 8])
def test_words_beside_pme_and_alone(order, bricks):
    """Sums of words: whole = (tuples alone) + (the rest), to the word."""
    import dataclasses
    from mdir_amd.simulation import Simulation
    print(f"case: dipeptide, order {order}, bricks of {bricks} lines", flush=True)
    s = dataclasses.replace(dipeptide(rigid_water=True, hydrogen_bonds=False, pme=True),
                            pme_order=order)
    sim = Simulation(s)
    sim.launch_shape = (16, bricks, 0)
    F, e = sim.forces()
    Ft, et = sim.force_terms(rt.TERM_BONDED)
    Fr, er = sim.force_terms(rt.TERM_PAIRS | rt.TERM_SPECIAL | rt.TERM_RECIP)
    assert np.abs(Ft).max() > 100.0
    assert np.array_equal(np.rint(F * 2.0 ** 32), np.rint(Ft * 2.0 ** 32) + np.rint(Fr * 2.0 ** 32))
    for k in ("bonds", "angles", "dihedrals"):
        i = rt.ENERGY_NAMES.index(k)
        assert et[i] != 0.0 and e[i] == et[i] and er[i] == 0.0
    # in a run: the tuples of every step, against the steps without graphs
    sim.run(6, 0.0005, graph=3)
    again = Simulation(s)
    again.launch_shape = (16, bricks, 0)
    again.run(6, 0.0005, graph=0)
    assert np.array_equal(sim.positions, again.positions)
    sim.close()
    again.close()
