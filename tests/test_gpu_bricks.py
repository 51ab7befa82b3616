"""Spread and gather by bricks: edges that are no multiple of a brick (a
partial brick at the wrap), every order and brick shape, one and two
threads to an atom, and charges beyond the range of the short conversion to
grid words, against the oracle."""
import numpy as np
import pytest

from mdir_amd import runtime as rt
from mdir_amd import systems as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def charged(grid, order, big, n=300):
    """Charges scattered over a 2.5 nm box, one of them `big` (forces stay
    below the 2^31 kJ/mol/nm that a force word holds)."""
    rng = np.random.default_rng(sum(grid) + order)
    q = rng.uniform(-1.0, 1.0, n)
    q[7] = big
    return S.System(positions=rng.uniform(0.0, 2.5, (n, 3)), masses=np.ones(n), charges=q,
                    types=np.zeros(n, np.int32), sigma=np.full((1, 1), 0.3),
                    epsilon=np.zeros((1, 1)), box=np.full(3, 2.5), beta=S.ewald_beta(0.9),
                    pme_grid=grid, pme_order=order)


@pytest.mark.parametrize("bricks", [8, 4, 2, 1])
@pytest.mark.parametrize("grid,order", [((16, 21, 18), 4), ((25, 18, 27), 6), ((30, 35, 20), 8),
                                        ((49, 50, 28), 4), ((63, 42, 36), 6), ((18, 20, 21), 4)])
def test_reciprocal_forces_by_bricks(grid, order, bricks):
    """The reciprocal forces at the 5e-6 relative RMS bar (49 x 50 and
    63 x 42 in bricks of one line: more blocks than the two-thread form
    takes)."""
    from mdir_amd.simulation import Simulation
    print(f"case: grid {grid}, order {order}, bricks of {bricks} lines", flush=True)
    s = charged(grid, order, 1.0)
    sim = Simulation(s)
    sim.launch_shape = (16, bricks, 0)
    F, _ = sim.force_terms(rt.TERM_RECIP)
    assert O.rel_rms(F, O.Oracle(s).pme()[0]) < 5e-6
    sim.close()


@pytest.mark.parametrize("big", [900.0, 1023.0, 1025.0])
def test_large_charges(big):
    """Grid words of a charge on both sides of the short conversion's range.
    The potential is f32 and its largest part the charge's own, `big` times
    that of the others, which the sums over the stencil cancel: the bar is 5
    roundings of 2^-24 of it.  A word out of range is wrong by its size.
    (A brick's part of the charge's own force, some f q^2 K beta / L = 2e9 at
    1,100 e, has to stay below the 2^31 of a force word, which bounds the
    charge from above.)"""
    from mdir_amd.simulation import Simulation
    print(f"case: charges of {big} e", flush=True)
    s = charged((24, 28, 30), 4, big)
    sim = Simulation(s)
    F, _ = sim.force_terms(rt.TERM_RECIP)
    Fo, _ = O.Oracle(s).pme()
    assert np.abs(Fo).max() < 2.0 ** 30
    small = np.abs(s.charges) <= 1.0
    assert O.rel_rms(F, Fo) < 5 * 2.0 ** -24 * big
    assert O.rel_rms(F[small], Fo[small]) < 5 * 2.0 ** -24 * big
    sim.close()
