"""The energies summed on the GPU: the kinetic energy at counts around the
blocks' strides against the host's sum, and the terms of an evaluation
against those taken one at a time."""
import numpy as np
import pytest

from mdir_amd import runtime as rt
from mdir_amd import systems as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 256, 257, 32768, 32769, 70001])
def test_kinetic_energy(n):
    """Sums of n positive terms in another order: sqrt(n) roundings."""
    from mdir_amd.simulation import Simulation
    print(f"case: kinetic energy of {n} atoms", flush=True)
    rng = np.random.default_rng(n)
    edge = max(2.5, (n / 30.0) ** (1 / 3))
    s = S.System(positions=rng.uniform(0, edge, (n, 3)), masses=rng.uniform(1.0, 40.0, n),
                 charges=np.zeros(n), types=np.zeros(n, np.int32), sigma=np.full((1, 1), 0.3),
                 epsilon=np.zeros((1, 1)), box=np.full(3, edge))
    sim = Simulation(s)
    sim.velocities = v = rng.normal(0, 0.5, (n, 3))
    want = 0.5 * (s.masses * (v * v).sum(1)).sum()
    _, e = sim.forces()
    got = dict(zip(rt.ENERGY_NAMES, e))["kinetic"]
    assert abs(got - want) < 4e-16 * np.sqrt(n) * want + 1e-15 * want
    # no forces: a run of no length in time keeps the velocities
    assert abs(sim.run(1, 1e-9) - want) < 1e-12 * want
    sim.close()


def test_terms_one_at_a_time():
    """Every energy of one evaluation is the energy of its term alone."""
    from mdir_amd.simulation import Simulation
    print("case: 512 waters, the energy terms alone and together", flush=True)
    sim = Simulation(S.tip3p_box(512, 2.5, seed=3, grid=(24, 24, 24)))
    _, whole = sim.forces()
    alone = [sim.force_terms(t)[1] for t in (rt.TERM_PAIRS, rt.TERM_SPECIAL, rt.TERM_RECIP)]
    names = dict(zip(rt.ENERGY_NAMES, range(len(whole))))
    fixed = [i for k, i in names.items() if k in ("coul_self", "disp_corr", "kinetic")]
    for i in range(len(whole)):
        parts = [a[i] for a in alone]
        if i not in fixed and any(parts):
            assert whole[i] == sum(parts), i
    sim.close()
