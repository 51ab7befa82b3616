"""The integration's blocks at their edges: 64 waters, 38 constraint
clusters or 64 free atoms to a block, one more and one fewer, systems of one
kind of unit and of all, against the oracle's steps.  First with no forces (no
charges, no Lennard-Jones), where both sides do the same f64 operations but
for the reciprocals in a cluster's equations and the noise's mathematics;
then with them, with and without PME's own force words."""
import dataclasses

import numpy as np
import pytest

from mdir_amd import systems as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def molecules(waters, clusters, free):
    """Waters, clusters of 2 to 5 atoms (the centre anywhere in the cluster)
    and free atoms, scattered over a 5 nm box."""
    rng = np.random.default_rng(waters + 1000 * clusters + 7 * free)
    d_oh, d_hh = S.TIP3P["d_oh"], S.TIP3P["d_hh"]
    height = np.sqrt(d_oh ** 2 - (0.5 * d_hh) ** 2)
    water = np.array([[0, 0, 0], [height, 0.5 * d_hh, 0], [height, -0.5 * d_hh, 0]])
    arms = np.array([[1, 1, 1], [1, -1, -1], [-1, 1, -1], [-1, -1, 1]]) / np.sqrt(3.0)
    x, masses, first, bonds, lengths = [], [], [], [], []

    def place(local):
        q, _ = np.linalg.qr(rng.normal(size=(3, 3)))
        x.extend(rng.uniform(0.3, 4.7, 3) + local @ q.T)

    for _ in range(waters):
        first.append(len(x))
        place(water)
        masses.extend([15.9994, 1.008, 1.008])
    for c in range(clusters):
        size = 2 + c % 4
        centre = c % size
        arm = rng.uniform(0.09, 0.13, size)
        local = np.zeros((size, 3))
        others = [m for m in range(size) if m != centre]
        for k, m in enumerate(others):
            local[m] = arm[m] * arms[k]
            bonds.append((len(x) + centre, len(x) + m))
            lengths.append(arm[m])
        place(local)
        masses.extend(12.011 if m == centre else 1.008 for m in range(size))
    for _ in range(free):
        place(np.zeros((1, 3)))
        masses.append(22.99)
    n = len(x)
    return S.System(positions=np.array(x), masses=np.array(masses), charges=np.zeros(n),
                    types=np.zeros(n, np.int32), sigma=np.full((1, 1), 0.3),
                    epsilon=np.zeros((1, 1)), box=np.full(3, 5.0),
                    waters=np.array(first, np.int32),
                    constraints=np.array(bonds, np.int32).reshape(-1, 2),
                    constraint_length=np.array(lengths))


@pytest.mark.parametrize("langevin", [False, True])
@pytest.mark.parametrize("units", [(64, 0, 0), (65, 0, 0), (1, 1, 1), (63, 38, 2), (64, 39, 64),
                                   (0, 77, 0), (0, 0, 64), (0, 0, 65), (0, 3, 193)])
def test_units_at_block_edges(units, langevin):
    """A step adds roundings of some 1e-15 nm and 1e-12 nm/ps (1 / dt times
    those); the Newton sweeps of a cluster converge to its roundings on both
    sides.  The bars are a thousand times that, and a wrong member, centre,
    mass or noise moves an atom by 1e-4 nm."""
    from mdir_amd.simulation import Simulation
    print(f"case: {units} waters, clusters, free atoms; langevin={langevin}", flush=True)
    s = molecules(*units)
    o = O.Oracle(s)
    v0 = S.initial_velocities(s, 5, 300.0)
    v0 = o.rattle_velocities(s.positions, o.settle_velocities(s.positions, v0))
    sim = Simulation(s, skin=0.2)
    sim.velocities = v0
    done = 0
    if langevin:
        sim.step_count = 7
        sim.set_langevin(300.0, 2.0, seed=11)
    for steps, graph in ((1, 0), (7, 3), (12, 0)):
        sim.run(steps - done, 0.001, graph=graph)
        done = steps
        x, v = sim.positions, sim.velocities
        if langevin:
            xo, vo, _ = o.langevin(s.positions, v0, 0.001, steps, seed=11, friction=2.0,
                                   temperature=300.0, first_step=7)
        else:
            xo, vo, _ = o.nve(s.positions, v0, 0.001, steps)
        print(f"  {steps} steps: |dx| {np.abs(x - xo).max():.1e}, |dv| {np.abs(v - vo).max():.1e}",
              flush=True)
        assert np.abs(x - xo).max() < 1e-12
        assert np.abs(v - vo).max() < 1e-9
    sim.close()


def interacting(waters, clusters, free, pme):
    """molecules() on the sites of a lattice 0.83 nm apart, with Lennard-Jones
    and charges (waters TIP3P's, clusters neutral, free atoms +-0.5 e),
    nothing within a unit."""
    s = molecules(waters, clusters, free)
    sizes = [3] * waters + [2 + c % 4 for c in range(clusters)] + [1] * free
    first = np.concatenate([[0], np.cumsum(sizes)])[:-1]
    rng = np.random.default_rng(len(sizes))
    site = np.stack(np.unravel_index(rng.permutation(len(sizes)), (6, 6, 6)), 1)
    x, q, types, excluded = s.positions.copy(), np.zeros(s.n), np.zeros(s.n, np.int32), []
    for u, (a, k) in enumerate(zip(first, sizes)):
        x[a:a + k] += (site[u] + 0.5) * 0.83 + rng.uniform(-0.1, 0.1, 3) - x[a:a + k].mean(0)
        if u < waters:
            q[a:a + 3] = [-0.834, 0.417, 0.417]
        elif k == 1:
            q[a] = 0.5 if u % 2 else -0.5
        else:
            q[a:a + k] = 0.3
            q[a + k - 1] = -0.3 * (k - 1)
        types[a:a + k] = u % 2
        excluded += [(a + i, a + j) for i in range(k) for j in range(i + 1, k)]
    return dataclasses.replace(
        s, positions=x, charges=q, types=types,
        sigma=np.array([[0.55, 0.58], [0.58, 0.62]]), epsilon=np.array([[0.9, 0.7], [0.7, 0.6]]),
        beta=S.ewald_beta(0.9) if pme else 0.0, pme_grid=(40, 40, 40) if pme else (0, 0, 0),
        exclusions=np.array(excluded, np.int32).reshape(-1, 2))


@pytest.mark.parametrize("pme", [False, True])
@pytest.mark.parametrize("langevin", [False, True])
@pytest.mark.parametrize("units", [(65, 0, 0), (1, 1, 1), (63, 38, 2), (64, 39, 64), (0, 77, 0),
                                   (0, 0, 65), (0, 3, 193)])
def test_units_at_block_edges_with_forces(units, langevin, pme):
    """Launch by launch and from graphs, so that the first, the between and
    the closing launches all take and clear force words, place-ordered ones
    alone and with PME's.  The forces are f32 sums good to 5e-6 of their RMS;
    the bar gives an atom's 20 times that, in one direction for the whole run.
    It is under a tenth of what one lost, doubled or misplaced half kick of
    that RMS changes the heaviest atom by."""
    from mdir_amd.simulation import Simulation
    print(f"case: {units} waters, clusters, free atoms with forces; langevin={langevin}, "
          f"pme={pme}", flush=True)
    s = interacting(*units, pme)
    o = O.Oracle(s)
    Fo, _ = o.total()
    rms = np.sqrt((Fo ** 2).mean())
    v0 = S.initial_velocities(s, 5, 300.0)
    v0 = o.rattle_velocities(s.positions, o.settle_velocities(s.positions, v0))
    dt, steps = 0.001, 12
    if langevin:
        xo, vo, _ = o.langevin(s.positions, v0, dt, steps, seed=11, friction=2.0,
                               temperature=300.0, first_step=7)
    else:
        xo, vo, _ = o.nve(s.positions, v0, dt, steps)
    bar = steps * dt * 20 * 5e-6 * rms / s.masses.min()
    one_kick = 0.5 * dt * rms / s.masses.max()   # what a lost kick changes at least
    assert bar < 0.1 * one_kick
    for graph in (0, 3):
        sim = Simulation(s, skin=0.2)
        sim.velocities = v0
        if langevin:
            sim.step_count = 7
            sim.set_langevin(300.0, 2.0, seed=11)
        for part in (1, 5, 6):
            sim.run(part, dt, graph=graph)
        x, v = sim.positions, sim.velocities
        print(f"  graph {graph}: |dx| {np.abs(x - xo).max():.1e}, |dv| {np.abs(v - vo).max():.1e},"
              f" bar {bar:.1e}, a kick {one_kick:.1e}", flush=True)
        assert np.abs(v - vo).max() < bar
        assert np.abs(x - xo).max() < bar * steps * dt
        sim.close()
