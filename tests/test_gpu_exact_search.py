"""The search's test of atom pairs (boxes of 64,000 atoms and more): on both
sides of the line the pairs within the cut-off and within the whole reach
are all listed, the forces of a step's list equal those of a fresh one, and
a box of columns of very uneven filling keeps its pairs."""
import numpy as np
import pytest

from mdir_amd import systems as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def gas(n, edge, seed, clumped):
    rng = np.random.default_rng(seed)
    x = rng.uniform(0.0, edge, (n, 3))
    if clumped:  # half the box nearly empty
        x[: n // 8, 0] *= 0.5
        x[n // 8:, 0] = edge * (0.5 + 0.5 * rng.uniform(0, 1, n - n // 8))
    return S.System(positions=x, masses=np.full(n, 39.95), charges=np.zeros(n),
                    types=np.zeros(n, np.int32), sigma=np.full((1, 1), 0.2),
                    epsilon=np.full((1, 1), 1e-6), box=np.array([edge, edge, edge]), cutoff=0.6)


@pytest.mark.parametrize("clumped", [False, True])
@pytest.mark.parametrize("n", [63999, 64000, 64003])
def test_every_pair_is_listed(n, clumped):
    """The pairs at two reaches against a k-d tree's (f64): all of them, and
    none beyond the export's margin of 3e-6 of the box edges' sum; 5e-6 nm
    for the f32 rounding of the distances."""
    from scipy.spatial import cKDTree
    from mdir_amd.simulation import Simulation
    print(f"case: {n} atoms, clumped={clumped}", flush=True)
    s = gas(n, 16.0, n, clumped)
    sim = Simulation(s, skin=0.1)
    tree = cKDTree(s.positions % 16.0, boxsize=16.0)
    for reach in (0.6, 0.69):
        got = sim.neighbor_pairs(reach)
        got = set(map(tuple, np.asarray(got).reshape(-1, 2).tolist()))
        inner = tree.query_pairs(reach - 5e-6)
        outer = tree.query_pairs(reach + 3e-6 * 48.0 + 5e-6)
        assert inner <= got <= outer
    sim.close()


def test_forces_between_rebuilds():
    """65,856 atoms of TIP3P: forces of the list in use after 40 steps
    against the oracle (5e-6 relative RMS), and every pair of the list's
    cut-off taken by the pair loop."""
    from mdir_amd.simulation import Simulation
    unit = S.tip3p_box(2744, S.water_edge(2744), seed=8, grid=(40, 40, 40))
    base = Simulation(unit)
    base.minimize(40, 0.01)
    unit = unit.copy()
    unit.positions = base.positions
    base.close()
    cells = np.array([(i, j, k) for i in range(2) for j in range(2) for k in range(2)])
    first = np.arange(8) * unit.n
    rep = lambda a: np.tile(a, 8)
    import dataclasses
    w = dataclasses.replace(
        unit, positions=(unit.positions[None] + (cells * unit.box)[:, None]).reshape(-1, 3),
        box=unit.box * 2, masses=rep(unit.masses), charges=rep(unit.charges),
        types=rep(unit.types), pme_grid=(80, 80, 80),
        exclusions=(unit.exclusions[None] + first[:, None, None]).reshape(-1, 2).astype(np.int32),
        waters=(unit.waters[None] + first[:, None]).reshape(-1).astype(np.int32))
    assert w.n >= 64000
    print(f"case: {w.n} atoms, forces between rebuilds", flush=True)
    sim = Simulation(w, skin=0.15)
    sim.velocities = S.initial_velocities(w, 3, 300.0)
    sim.run(40, 0.002, graph=20)
    F, _, counts = sim.check_list()
    assert counts["list"] == counts["pair_loop"]
    Fo, _ = O.Oracle(w).total(sim.positions)
    assert O.rel_rms(F, Fo) < 5e-6
    sim.close()
