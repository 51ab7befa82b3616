"""The search's test of atom pairs (boxes of 64,000 atoms and more): on both
sides of the line the pairs within the cut-off and within the whole reach
are all listed, a run's list (and its pruned rows) holds every pair within the
cut-off between rebuilds, and a box of columns of very uneven filling keeps
its pairs."""
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


def keys(pairs, n):
    """Unordered pairs as sorted unique numbers."""
    a = np.asarray(pairs, np.int64).reshape(-1, 2)
    return np.unique(a.min(1) * n + a.max(1))


@pytest.mark.parametrize("prune_skin", [0.0, 0.05])
def test_forces_between_rebuilds(prune_skin):
    """65,856 atoms of TIP3P after 40 steps: the forces of the list in use
    against the oracle (5e-6 relative RMS), and that list's pairs (with
    pruning, also the pruned rows' that the pair loop runs over) against a
    k-d tree's in f64 without the excluded ones: all of them within the
    cut-off, none beyond the export's margin of 3e-6 of the box edges' sum;
    5e-6 nm for the f32 rounding of the distances."""
    import dataclasses
    from scipy.spatial import cKDTree
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
    w = dataclasses.replace(
        unit, positions=(unit.positions[None] + (cells * unit.box)[:, None]).reshape(-1, 3),
        box=unit.box * 2, masses=rep(unit.masses), charges=rep(unit.charges),
        types=rep(unit.types), pme_grid=(80, 80, 80),
        exclusions=(unit.exclusions[None] + first[:, None, None]).reshape(-1, 2).astype(np.int32),
        waters=(unit.waters[None] + first[:, None]).reshape(-1).astype(np.int32))
    assert w.n >= 64000
    print(f"case: {w.n} atoms, forces between rebuilds, pruned by {prune_skin}", flush=True)
    sim = Simulation(w, skin=0.15, prune_skin=prune_skin)
    sim.velocities = S.initial_velocities(w, 3, 300.0)
    sim.run(40, 0.002, graph=20)
    F, _, counts = sim.check_list()
    x = sim.positions
    Fo, _ = O.Oracle(w).total(x)
    assert O.rel_rms(F, Fo) < 5e-6
    tree = cKDTree(x % w.box, boxsize=w.box)
    excluded = keys(w.exclusions, w.n)
    inner, outer = (np.setdiff1d(keys(tree.query_pairs(r, output_type="ndarray"), w.n), excluded)
                    for r in (w.cutoff - 5e-6, w.cutoff + 3e-6 * w.box.sum() + 5e-6))
    assert len(inner) > 40 * w.n
    for pruned in ([False, True] if prune_skin > 0 else [False]):
        got = keys(sim.list_pairs(w.cutoff, pruned=pruned), w.n)
        assert len(np.setdiff1d(inner, got)) == 0
        assert len(np.setdiff1d(got, outer)) == 0
        assert len(got) == counts["pair_loop" if pruned else "list"]
    if prune_skin > 0:  # two sets of rows, the same pairs
        assert counts["list"] == counts["pair_loop"]
    sim.close()
