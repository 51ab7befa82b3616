"""The pair loop's pieces: boxes on both sides of the lines where a wave's
share of a row is halved (4, 8 and 16 entries), with each segment length,
against the oracle."""
import pytest

from mdir_amd import systems as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waters", [216, 500, 800, 1100, 1500])
@pytest.mark.parametrize("segment", [16, 24, 48])
def test_forces_of_every_piece(waters, segment):
    """The 5e-6 relative RMS bar of the f32 pair loop and PME."""
    from mdir_amd.simulation import Simulation
    print(f"case: {waters} waters, segments of {segment}", flush=True)
    edge = max(S.water_edge(waters), 2.05)
    w = S.tip3p_box(waters, edge, seed=waters, grid=(24, 24, 24) if edge < 2.6 else (32, 32, 32))
    sim = Simulation(w)
    sim.minimize(10, 0.01)
    sim.launch_shape = (segment, 8, 0)
    F, e = sim.forces()
    Fo, eo = O.Oracle(w).total(sim.positions)
    assert O.rel_rms(F, Fo) < 5e-6
    # the sums over the pieces' energy slots: f32 pair energies, f64 sums
    for k in (O.E_LJ, O.E_COUL_DIRECT):
        assert abs(e[k] - eo[k]) < 2e-6 * max(abs(eo[O.E_LJ]), abs(eo[O.E_COUL_DIRECT]))
    sim.close()
