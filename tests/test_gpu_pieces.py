"""The pair loop's pieces: boxes on both sides of the lines where a wave's
share of a row is halved, against the oracle.  Segments of 16 entries come
down to pieces of 4, 8 and 16 in these boxes, segments of 24 and 48 to 6 and
12; test_whole_segments takes boxes that keep 24 and 48 whole."""
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


@pytest.mark.parametrize("waters,segment", [(1800, 24), (2200, 24), (3600, 48), (4400, 48)])
def test_whole_segments(waters, segment):
    """Boxes on both sides of the lines above which a wave takes a whole
    segment of 24 (1,700 waters) or 48 entries (3,700), at the same bars."""
    test_forces_of_every_piece(waters, segment)


def test_segments_of_one_piece_are_timed_once():
    """In a box of 500 waters segments of 24 and 48 are both pieces of 6, one
    launch: the trial gives them one time.  16 (pieces of 4) is another, and
    in a box of 4,400 waters all three differ."""
    from mdir_amd.simulation import Simulation
    for waters, alike in ((500, True), (4400, False)):
        print(f"case: {waters} waters, trial of the segment lengths", flush=True)
        edge = S.water_edge(waters)
        w = S.tip3p_box(waters, edge, seed=7, grid=(24, 24, 24) if edge < 2.6 else (48, 48, 48))
        sim = Simulation(w)
        sim.minimize(10, 0.01)
        ms = {k[2]: t for k, t in
              sim.autotune(Simulation.TUNE_SEGMENTS, steps=5, graphs=1).items()}
        assert set(ms) == {16, 24, 48}
        assert (ms[24] == ms[48]) == alike
        assert ms[16] != ms[24]
        sim.close()
