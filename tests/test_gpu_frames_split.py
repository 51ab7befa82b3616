"""Batches on both sides of the line where the bricks' launches take one
thread to an atom instead of two: a frame has the same bits in either."""
import dataclasses

import numpy as np
import pytest

from mdir_amd import systems as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [4, 6, 8])
def test_a_frame_has_the_same_bits_in_every_batch(order):
    """240 bricks a frame: one frame takes two threads to an atom, five take
    one.  Forces, energies and Hessian products to the bit; the products in
    the tunables, summed over the frames in f64, to its rounding."""
    from mdir_amd.frames import FrameEvaluator
    print(f"case: 5 frames of 960 atoms on 60 x 64 x 32, order {order}", flush=True)
    s = dataclasses.replace(S.solvated_solutes(nwaters=300, nsolutes=12, seed=5,
                                               grid=(60, 64, 32)), pme_order=order)
    X = S.perturbed_frames(s, 5, seed=2)
    rng = np.random.default_rng(3)
    G, g = rng.normal(size=X.shape), rng.normal(size=5)
    ev, one = FrameEvaluator(s, max_frames=5), FrameEvaluator(s, max_frames=1)
    a = ev.evaluate(X)
    H, p = ev.hvp(G), a.vjp(g, positions=G)
    total = {k: np.zeros_like(v) for k, v in p.items()}
    for n in range(5):
        r = one.evaluate(X[n:n + 1])
        assert np.array_equal(r.forces[0], a.forces[n])
        assert np.array_equal(r.terms[0], a.terms[n])
        assert np.array_equal(one.hvp(G[n:n + 1])[0], H[n])
        for k, v in r.vjp(g[n:n + 1], positions=G[n:n + 1]).items():
            total[k] += v
    for k in p:
        np.testing.assert_allclose(total[k], p[k], rtol=1e-12, atol=1e-12 * np.abs(p[k]).max())
    ev.close()
    one.close()
