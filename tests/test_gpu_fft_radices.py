"""The transforms' radices 2 to 10 (an axis takes the fewest passes they
allow): grids whose edges use each of them, one pass, two and three, through
the runtime ABI against numpy's transform, and through PME against the
oracle (planes held in LDS with edges that need true quotients, and tiles of
lines)."""
import ctypes as C

import numpy as np
import pytest

from mdir_amd import runtime as rt
from mdir_amd import systems as S
from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [(6, 9, 10), (54, 36, 90), (70, 18, 60), (162, 14, 8),
                               (7, 5, 6), (2, 3, 4), (250, 4, 252)])
@pytest.mark.parametrize("single", [True, False])
def test_forward_and_backward(K, single):
    """The bars of the ABI's own tests: 3e-6 of the largest value in f32
    (passes of at most log2 K roundings of 6e-8 each), 1e-12 in f64."""
    print(f"case: radices {K} single={single}", flush=True)
    L = rt.lib()
    s = L.mgpuStreamCreate()
    real = np.random.default_rng(sum(K)).standard_normal(K)
    dt = np.float32 if single else np.float64
    h = K[2] // 2 + 1
    host, spec = real.astype(dt), np.zeros((K[0], K[1], h, 2), dt)
    r_dev = L.mgpuMemAlloc(host.nbytes, s, False)
    c_dev = L.mgpuMemAlloc(spec.nbytes, s, False)
    L.mgpuMemcpy(r_dev, host.ctypes.data, host.nbytes, s)
    rb = rt.Buffer1(r_dev, r_dev, 0, real.size, 1)
    cb = rt.Buffer1(c_dev, c_dev, 0, spec.size, 1)
    name = "F32" if single else ""
    getattr(L, "_mlir_ciface_mdrtCudaFFTForward3D" + name)(C.byref(rb), C.byref(cb), *K)
    L.mgpuMemcpy(spec.ctypes.data, c_dev, spec.nbytes, s)
    L.mgpuStreamSynchronize(s)
    ref = np.fft.rfftn(host.astype(np.float64))
    tol = 3e-6 if single else 1e-12
    assert np.abs(spec[..., 0] + 1j * spec[..., 1] - ref).max() <= tol * np.abs(ref).max()
    spec = np.stack([ref.real, ref.imag], -1).astype(dt)
    L.mgpuMemcpy(c_dev, spec.ctypes.data, spec.nbytes, s)
    getattr(L, "_mlir_ciface_mdrtCudaFFTBackward3D" + name)(C.byref(cb), C.byref(rb), *K)
    back = np.zeros(K, dt)
    L.mgpuMemcpy(back.ctypes.data, r_dev, back.nbytes, s)
    L.mgpuStreamSynchronize(s)
    assert np.abs(back / real.size - real).max() <= 10 * tol * np.abs(real).max()
    L.mgpuMemFree(r_dev, s)
    L.mgpuMemFree(c_dev, s)


@pytest.mark.parametrize("grid", [(36, 42, 40), (24, 28, 30), (54, 60, 50), (18, 20, 16),
                                  (70, 72, 60)])
def test_reciprocal_forces(grid):
    """The reciprocal forces alone at the 5e-6 relative RMS bar."""
    from mdir_amd.simulation import Simulation
    print(f"case: PME grid {grid}", flush=True)
    w = S.tip3p_box(512, 2.5, seed=11, grid=grid)
    sim = Simulation(w)
    F, e = sim.force_terms(rt.TERM_RECIP)
    Fo, _ = O.Oracle(w).pme()
    assert O.rel_rms(F, Fo) < 5e-6
    sim.close()
