"""Diagnostics of an ensemble's runs (one pass over the compact state of all of
them) and the mode counts of the shell spectrum (counted on the device)."""
import numpy as np
import pytest

from spectral2d_amd import DEALIAS_3_2_RULE, NO_DEALIASING, S2DError
from spectral2d_amd.ensemble import Ensemble
from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [FP64, FP32])
def test_runs_equal_the_runs_alone(prec):
    """Every value bitwise, from a fresh state and after steps."""
    sizes = [64, 512, 128, 64, 256]
    e = Ensemble(sizes, prec)
    e.set_viscosity(1e-3)
    e.set_turbulence(np.arange(5), 6.0, 0.5)
    alone = []
    for r, n in enumerate(sizes):
        s = Spectral2D(n, precision=prec)
        s.SetTurbulence(r, 6.0, 0.5)
        alone.append(s)
    for steps in (0, 3):
        e.steps(steps, cfl=0.5)
        got = e.diagnostics()
        for r, s in enumerate(alone):
            s.rk3_steps(steps, 1e-3, 0.0, 0.5)
            assert got[r] == s.diagnostics(), (steps, r)
    w = np.zeros(e.ndoubles(2))
    w[2 * 5] = np.nan
    e.set_vorticity(2, w)
    with pytest.raises(S2DError, match="run 2"):
        e.diagnostics()
    e.close()
    for s in alone:
        s.close()


@pytest.mark.parametrize("nx,ny,dealias", [(24, 36, NO_DEALIASING), (36, 18, DEALIAS_3_2_RULE),
                                           (96, 64, DEALIAS_3_2_RULE)])
def test_shell_counts(nx, ny, dealias):
    s = Spectral2D(nx, ny, dealias=dealias)
    cnt = s.ComputeSpectrum()[1]
    k = np.sqrt(s.kx[None, :].astype(float) ** 2 + s.ky[:, None].astype(float) ** 2)
    wt = np.where((s.kx == 0) | (s.kx == s.nxG // 2), 1, 2)
    ref = np.bincount(np.floor(k + 0.5).astype(int).ravel(),
                      np.broadcast_to(wt, k.shape).ravel(), cnt.size).astype(int)
    assert np.array_equal(cnt, ref)
    s.close()
