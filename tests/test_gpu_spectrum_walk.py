"""The shell walk of the device spectrum on ragged grids: every mode counted
once and in its shell, against a sum over the whole grid in NumPy."""
import numpy as np
import pytest

from spectral2d_amd._lib import NO_DEALIASING
from spectral2d_amd.spectral import FP64, Spectral2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(4, 4), (8, 6), (48, 32), (32, 96), (54, 48), (162, 6),
                                   (6, 162), (256, 192)])
def test_walk_meets_every_mode_once(nx, ny):
    print(f"[spectrum] walk {nx}x{ny}", flush=True)
    s = Spectral2D(nx, ny, dealias=NO_DEALIASING, precision=FP64)
    rng = np.random.default_rng(nx * 1000 + ny)
    w = rng.standard_normal(2 * s.cISize * s.nyG)
    s.set_field("psi", w)
    ek, cnt, *_ = s.ComputeSpectrum(1e-3)
    p = w.view(np.complex128).reshape(s.nyG, s.cISize)
    kx = np.arange(s.cISize)
    ky = np.arange(s.nyG)
    ky = np.where(ky <= s.nyG // 2, ky, ky - s.nyG)
    q = kx[None, :] ** 2 + ky[:, None] ** 2
    shell = np.floor(np.sqrt(q) + 0.5).astype(int)
    # the Nyquist wavenumbers are masked in the derivative along their axis
    e = np.abs(p) ** 2 * ((kx * (kx != nx // 2))[None, :] ** 2 + (ky * (ky != ny // 2))[:, None] ** 2)
    edge = (kx == 0) | (kx == nx // 2)
    e = e * np.where(edge, 0.5, 1.0)[None, :]
    n = np.where(edge, 1, 2)[None, :] * np.ones_like(q)
    keep = shell < len(ek)
    ref = np.bincount(shell[keep], e[keep], len(ek))
    ref_n = np.bincount(shell[keep], n[keep], len(ek)).astype(int)
    assert np.array_equal(cnt, ref_n)
    # double sums of nonnegative terms: n eps of the shell's own energy
    assert np.all(np.abs(ek - ref) <= 1e-13 * ref.max())
    s.close()
