"""Field transfers on both sides of the staging buffer's size (512 KiB), from
buffers at odd addresses: what goes in comes out, to the bit."""
import numpy as np
import pytest

from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("nx,ny", [(4, 4), (192, 128), (144, 216), (192, 192), (256, 192),
                                   (256, 256)])
def test_round_trip(nx, ny, prec):
    print(f"[staging] {nx}x{ny} precision={prec}", flush=True)
    s = Spectral2D(nx, ny, precision=prec)
    n = 2 * s.cISize * s.nyG
    rng = np.random.default_rng(nx + ny)
    raw = np.empty(n + 1)
    a, b = raw[1:], rng.standard_normal(n).astype(np.float32).astype(np.float64)
    a[:] = rng.standard_normal(n).astype(np.float32)
    s.set_field("u", a)
    s.set_field("v", b)
    out = np.zeros(n + 1)[1:]
    assert np.array_equal(s.get_field("u", out), a)
    assert np.array_equal(s.get_field("v"), b)
    s.close()
