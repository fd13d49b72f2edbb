"""Field transfers to and from page-locked buffers, which are copied directly at
every size, next to ordinary ones: the same values."""
import numpy as np
import pytest
import torch

from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("nx,ny", [(4, 4), (64, 64), (144, 216), (192, 192)])
def test_page_locked_buffers(nx, ny, prec):
    print(f"[staging] page-locked {nx}x{ny} precision={prec}", flush=True)
    s = Spectral2D(nx, ny, precision=prec)
    rng = np.random.default_rng(nx + ny)
    a, b = (torch.empty(s.ndoubles, dtype=torch.float64, pin_memory=True).numpy() for _ in "ab")
    for k in range(3):
        a[:] = rng.standard_normal(s.ndoubles).astype(np.float32)
        s.set_field("u", a)
        want = a.copy()
        a[:] = 0.0  # (the call has taken its values)
        s.set_field("v", want)
        b[:] = 0.0
        assert np.array_equal(s.get_field("u", b), want)
        assert np.array_equal(s.get_field("u"), want) and np.array_equal(s.get_field("v", b), want)
    s.close()
