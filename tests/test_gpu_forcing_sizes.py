"""s2d_set_forcing at the sizes whose fused step runs on the runtime plans."""
import numpy as np
import pytest

from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N", [32, 36, 48, 72, 144, 576])
def test_forcing_from_rest(N, prec):
    """One inviscid step from rest with a single-mode forcing (no nonlinear
    term): w = -dt F, to the rounding of three stages; none once cleared."""
    print(f"[forcing] N={N} prec={prec}", flush=True)
    dt, F = 0.25, 2.0 - 1.0j
    s = Spectral2D(N, precision=prec)
    f = s.field()
    s.cview(f)[4, 3] = F
    s.set_field("tmp", f)
    s.set_forcing("tmp")
    s.zero_field("w")
    s.rk3_steps(1, 0.0, dt)
    w = s.cview(s.get_field("w")).copy()
    s.clear_forcing()
    s.zero_field("w")
    s.rk3_steps(1, 0.0, dt)
    assert not np.any(s.get_field("w"))
    s.close()
    eps = 2.3e-16 if prec == FP64 else 1.2e-7
    assert abs(w[4, 3] + dt * F) < 8 * eps
    w[4, 3] = 0.0
    assert np.abs(w).max() < 8 * eps
