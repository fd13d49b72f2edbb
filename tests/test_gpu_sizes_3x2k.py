"""The fused step's compiled kernels of the padded sizes 144 * 2^k (N = 96,
192, ..., 1536): lane groups of 12 * 2^k lanes."""
import os

import numpy as np
import pytest

import oracle
from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


def rel(a, b):
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


def make(N, prec, generic):
    os.environ["S2D_GENERIC_KERNELS"] = "1" if generic else "0"
    try:
        return Spectral2D(N, precision=prec)
    finally:
        os.environ.pop("S2D_GENERIC_KERNELS", None)


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("N", [96, 192, 384, 768, 1536])
def test_compiled_against_runtime_plans(N, prec):
    """Three CFL steps, two fixed ones and a step clamped to an end time, from
    a turbulent state with a strong mode at (N/2, 0) (the last column, which
    passes A and C write without a transform), on both sets of kernels. The
    bars are those of the other sizes: 1e-13 in FP64 (here 6 steps instead of
    20), and in FP32 that of a schedule variant, 1e-5."""
    print(f"[3x2k] N={N} prec={prec}", flush=True)
    o = oracle.Oracle(N)
    st = o.new_state()
    o.set_turbulence(st["w"], st["psi"], 7, 8.0, 0.5)
    o.cview(st["w"])[0, N // 2] += 30.0 - 20.0j
    out = []
    for generic in (True, False):
        s = make(N, prec, generic)
        s.set_field("w", st["w"])
        s.rk3_steps(3, 1e-4, 0.0, 0.5)
        dt = s.ComputeTimeStep(0.5)
        if not out:
            fixed = 0.5 * dt
        s.rk3_steps(2, 1e-4, fixed)
        t = s.get_time()[0]
        s.set_end_time(t + 0.25 * fixed)
        s.rk3_steps(2, 1e-4, fixed)
        assert s.get_time()[1] == 6  # the last step is at the end time already
        out.append((s.cview(s.get_field("w")).copy(), s.cview(s.get_field("psi")).copy(), dt))
        s.close()
    tol = 1e-13 if prec == FP64 else 1e-5
    assert rel(out[1][0], out[0][0]) < tol
    assert rel(out[1][1], out[0][1]) < tol
    assert abs(out[1][2] - out[0][2]) < tol * out[0][2]
    m = [x[0][0, N // 2] for x in out]
    assert abs(m[1] - m[0]) < tol * abs(m[0])


@pytest.mark.parametrize("prec", [FP64, FP32])
def test_forcing(prec):
    """One inviscid step from rest with a single-mode forcing (no nonlinear
    term): w = -dt F, to the rounding of three stages."""
    N, dt = 96, 0.25
    s = Spectral2D(N, precision=prec)
    f = s.field()
    s.cview(f)[4, 3] = 2.0 - 1.0j
    s.set_field("tmp", f)
    s.set_forcing("tmp")
    s.zero_field("w")
    s.rk3_steps(1, 0.0, dt)
    w = s.cview(s.get_field("w"))
    eps = 2.3e-16 if prec == FP64 else 1.2e-7
    assert abs(w[4, 3] + dt * (2.0 - 1.0j)) < 8 * eps
    w[4, 3] = 0.0
    assert np.abs(w).max() < 8 * eps
    s.close()
