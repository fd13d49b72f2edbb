"""The compiled reference-layout transforms and the three-launch ComputeRHS
and IntegrateOneStep against the runtime plans (S2D_GENERIC_KERNELS=1) and
against the routines called one by one."""
import os

import numpy as np
import pytest

from spectral2d_amd import DEALIAS_3_2_RULE, NO_DEALIASING
from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu

# lane groups of 4, 6, 8, 12, 16, 24, 48, 64, 96, 128, 192 and 256 lanes (the
# last two longer than a wave's rows), ragged last tiles, unequal sides
GRIDS = [(64, 96, DEALIAS_3_2_RULE), (96, 64, DEALIAS_3_2_RULE), (128, 32, DEALIAS_3_2_RULE),
         (48, 128, DEALIAS_3_2_RULE), (192, 512, DEALIAS_3_2_RULE), (384, 96, DEALIAS_3_2_RULE),
         (768, 192, DEALIAS_3_2_RULE), (1536, 64, DEALIAS_3_2_RULE), (64, 1536, DEALIAS_3_2_RULE),
         (1024, 64, DEALIAS_3_2_RULE), (64, 2048, DEALIAS_3_2_RULE), (2048, 64, DEALIAS_3_2_RULE),
         (64, 64, NO_DEALIASING), (256, 128, NO_DEALIASING), (512, 256, NO_DEALIASING)]


def pair(nx, ny, dealias, prec):
    out = []
    for flag in ("1", "0"):
        os.environ["S2D_GENERIC_KERNELS"] = flag
        try:
            out.append(Spectral2D(nx, ny, dealias=dealias, precision=prec))
        finally:
            os.environ.pop("S2D_GENERIC_KERNELS", None)
    return out


def physical(s, seed):
    """A real field with content in every mode (padding reals zero)."""
    rng = np.random.default_rng(seed)
    buf = s.field()
    s.rview(buf)[:, : s.nxG] = rng.standard_normal((s.nyG, s.nxG))
    return buf


def kept_modes(s):
    """Where the dW of a truncated state means something: past the kept modes
    it is -nu k^2 times the rounding of a zero."""
    return s.kx[None, :].astype(int) ** 2 + s.ky[:, None].astype(int) ** 2 <= (s.nx // 2) ** 2


def close(a, b, tol):
    scale = np.linalg.norm(b)
    assert np.isfinite(a).all()
    assert np.linalg.norm(a - b) <= tol * scale, np.linalg.norm(a - b) / scale


# relative L2 bars: a transform's rounding grows as log2 of its points (the
# parity suite's 1e-14 log2 n^2 in FP64, 2^29 times that in FP32, rounded);
# a right-hand side and a step hold a few transforms and a division each
TOL = {FP64: 1e-13, FP32: 2e-5}


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("nx,ny,dealias", GRIDS)
def test_against_runtime_plans(nx, ny, dealias, prec):
    print(f"[ref] {nx}x{ny} dealias={dealias} prec={prec}", flush=True)
    a, b = pair(nx, ny, dealias, prec)
    buf = physical(a, nx + ny)
    got = []
    for s in (a, b):
        s.set_field("tmp", buf)
        s.TransformR2C("tmp")
        r2c = s.get_field("tmp")
        s.TransformC2R("tmp")
        c2r = s.get_field("tmp")
        # an untruncated vorticity, its streamfunction, the right-hand side
        s.set_field("w", buf)
        s.TransformR2C("w")
        s.copy_field("w", "wS")
        s.ComputePsi("wS", "psiS")
        s.ComputeRHS(1e-3, "u", "v", "wS", "psiS", "dW")
        rhs = [s.get_field(f) for f in ("u", "v", "wS", "dW", "psiS")]
        # a whole step from it
        s.ComputePsi()
        s.IntegrateOneStep(1e-3, 1e-4)
        step = [s.get_field(f) for f in ("w", "psi", "u", "v", "wS", "psiS", "dW")]
        step[-1] = s.cview(step[-1])[kept_modes(s)]
        got.append([r2c, c2r] + rhs + step)
        s.close()
    names = ("r2c", "c2r", "u", "v", "wS", "dW", "psiS", "step w", "step psi", "step u", "step v",
             "step wS", "step psiS", "step dW")
    for name, x, y in zip(names, got[1], got[0]):
        print(" ", name, flush=True)
        close(x, y, TOL[prec])
    assert np.all(got[1][1].reshape(a.nyG, a.rISize)[:, a.nxG:] == 0.0)


@pytest.mark.parametrize("prec", [FP64, FP32])
def test_shared_slots_keep_the_routines_order(prec):
    """ComputeRHS with one slot in two roles runs routine by routine."""
    a, b = pair(96, 96, DEALIAS_3_2_RULE, prec)
    buf = physical(a, 3)
    got = []
    for s in (a, b):
        s.set_field("w", buf)
        s.TransformR2C("w")
        s.Truncate("w")
        s.copy_field("w", "wS")
        s.ComputeRHS(1e-3, "u", "v", "wS", "wS", "dW")  # psi in w's slot
        # (dW is left out: with psi = w the two derivatives cancel to rounding)
        got.append([s.get_field(f) for f in ("u", "v", "wS")])
        s.close()
    for x, y in zip(got[1], got[0]):
        close(x, y, TOL[prec])


def test_nonfinite_values_spread():
    """A NaN or an infinity in the state reaches every kept mode of the step,
    as on the runtime plans; tiny values keep their size."""
    for bad in (np.nan, np.inf):
        s = Spectral2D(96)
        buf = s.field()
        s.cview(buf)[3, 2] = bad
        s.set_field("w", buf)
        s.ComputePsi()
        s.IntegrateOneStep(1e-3, 1e-4)
        w = s.cview(s.get_field("w"))
        assert not np.isfinite(w[kept_modes(s)][1:]).any()  # (the first is the mean)
        s.close()
    s = Spectral2D(96)
    buf = s.field()
    s.rview(buf)[:, : s.nxG] = 1e-295 * (1.0 + np.arange(s.nxG) % 7)
    s.set_field("tmp", buf)
    s.TransformR2C("tmp")
    ref = np.fft.rfft2(s.rview(buf)[:, : s.nxG] * 1e295) / (s.nxG * s.nyG)
    got = s.cview(s.get_field("tmp")) * 1e295
    assert np.abs(got - ref).max() < 1e-13
    s.close()
