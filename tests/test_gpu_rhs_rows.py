"""ComputeRHS's rows with a lane group to a field and with one group to a row
(on either side of the rule that chooses), against the runtime plans, and
repeated on the same input to the bit."""
import os

import numpy as np
import pytest

from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu

# relative L2: a few transforms of up to 2^20 points, 1e-14 log2 n^2 in FP64
# and 2^29 times that in FP32, rounded
TOL = {FP64: 1e-13, FP32: 2e-5}


def _rhs(nx, ny, prec, flag):
    os.environ["S2D_GENERIC_KERNELS"] = flag
    try:
        s = Spectral2D(nx, ny, precision=prec)
    finally:
        os.environ.pop("S2D_GENERIC_KERNELS", None)
    s.set_field("w", np.random.default_rng(nx + ny).standard_normal(2 * s.cISize * s.nyG))
    s.TransformC2R("w")  # a real field, so that the mirrored modes agree
    s.TransformR2C("w")
    s.ComputePsi()
    out = []
    for _ in range(2):
        s.copy_field("w", "wS")
        s.copy_field("psi", "psiS")
        s.ComputeRHS(1e-4, "u", "v", "wS", "psiS", "dW")
        out.append(s.get_field("dW"))
    s.close()
    assert np.array_equal(*out)
    return out[0]


@pytest.mark.parametrize("prec", [FP64, FP32])
@pytest.mark.parametrize("nx,ny", [(64, 32), (96, 64), (128, 48), (192, 144), (256, 512),
                                   (256, 768), (384, 256), (512, 256), (512, 384), (512, 1024),
                                   (512, 2048)])
def test_rows_match_the_runtime_plans(nx, ny, prec):
    print(f"[rhs rows] {nx}x{ny} precision={prec}", flush=True)
    a, b = _rhs(nx, ny, prec, "0"), _rhs(nx, ny, prec, "1")
    assert np.isfinite(a).all()
    assert np.linalg.norm(a - b) <= TOL[prec] * np.linalg.norm(b)
