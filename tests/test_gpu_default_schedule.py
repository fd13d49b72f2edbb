"""The default schedule's choices on the GPU: calls that replay a captured
step and calls that launch theirs one by one give the same bits, and the
default kernels of the largest sizes agree with their alternatives."""
import numpy as np
import pytest

from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


def _run(N, prec, sched, calls, graph):
    s = Spectral2D(N, precision=prec)
    s.SetTurbulence(9, max(2.0, N / 32), 0.5)
    s.set_schedule(*sched, step_graph=graph)
    for k in calls:
        s.rk3_steps(k, 1e-4, 0.0, 0.5)
    w = s.get_field("w")
    s.close()
    return w


@pytest.mark.parametrize("N,prec", [(64, FP32), (96, FP64), (512, FP64), (1024, FP32)])
def test_short_and_long_calls_equal_eager(N, prec):
    """Replays (1 and 3 steps), long calls (4 and 5) and replays after them."""
    calls = (1, 3, 4, 5, 2)
    print(f"[schedule] N={N} precision={prec} calls={calls}", flush=True)
    assert np.array_equal(_run(N, prec, (0, 0, 0), calls, True),
                          _run(N, prec, (0, 0, 0), calls, False))


@pytest.mark.parametrize("N,prec,sched", [(1024, FP32, (2, 0, 0)), (2048, FP32, (2, 0, 0)),
                                          (2048, FP64, (0, 2, 0))])
def test_default_agrees_with_its_alternative(N, prec, sched):
    """Same mathematics, other order of rounding: the variants' tolerances
    (1e-12, 1e-5), and not the same kernel (the bits differ)."""
    print(f"[schedule] N={N} precision={prec} default vs {sched}", flush=True)
    a, b = (_run(N, prec, s, (2,), False) for s in ((0, 0, 0), sched))
    err = float(np.linalg.norm(a - b) / np.linalg.norm(b))
    assert 0 < err < (1e-12 if prec == FP64 else 1e-5)
