"""Diagnostics of a batch of more runs than a reduction has blocks."""
import numpy as np
import pytest

from spectral2d_amd.ensemble import Ensemble
from spectral2d_amd.spectral import FP32, Spectral2D

pytestmark = pytest.mark.gpu


def test_runs_equal_the_runs_alone():
    """600 runs at 512^2 (1155 blocks' worth of modes each): the same values,
    bitwise, as the runs by themselves."""
    N, M = 512, 600
    s = Spectral2D(N, precision=FP32)
    e = Ensemble([N] * M, FP32)
    for r in (0, 311, M - 1):
        s.SetTurbulence(r, 6.0, 0.5)
        e.set_vorticity(r, s.get_field("w"))
    got = e.diagnostics()
    for r in (0, 311, M - 1):
        s.SetTurbulence(r, 6.0, 0.5)
        alone = s.diagnostics()
        print(f"[diag] run {r}: {got[r]} alone {alone}", flush=True)
        assert got[r] == alone
    assert got[1]["tke"] == 0.0 and got[1]["max_abs_w"] == 0.0
    e.close()
    s.close()
