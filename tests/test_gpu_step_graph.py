"""The step_graph setting on the GPU: what the schedule calls report, that
every setting gives the same bits, and that the tuner leaves lines measured
under another meaning of its fields alone."""
import json

import numpy as np
import pytest

from spectral2d_amd.spectral import FP32, FP64, Spectral2D

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,prec", [(64, FP64), (512, FP32), (1024, FP64)])
def test_settings_give_the_same_bits(N, prec):
    print(f"[step_graph] N={N} precision={prec}", flush=True)
    out = []
    for setting in (None, True, False, 2, 3):
        s = Spectral2D(N, precision=prec)
        assert s.get_schedule()["step_graph"] == 2
        if setting is not None:
            s.set_schedule(step_graph=setting)
            assert s.get_schedule()["step_graph"] == int(setting)
        s.SetTurbulence(9, max(2.0, N / 32), 0.5)
        for k in (1, 1, 6, 2, 5):
            s.rk3_steps(k, 1e-4, 0.0, 0.5)
        out.append(s.get_field("w").copy())
        s.close()
    for w in out[1:]:
        assert np.array_equal(w, out[0])


@pytest.mark.parametrize("N,prec", [(64, FP32), (96, FP64), (512, FP64)])
def test_changing_dt(N, prec):
    """New, repeated and earlier time steps and viscosities, launched and
    replayed, in calls of one and more steps."""
    print(f"[step_graph] changing dt N={N} precision={prec}", flush=True)
    dt = 0.05 / N
    out = []
    for setting in (2, True, False):
        s = Spectral2D(N, precision=prec)
        s.set_schedule(step_graph=setting)
        s.SetTurbulence(9, max(2.0, N / 32), 0.5)
        for k, f, nu in ((1, 1, 1), (1, 2, 1), (1, 3, 1), (1, 3, 1), (1, 3, 1), (2, 1, 1), (1, 3, 1),
                         (5, 4, 1), (1, 4, 1), (1, 4, 2), (1, 4, 2), (1, 4, 2)):
            s.rk3_steps(k, nu * 1e-4, f * dt)
        out.append(s.get_field("w").copy())
        assert s.get_time()[1] == 17
        s.close()
    assert np.array_equal(out[0], out[2]) and np.array_equal(out[1], out[2])


def test_tuned_setting_and_former_cache_lines(tmp_path):
    cache, old = str(tmp_path / "tune.jsonl"), str(tmp_path / "old.jsonl")
    s = Spectral2D(512, precision=FP64)
    s.SetTurbulence(3, 10.0, 0.5)
    r = s.tune(1e-4, cfl=0.5, cache=cache)
    print(f"[step_graph] tuned: {r}", flush=True)
    assert r["step_graph"] in (0, 1, 3) and s.get_schedule()["step_graph"] == r["step_graph"]
    entry = json.loads(open(cache).read())
    assert entry["step_graph"] == r["step_graph"]
    # a line from when step_graph 0 meant no replays of long calls
    line = dict(entry, key=entry["key"][: entry["key"].rindex("/")], step_graph=0, pass_b=1)
    open(old, "w").write(json.dumps(line) + "\n")
    t = Spectral2D(512, precision=FP64)
    u = t.tune(1e-4, cfl=0.5, cache=old, cache_only=True)
    assert u["from_cache"] == 0 and u["step_graph"] == 2 and u["pass_b"] == 0
    u = t.tune(1e-4, cfl=0.5, cache=cache, cache_only=True)
    assert u["from_cache"] == 1 and u["step_graph"] == r["step_graph"]
    s.close()
    t.close()
