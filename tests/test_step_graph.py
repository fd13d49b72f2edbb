"""step_graph.hpp: which calls replay a captured step, and what a measurement
chooses (host code)."""
import subprocess

from spectral2d_amd import build

PROGRAM = r"""
#include "step_graph.hpp"
#include <cstdio>
#include <initializer_list>
using namespace s2d;

static int bad = 0;
#define CHECK(x) if (!(x)) std::printf("%s\n", #x), ++bad

int main()
{
    for (int np : {48, 96, 144, 768, 1536, 3072})
        for (int n = 1; n < 40; ++n) {
            CHECK(step_replays(STEP_REPLAY, n, np));
            CHECK(!step_replays(STEP_LAUNCH, n, np));
            CHECK(step_replays(STEP_REPLAY_SHORT, n, np) == (n <= 3));
            CHECK(step_replays(STEP_DEFAULT, n, np) == (n <= 3 || np < 144));
        }
    for (int v = 0; v < 4; ++v) CHECK(step_graph_setting(v) == v);
    CHECK(step_graph_setting(4) == STEP_REPLAY && step_graph_setting(-1) == STEP_REPLAY);
    // launched over 8 steps, replayed over 8, launched single, replayed single
    CHECK(step_graph_choice(2.0, 1.0, 1.0, 2.0) == STEP_REPLAY);
    CHECK(step_graph_choice(1.0, 2.0, 2.0, 1.0) == STEP_REPLAY_SHORT);
    CHECK(step_graph_choice(1.0, 2.0, 1.0, 2.0) == STEP_LAUNCH);
    CHECK(step_graph_choice(1.0, 1e300, 1e300, 1e300) == STEP_LAUNCH); // no graph to replay
    // a capture pays for a call like the last one or the captured one, or for four steps
    const StepArgs none;
    StepArgs a, b;
    a.nu = 1e-4, a.dt = 1e-3, a.var[0] = a.var[1] = a.var[2] = 0;
    b = a, b.dt = 2e-3;
    for (int n = 1; n < 8; ++n) {
        CHECK(step_capture_pays(n, a, none, none) == (n >= 4));
        CHECK(step_capture_pays(n, b, none, a) == (n >= 4));
        CHECK(step_capture_pays(n, b, a, a) == (n >= 4));
        CHECK(step_capture_pays(n, a, none, a));
        CHECK(step_capture_pays(n, a, a, b));
    }
    for (int k = 0; k < 6; ++k) { // every argument counts
        b = a;
        if (k == 0) b.nu = 0.0;
        else if (k == 1) b.cfl = 0.5;
        else if (k == 2) b.forcing = &b;
        else b.var[k - 3] = 1;
        CHECK(!(a == b) && !step_capture_pays(1, a, b, b));
    }
    return bad;
}
"""


def test_step_graph(tmp_path):
    src, exe = tmp_path / "step_graph.cpp", tmp_path / "step_graph"
    src.write_text(PROGRAM)
    r = subprocess.run(["g++", "-std=c++17", "-I", build.CSRC, str(src), "-o", str(exe)],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
