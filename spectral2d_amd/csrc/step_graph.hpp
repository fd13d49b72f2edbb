// step_graph.hpp -- which calls of the fused step replay a captured step
// (hipGraph) and which launch their steps' nine kernels one by one. The bits
// are the same either way.
//
// A replay starts about 10 us sooner than nine launches do, but leaves about
// 4.5 us of gap before the next replay (launches that run ahead of the device
// leave none): us per call of 1 / 2 / 8 steps, replayed / launched, FP64:
// N = 96 79 / 90, 136 / 144, 474 / 461; N = 512 121 / 129, 218 / 223,
// 803 / 785; N = 1024 (10 steps) 1672 / 1627. A step at N = 64 (44 us) is as
// short as its nine launches take on a slow host (8 steps 398 / 418, on a fast
// one 400 / 386).
#pragma once

namespace s2d {

// s2d_schedule::step_graph
enum StepGraph { STEP_LAUNCH = 0, STEP_REPLAY = 1, STEP_DEFAULT = 2, STEP_REPLAY_SHORT = 3 };

inline int step_graph_setting(int value)
{
    return value == STEP_LAUNCH || value == STEP_DEFAULT || value == STEP_REPLAY_SHORT ? value
                                                                                      : STEP_REPLAY;
}

// Whether a call of nsteps steps at padded size np replays under a setting:
// all, those of up to three steps, or (by default) those and, below Np = 144,
// all.
inline bool step_replays(int setting, int nsteps, int np)
{
    return setting == STEP_REPLAY || (setting != STEP_LAUNCH && nsteps < 4) ||
           (setting == STEP_DEFAULT && np < 144);
}

// What a captured step has baked in.
struct StepArgs {
    double nu = 0.0, dt = 0.0, cfl = 0.0;
    const void *forcing = nullptr; // its buffer, or null
    int var[3] = {-1, -1, -1};     // the passes' variants (none yet)

    bool operator==(const StepArgs &o) const
    {
        return nu == o.nu && dt == o.dt && cfl == o.cfl && forcing == o.forcing &&
               var[0] == o.var[0] && var[1] == o.var[1] && var[2] == o.var[2];
    }
};

// Whether a call that may replay does: a step captured with its arguments is
// there, or a capture pays, for four steps or for a call like the last one. A
// program with another dt at every step (the CFL step of its own making) would
// capture at every call: N = 64 / 96 / 512 / 1024 FP64 126 / 137 / 172 / 249 us
// a call, launched 74 / 75 / 108 / 181 (the same dt replayed 63 / 76 / 115 /
// 194).
inline bool step_capture_pays(int nsteps, const StepArgs &call, const StepArgs &captured,
                              const StepArgs &last)
{
    return call == captured || call == last || nsteps >= 4;
}

// The setting a measurement picks: replays of all calls where eight steps take
// least so, else replays of the short calls where one step with its wait does.
inline int step_graph_choice(double launch8, double replay8, double launch1, double replay1)
{
    return replay8 < launch8 ? STEP_REPLAY : replay1 < launch1 ? STEP_REPLAY_SHORT : STEP_LAUNCH;
}

} // namespace s2d
