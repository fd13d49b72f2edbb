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

// The setting a measurement picks: replays of all calls where eight steps take
// least so, else replays of the short calls where one step with its wait does.
inline int step_graph_choice(double launch8, double replay8, double launch1, double replay1)
{
    return replay8 < launch8 ? STEP_REPLAY : replay1 < launch1 ? STEP_REPLAY_SHORT : STEP_LAUNCH;
}

} // namespace s2d
