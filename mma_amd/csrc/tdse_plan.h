// How the resident TDSE kernels cover a grid (host only; tdse_resident.hip runs it).
#pragma once
#include <algorithm>
#include <cmath>

#include "tdse_internal.h"

// The largest grid they take, and the largest whose tables they read: byte offsets in a table, a window's buffer or
// a tiled state are 32-bit.
inline constexpr int kResidentPoints = (1 << 27) - (1 << 16);

// How the resident kernel covers nx points whose carries reach `reach` points: lanes of C points,
// waves and windows (TdseResident).  A function of the geometry alone, so an instance's results do
// not depend on the batch around it.  Costs in units of an instruction per lane and step: 55 per
// point and 330 for the scans, the phase and the sums (1210, 1650, 2090; a step of 8 full waves takes 5.6, 7.3 and 9.7 us).
//   One window: (C, waves) by the work of a CU per instance and step (8 waves fit one, so a CU holds
//   8 / waves workgroups), and within a quarter of the least by a step's latency: 16 points x 8 waves
//   rather than 32 x 4 for 8001 points, 18 % more work in half the time per step (200 steps of 256 instances 1.19 ms
//   against 1.38; with more than one a CU the work decides: 512 2.44 against 2.14, 2048 9.0 against 8.1).
//   That ends at 8177, 12265 and 16353 points: a grid may start up to C - 1 points into its first lane.
//   Several (the grid is larger than 8 waves x 32 lanes' points): `steps` steps between a window's load
//   and store cost a halo of steps x reach points at each inner edge; loading, b included, and
//   storing cost about 60 per point.
inline bool plan_resident(int nx, int reach, TdseResident &R)
{
    static const int kChunks[3] = {16, 24, 32};
    const int margin = reach + 2;  // per step: both recurrences, and the right-hand side's neighbours
    R.chunk = 0;
    if (nx > kResidentPoints) return false;
    auto per_step = [](int C) { return 55.0 * C + 330.0; };
    double least = INFINITY;
    for (int pass = 0; pass < 2; pass++) {
        double best = INFINITY;
        for (int C : kChunks) {
            if (reach > 16 * C) continue;
            const int waves = (nx + C - 1 + 64 * C - 1) / (64 * C);
            if (waves > TDSE_MAX_WAVES) continue;
            const double cost = per_step(C) / (TDSE_MAX_WAVES / waves);
            if (pass == 0) {
                least = std::min(least, cost);
            } else if (cost <= 1.25 * least && per_step(C) < best) {
                best = per_step(C);
                R.chunk = C;
                R.waves = waves;
            }
        }
    }
    R.reach = reach;
    R.windows = 1;
    R.steps = TDSE_RES_RING;
    R.stride = R.halo = 0;
    if (R.chunk) return true;
    double best = INFINITY;
    for (int C : kChunks) {
        if (reach > 16 * C) continue;
        const int lanes = 64 * TDSE_MAX_WAVES, total = (nx + C - 1 + C - 1) / C;
        for (int T = TDSE_RES_RING; T >= 1; T--) {
            const int halo = (T * margin + C - 1) / C, stride = lanes - 2 * halo;
            if (stride < 64) continue;
            const int n = 1 + (total - lanes + stride - 1) / stride;
            const double cost = n * (T * per_step(C) + 60.0 * C) / T;
            if (cost < best) {
                best = cost;
                R.chunk = C;
                R.waves = TDSE_MAX_WAVES;
                R.windows = n;
                R.steps = T;
                R.stride = stride;
                R.halo = halo;
            }
        }
    }
    return R.chunk > 0;
}

// Entries of a resident table of nx points in lanes of C: whole tiles, one zero chunk at least.
inline long long resident_entries(int nx, int C) { return (long long)(((nx + C - 1) / C + 1 + 63) / 64) * 64 * C; }

// Points before a run of pivots from the double ones, whose error of 1e-16 decays by rho^2 a point: to
// below 1e-20 (rho^reach = 1e-17).
inline int resident_warm(int reach) { return reach / 8 + 4; }

// The windows of one instance alone: lanes of 16 points (24 where carries reach further), four waves, one
// per SIMD, a window; as many steps per launch as leave at most kOneWindows windows.  With 16001
// points at dt 0.25, dx 0.1 (carries reach 151): 30 windows of 4096 points, 12 steps a launch.
inline constexpr int kOneWindows = 64;
inline bool plan_one(int nx, int reach, TdseResident &R)
{
    R.chunk = 0;
    if (nx > kResidentPoints || reach > 16 * 24) return false;
    const int C = reach <= 16 * 16 ? 16 : 24, total = (nx + C - 1 + C - 1) / C, margin = reach + 2;
    R.chunk = C;
    R.reach = reach;
    R.windows = 1;
    R.steps = TDSE_RES_RING;
    R.stride = R.halo = 0;
    R.waves = std::min(TDSE_ONE_WAVES, (total + 63) / 64);
    const int lanes = 64 * TDSE_ONE_WAVES;
    if (total <= lanes) return true;
    for (int T = TDSE_RES_RING; T >= 1; T--) {
        const int halo = (T * margin + C - 1) / C, stride = lanes - 2 * halo;
        if (stride < 1) continue;
        R.windows = 1 + (total - lanes + stride - 1) / stride;
        R.steps = T;
        R.stride = stride;
        R.halo = halo;
        if (R.windows <= kOneWindows || T == 1) return true;
    }
    return true;
}
