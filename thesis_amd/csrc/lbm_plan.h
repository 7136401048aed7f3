// How many steps a launch, or a barrier of the batch, takes: rules on sizes, from
// measured costs (MI355X, microseconds).  Host code without the runtime, so that
// tests/test_plan.py holds them against measured times on any machine.
#pragma once
#include <algorithm>
#include <cmath>
#include <cstddef>

namespace lbm {

inline long squares_of(int nx, int ny, int side) { return (long)((nx + side - 1) / side) * ((ny + side - 1) / side); }
inline long rounds_of(long n, long width) { return (n + width - 1) / width; }

// Steps of a launch: at most `most` (1: one launch a step throughout), and at least
// `least`; what a call leaves over below that goes one launch a step.
struct StepPlan {
    int most, least;
};
// The plan with the least time a step among launches of up to `top` steps, where
// launch(t) < `win` t single; single: one launch for one step.
template <class Launch> inline StepPlan step_plan(int top, double single, double win, Launch launch) {
    StepPlan p{1, 2};
    double best = win * single;
    for (int t = 2; t <= top; ++t)
        if (launch(t) / t < best) { best = launch(t) / t; p.most = t; }
    while (p.least < p.most && launch(p.least) >= win * single * p.least) ++p.least;
    return p;
}

// D2Q9 lattice of nx x ny nodes, nf of them not solid, FP64 or FP32 (lbm_multi2.hip).
//
// One step takes 5.2 us and 24 ns a thousand fluid nodes in FP64, 15.5 in FP32 (256 x
// 64 5.5 us, 1400 x 700 29.6 / 20.8, 2048 x 2048 105 / 68, 0.4 of them fluid 46 / 30).
// A launch of t steps works on the whole box, solid or not: squares of 32 - 2t inner
// nodes a side.  Up to 256 of them have a CU each and cost 7 + 1.65 t us (FP32 5.6 +
// 1.1 t), more go in rounds of 256 of 6 + 1.25 t us (FP32 2.6 + 0.65 t and 4 for the
// launch); with MRT a quarter more.  Measured a step at t = 1, 2, 3, 4, 5, 6, 8, 12:
// FP64 256 x 64 5.5, 6.0, 4.0, 3.5, 3.2, 3.0, 2.5, 2.1 (12 chosen), 500 x 120 6.2, 5.0,
// 4.2, 3.6, 3.3, 3.0, 2.7, 6.0 (8), 1021 x 256 10.8, 9.5, 7.5, 6.3, 7.4, 7.6, 8.6, 22 (4);
// 2048 x 2048 FP64 105, 99, 82, 72, 75, 78, 106, 313 (4), of which 0.6 fluid 64, 84, 74,
// 74 (1), FP32 of which 0.4 fluid 30, 39, 35, 36 (1).
inline StepPlan flow2_plan(int nx, int ny, size_t nf, bool f64, bool mrt) {
    const double single = 5.2 + (f64 ? 24e-6 : 15.5e-6) * (double)nf;
    return step_plan(14, single, 1.0, [&](int t) {
        const long sq = squares_of(nx, ny, 32 - 2 * t), r = rounds_of(sq, 256);
        const double c = sq <= 256 ? (f64 ? 7.0 + 1.65 * t : 5.6 + 1.1 * t)
                         : f64     ? (double)r * (6.0 + 1.25 * t)
                                   : 4.0 + (double)r * (2.6 + 0.65 * t);
        return mrt ? 1.25 * c : c;
    });
}

// Periodic two-phase D2Q9 box, FP64 or FP32, ho: 24-point stencil, enh: enhanced model
// (lbm_cg.hip).
//
// One step is a launch of tiles of 32 x 16 nodes: up to 256 of them 8.2 us (FP32 6.6),
// more in rounds of 512 of 18 us (10.5), where there are many 7.4 us (4.45) for each
// 256; a twentieth more with the 24-point stencil.  A launch of t steps is one of squares
// of 32 - 2 halo inner nodes, halo = t (1 + H) - 1, and costs, where every square has a
// CU of its own (up to 256), 6 + 2.6 t us (FP32 5 + 2 t); beyond, each round of 256
// squares 14.5 + 0.9 t us, with the 24-point stencil 12.6 + 0.7 t, in FP32 each round of
// 512 (two a CU) 12.4 + t us and the launch 4, with the 24-point stencil 12 + 0.9 t and
// 2; the enhanced model adds 6 %, FP64 with the 24-point stencil 12 %.  Measured per step
// at t = 1, 2, 3, 4, 5, 6, 8-point stencil: FP64 250 x 187 8.2, 6.7, 5.8, 5.1, 4.8, 7.5
// (5 chosen), 512 x 512 17.8, 15.6, 16.6, 18.1, 23.0, 37.4 (2), 1024 x 1024 69, 58, 54,
// 59, 84, 140 (3), 2048 x 2048 245, 232, 205, 223, 317, 540 (3); FP32 512 x 512 10.4, 8.9,
// 9.1, 10.2, 12.8, 19.7 (2), 1024 x 1024 43, 31, 26, 31, 45, 71 (3); 24-point FP64 512 x
// 512 19.2, 20.0, 19.5, 41.7 (1), with the enhanced model 19.0, 21.9, 22.0 (1), 1024 x
// 1024 76, 66, 75 (2), 2048 x 2048 enhanced 258, 278, 329 (1).
inline StepPlan cg2_plan(int nx, int ny, bool ho, bool enh, bool f64) {
    const double x = (double)((nx + 31) / 32) * ((ny + 15) / 16) / 256.0;
    double single = f64 ? 8.2 : 6.6;
    if (x > 1.0)
        single = f64 ? std::min(18.0 * std::ceil(x / 2), 10.0 + 7.4 * x)
                     : std::min(10.5 * std::ceil(x / 2), 6.0 + 4.45 * x);
    if (ho) single *= f64 ? 1.05 : 1.08;
    return step_plan(ho ? 5 : 8, single, 1.0, [&](int t) {
        const long sq = squares_of(nx, ny, 32 - 2 * (t * (ho ? 3 : 2) - 1));
        const double c = sq <= 256 ? (f64 ? 6.0 + 2.6 * t : 5.0 + 2.0 * t)
                         : !f64    ? (ho ? 2.0 + (double)rounds_of(sq, 512) * (12.0 + 0.9 * t)
                                         : 4.0 + (double)rounds_of(sq, 512) * (12.4 + 1.0 * t))
                         : ho      ? (double)rounds_of(sq, 256) * (12.6 + 0.7 * t)
                                   : (double)rounds_of(sq, 256) * (14.5 + 0.9 * t);
        return enh ? (ho && f64 ? 1.12 : 1.06) * c : c;
    });
}

// Steps a barrier of a batch that checks its residuals every `every` steps, the
// squares of all instances at that count, and the workgroups of the grid.
//
// A barrier costs 0.1 us a workgroup, and the check's step has two; a single step
// 6.5 us for each round of tiles, a phase of t steps 6 + 1.25 t us for each round of
// squares with a frame of t.  More squares than tiles make the grid, and so every
// barrier, larger, and steps that the check leaves over still pay for the whole frame:
// small batches with frequent checks keep one step a barrier.  Measured a step, one
// step / four / eight a barrier: 256 x 64 checked every step 12 / 14 / 19 us, every 8
// 8.0 / 5.0 / 4.7, every 100 7.3 / 3.2 / 2.6; eight of them 35 / 57 / 57, 21.7 / 17.6 /
// 14.1, 19.8 / 11.3 / 8.0; 64 channels of 3.65 M nodes every 3 160 / 137 (two: 130) /
// 180, every 100 131 / 64 / 81.  Several steps have to be expected a twentieth faster.
struct BatchPlan {
    int halo;
    long squares;
    int grid;
};
template <class Inst>   // of members nx and ny
inline BatchPlan batch_plan(const Inst* inst, int n, long tiles, int most_blocks, long every) {
    BatchPlan best{1, 0, (int)std::min<long>(tiles, most_blocks)};
    double least = 0;
    for (int t = 1; t <= 10 && t <= std::max(1l, every - 1); ++t) {
        long sq = 0;
        for (int k = 0; k < n && t > 1; ++k) sq += squares_of(inst[k].nx, inst[k].ny, 32 - 2 * t);
        if (sq > 0x7FFFFFFF) continue;
        const long g = std::min<long>(std::max(tiles, sq), most_blocks);
        const double bar = 0.1 * (double)g, single = bar + 6.5 * (double)rounds_of(tiles, g);
        auto phase = [&](long s) {
            return s < 2 ? (double)s * single : bar + (double)rounds_of(sq, g) * (6.0 + 1.25 * (double)s);
        };
        const long rest = every - 1, full = t > 1 ? rest / t : 0;
        const double c =
            bar + single + (t > 1 ? (double)full * phase(t) + phase(rest - full * t) : (double)rest * single);
        if (t == 1) least = 0.95 * c;
        else if (c <= least) { least = c; best = BatchPlan{t, sq, (int)g}; }
    }
    return best;
}

}  // namespace lbm
