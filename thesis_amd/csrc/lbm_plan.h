// How many steps a launch, or a barrier of the batch, takes: rules on sizes, from
// measured costs (MI355X, microseconds).  Host code without the runtime, so that
// tests/test_plan.py holds them against measured times on any machine.
#pragma once
#include <algorithm>
#include <cstddef>

namespace lbm {

inline long squares_of(int nx, int ny, int side) { return (long)((nx + side - 1) / side) * ((ny + side - 1) / side); }
inline long rounds_of(long n, long width) { return (n + width - 1) / width; }

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
        const double c = bar + single + (t > 1 ? (double)full * phase(t) + phase(rest - full * t) : (double)rest * single);
        if (t == 1) least = 0.95 * c;
        else if (c <= least) { least = c; best = BatchPlan{t, sq, (int)g}; }
    }
    return best;
}

}  // namespace lbm
