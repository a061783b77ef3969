// Which of two timed plans takes which run lengths (host only).
//
// Tiles stage a pass of up to 256 steps once and compute more per step than the
// column kernels, which run 4 or 5 steps per pass, so which is faster depends
// on the run's length: FP32 [2048][1024][512], ms, strips / column pair: 20
// steps 8.5 / 7.6, 50 steps 17.8 / 18.8, 200 steps 63.7 / 75.3.  The autotuner
// times the fastest of either kind at these lengths.
#pragma once

#include <algorithm>
#include <cmath>

namespace bkma {

constexpr unsigned long long kRunSteps[] = {1, 2, 4, 5, 8, 12, 20, 32, 48, 96};
constexpr int kRuns = sizeof(kRunSteps) / sizeof(kRunSteps[0]);

// Runs of up to `up_to` steps take the one kind, longer runs the other.
struct RunChoice {
    bool tile_short = false, tile_long = false;
    unsigned long long up_to = 0;
};

// The choice between a tile plan (t, time of a run of kRunSteps[i] steps) and
// another (o).  Where the results depend on the steps per pass (FP32) and the
// two differ in them, one plan has to take every run beyond a pass of both,
// `shared` steps: the one with the smaller geometric mean from 8 steps on.
// Runs below, and all runs where the results are the same, are split where the
// least is lost over the measured lengths; a split has to gain 2%.
inline RunChoice choose_runs(const float *t, const float *o, unsigned long long shared) {
    auto loss = [&](int i, bool tile) { return std::log((tile ? t[i] : o[i]) / std::min(t[i], o[i])); };
    bool may[2] = {true, true};  // the other plan, the tiles: take the long runs
    if (shared < kRunSteps[kRuns - 1]) {
        double lt = 0, lo = 0;
        for (int i = 0; i < kRuns; ++i)
            if (kRunSteps[i] >= 8) {
                lt += loss(i, true);
                lo += loss(i, false);
            }
        may[lt < lo ? 0 : 1] = false;
    }
    RunChoice best;
    double least = 1e30;
    for (int tile = 0; tile < 2; ++tile) {
        if (!may[tile]) continue;
        for (int k = 0; k < kRuns && (k == 0 || kRunSteps[k - 1] <= shared); ++k) {  // lengths [0, k): the other kind
            double sum = k ? 0.02 : 0.0;
            for (int i = 0; i < kRuns; ++i) sum += loss(i, (i >= k) == (tile != 0));
            if (sum >= least) continue;
            least = sum;
            best.tile_long = tile != 0;
            best.tile_short = (k == 0) == best.tile_long;
            best.up_to = k ? kRunSteps[k - 1] : 0;
        }
    }
    return best;
}

}  // namespace bkma
