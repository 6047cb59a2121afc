// How the kernel for short causal windows (fmha_window.hip.h) cuts the rows of a (batch, kv head) pair into runs.
#pragma once

#include <cstdint>

namespace singe_hip {

// Steps to a run: runs of one length that fill the chip's places in whole rounds, a run's first keys counted as a step.  Runs
// from one up to four to a place; what they cost only changes where their length does, so one candidate to a length is looked
// at (64 / 8 heads x 8192: 31 in place of 256, 0.5 us a call and not 2.9; one pair of 2048 steps: 89, 1.4 and 22.6).
constexpr uint64_t window_run_steps(uint64_t steps, uint64_t pairs, uint64_t places) {
    uint64_t best = ~0ull, best_steps = steps;
    for (uint64_t runs = 1; runs <= steps && (runs - 1) * pairs <= 4 * places;) {
        const uint64_t run_steps = (steps + runs - 1) / runs;
        const uint64_t rounds = (pairs * ((steps + run_steps - 1) / run_steps) + places - 1) / places, cost = rounds * (run_steps + 1);
        if (cost < best) best = cost, best_steps = run_steps;
        if (run_steps == 1) break;
        runs = (steps + run_steps - 2) / (run_steps - 1);  // the fewest runs that are shorter
    }
    return best_steps;
}

}  // namespace singe_hip
