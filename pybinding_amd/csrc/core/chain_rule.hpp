// When a run takes the chained recurrence (several Chebyshev steps per launch).
#pragma once
#include <algorithm>
#include <cstdint>

namespace kpmx {

// Estimated microseconds of a single step on vw columns of n rows of `scalar` bytes: three passes at
// 5.6 TB/s, no less than a launch.
inline double single_step_us(int64_t n, int64_t vw, size_t scalar) {
    return std::max(5.5, 3.0 * (double)n * (double)vw * (double)scalar / 5.6e6);
}

// Whether a run of `steps` single steps of single_us each pays for a plan in its first pass.  A plan
// with its buffers costs about 0.13 ms and 2 us per thousand rows up to half a millisecond; chained steps
// save 60 % of launch-bound steps and 40 % or more of the others.  First passes measured with a plan and
// with single steps: 15 k sites, 80 steps 0.36 and 0.40 ms; 61 k sites, 80 steps 0.48 and 0.52 ms; but
// 180 k sites, 10 vectors, 50 steps 1.18 and 0.99 ms.  Below 0.4 ms nothing is tried.  What ran
// before does not enter, so the same call takes the same form (but for calls that build no plans and use
// one that is there, and for plans that there was no memory for).
inline bool chain_pays(int64_t n, double single_us, int64_t steps) {
    const double plan_us = 130 + std::min(2e-3 * (double)n, 500.0);
    return single_us * (double)steps >= std::max(400.0, plan_us / (single_us <= 5.5 ? 0.6 : 0.4));
}

// The same for a batch of n rows in column groups of `cols` vectors.  A plan takes 0.1 ms and 0.22 us per
// thousand rows, and 45 ns per thousand rows and column of the group (more tiles, larger vectors: their
// allocation is most of it); chained steps save more than half of launch-bound steps (two launches, 10 us)
// and, of the three passes that single_us counts and the walkers' steps exceed, 80 % or more.  First
// passes measured with walkers and with a plan: 10 systems of 100 k sites, 8 vectors, 20 steps 1.44 and 1.53 ms,
// 30 steps 2.04 and 1.75 ms; 4 vectors, 25 steps 1.14 and 1.32 ms, 40 steps 1.61 and 1.59 ms; 10 systems of 10 k
// sites, 40 steps 0.65 and 0.58 ms.
inline bool batch_chain_pays(int64_t n, int cols, double single_us, int64_t steps) {
    const double plan_us = 100 + (double)n * (0.22e-3 + 0.045e-3 * cols);
    return single_us * (double)steps >= std::max(400.0, plan_us / (single_us <= 10 ? 0.55 : 0.8));
}

}  // namespace kpmx
