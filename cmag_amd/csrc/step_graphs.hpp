// step_graphs.hpp - the captured steps run() launches: a graph of one step, and
// one of several.
//
// A graph launch costs the host and the gap to the next one what two or three
// of a step's six or seven kernels do, so steps are launched several at a time
// once a second run() in a row asks for as many: the first pass captures one
// step only, and counts that change never capture again (a larger graph
// replaces a smaller one, so MANY_STEPS - 1 times at most).  The capture costs
// the second run() of a system that stands still 75 to 150 us and saves every
// later one 65 (10 steps) to 110 us (16); behind queued work, as between a
// rollout's checkpoints, it hides (whole rollouts of 2 x 4 to 10 x 20 steps with
// 2,000 and 17,000 particles, graphs captured anew in each: 0.4 to 10 % faster
// than one step at a time).
#pragma once

#include <cstdint>

namespace cmag {

template <typename Graph>
struct StepGraphs {
    static constexpr uint32_t MANY_STEPS = 16;
    Graph one{}, many{};
    uint32_t many_steps = 0, last_run = 0;
    uint32_t refused = 0;  // bit k: a capture of k steps failed

    // in front of a run of `steps`: capture(steps, &graph) -> 0 or an error,
    // drop(graph) ends one that may be running.  Fails only without the one-step
    // graph: where several steps cannot be captured, the run goes step by step
    // (and the count is not tried again)
    template <typename Capture, typename Drop>
    int prepare(uint32_t steps, Capture&& capture, Drop&& drop) {
        if (!one) {
            const int rc = capture(1u, &one);
            if (rc != 0) return rc;
        }
        const uint32_t want = steps < MANY_STEPS ? steps : MANY_STEPS;
        const bool again = want == last_run;
        last_run = want;
        if (!again || want < 2 || want <= many_steps || (refused >> want & 1u)) return 0;
        Graph g{};
        if (capture(want, &g) != 0) {
            refused |= 1u << want;
            return 0;
        }
        if (many) drop(many);
        many = g;
        many_steps = want;
        return 0;
    }

    // the next launch of a run with `left` steps to go: its graph and its steps
    Graph next(uint32_t left, uint32_t& steps) const {
        const bool several = many && left >= many_steps;
        steps = several ? many_steps : 1u;
        return several ? many : one;
    }
};

}  // namespace cmag
