// How a session replays its captured step: one by one, or, once that is worth it, several per replay.
#ifndef NATIVE_HIP_STEP_REPLAYS_H
#define NATIVE_HIP_STEP_REPLAYS_H

#include <cstddef>

namespace nh {

// The graph of several steps is a gain only: nothing needs it, and what it costs has to come back.
class StepReplays {
public:
    static constexpr size_t STEPS = 8;  // per replay of the longer graph

    // nodes: of the graph of one step.  Between two replays the GPU waits 4 to 5 us for the next one's first packet; a node
    // of the longer graph costs the host 2.7 to 3.9 us (one session of 4 layers of an 8B model: 22 nodes, 0.55 ms; of 32: 162,
    // 3.5; eight sequences: 39 and 291, 0.94 and 7.7).
    void set_nodes(size_t nodes) { worth_ = STEPS * nodes * MAKE_NS / LOST_NS; }
    size_t worth() const { return worth_; }

    // n steps: many() is STEPS of them, one() a single one; 0 on success, else what failed returned.
    template <typename One, typename Many> int run(size_t n, One &&one, Many &&many) {
        while (n > 0) {
            const bool enough = n >= STEPS, together = made_ && enough;
            if (const int rc = together ? many() : one()) return rc;
            if (enough && !made_) missed_++;
            n -= together ? STEPS : 1;
        }
        return 0;
    }
    // To be called when a run has been enqueued: makes the longer graph (0 on success) once the single replays that it
    // would have taken have lost what it costs, so that a session which ends before never pays for it, and neither does one
    // whose runs are short.  It is tried once: a session goes on with single replays if it cannot be made.
    template <typename Make> void offer(Make &&make) {
        if (made_ || refused_ || missed_ == 0 || missed_ < worth_) return;
        made_ = make() == 0;
        refused_ = !made_;
    }

private:
    static constexpr size_t MAKE_NS = 3300, LOST_NS = 4500;  // per node of the longer graph, per single replay
    size_t worth_ = 0, missed_ = 0;
    bool made_ = false, refused_ = false;
};

}  // namespace nh
#endif
