// Which set of tile counters a persistent launch takes. Plain C++: no device, no HIP.
#pragma once

namespace ngx {

// Two sets that launches take in turn, each zeroing the other's as it runs, so that a launch finds its own zero without a
// kernel before it. A frame that an error ends half launched may have taken a set without the next being zeroed: the sets
// are then dirty until they are zeroed from outside, whatever other frames, which take none, are drawn before that.
struct CounterTurns {
    int set = 0;         // which of the two the next launch takes
    bool dirty = false;  // both must be zeroed before it

    // One frame's launches, closed after the last. Null: the frame takes none.
    class Frame {
        CounterTurns *turns;

      public:
        explicit Frame(CounterTurns *t) : turns(t) {}
        Frame(const Frame &) = delete;
        Frame &operator=(const Frame &) = delete;
        ~Frame() {
            if (turns) turns->dirty = true;
        }
        void close() { turns = nullptr; }
    };
};

}  // namespace ngx
