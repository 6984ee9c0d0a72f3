// What a call of some shape needs besides its pointers - kernel choice, workspace carve - computed once per thread and
// shape: the rules behind them loop over tile shapes with divisions and were evaluated several times per call, 1.0 us of
// the 4.4 us that a small linear spent below Python.  Direct-mapped by a hash with the multipliers of the splitmix64
// generator's mixer; a tuning run, whose choices follow the environment, never reads it.
#pragma once
#include <stdint.h>

#include "tuning.h"

namespace phyai {

template <class Value, int SLOTS>
class CallMemo {
    struct Slot {
        int64_t key[4];
        Value value;
        bool full;
    };
    Slot slots_[SLOTS] = {};

public:
    template <class Make>
    const Value& get(int64_t a, int64_t b, int64_t c, int64_t d, Make make) {
        uint64_t h = (uint64_t)a * 0x9E3779B97F4A7C15ull;
        h = (h ^ (h >> 29) ^ (uint64_t)b) * 0xBF58476D1CE4E5B9ull;
        h = (h ^ (h >> 29) ^ (uint64_t)c) * 0x94D049BB133111EBull;
        h = (h ^ (h >> 29) ^ (uint64_t)d) * 0x9E3779B97F4A7C15ull;
        Slot& s = slots_[(h >> 32) % SLOTS];
        if (!s.full || s.key[0] != a || s.key[1] != b || s.key[2] != c || s.key[3] != d || tuning_enabled()) {
            s.full = false;
            s.value = make();
            s.key[0] = a; s.key[1] = b; s.key[2] = c; s.key[3] = d;
            s.full = true;
        }
        return s.value;
    }
};

}  // namespace phyai
