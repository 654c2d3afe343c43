// gtap_steps.hpp -- walks over counted items in fixed steps, for device and host code.
#pragma once

#include <cstdint>

#if defined(__HIPCC__)
#define GTAP_STEPS_FN __host__ __device__ __forceinline__
#else
#define GTAP_STEPS_FN inline
#endif

namespace gtap {

// A walk over n items, n any count that an int32 holds, `step` (a power of two) at a time from
// position `at`. Positions are unsigned: the one after the last step is up to n + step - 1, past an
// int32, where a signed position would overflow and the walk would not end.
struct Steps {
    uint32_t n, step, at;
    GTAP_STEPS_FN bool on() const { return at < n; }                        // items are left
    GTAP_STEPS_FN uint32_t left() const { return at < n ? n - at : 0u; }  // how many, this step's included
    GTAP_STEPS_FN bool more() const { return at + step < n; }               // a further step is needed
    GTAP_STEPS_FN void next() { at += step; }
    // How many steps the walk takes. A loop that counts them is one whose length the compiler
    // knows and unrolls, which it does not for positions that may wrap (tree of height 15: 219 us
    // against 209 us).
    GTAP_STEPS_FN uint32_t steps() const { return on() ? ((n - 1u - at) >> __builtin_ctz(step)) + 1u : 0u; }
};

}  // namespace gtap
