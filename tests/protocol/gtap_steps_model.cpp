// gtap_steps_model.cpp -- the stepped walks of the device code (gtap_steps.hpp) at the largest
// counts an int32 holds, run under the undefined-behaviour sanitizer by
// tests/test_protocol_model.py. Every walk must visit each of its positions once and end.
#include <cstdint>
#include <cstdio>
#include <initializer_list>

#include "gtap_steps.hpp"

static int g_failures = 0;

// A walk as the kernels' loops run it, with `sub` of `lanes` lanes: steps of `step` from `from`.
static void check(uint32_t n, uint32_t step, uint32_t from) {
    const uint64_t expect = n > from ? ((uint64_t)n - from + step - 1) / step : 0u;
    uint64_t steps = 0, items = 0;
    gtap::Steps s{n, step, from};
    if (s.steps() != expect) ++g_failures;
    for (; s.on() && steps <= expect; s.next()) {
        if (s.at != (uint64_t)from + steps * step) break;
        items += s.more() ? s.step : s.left();
        ++steps;
    }
    const uint64_t want = n > from ? n - from : 0u;
    if (steps != expect || items != want || s.on() || s.left() != 0u || s.more()) {
        fprintf(stderr, "FAIL n=%u step=%u from=%u: %llu steps (expected %llu), %llu items\n", n, step, from,
                (unsigned long long)steps, (unsigned long long)expect, (unsigned long long)items);
        ++g_failures;
    }
    // past the end, as a lane with a short row goes on beside one with a long row
    gtap::Steps beyond{n, step, (0x7FFFFFFFu / step + 1u) * step};
    if (beyond.at >= n && (beyond.on() || beyond.left() != 0u || beyond.more())) ++g_failures;
}

int main() {
    const uint32_t top = 0x7FFFFFFFu;  // INT32_MAX
    for (uint32_t step : {1u, 2u, 4u, 8u, 16u, 32u, 64u, 128u, 256u, 512u}) {
        for (uint32_t d : {0u, 1u, 7u, 63u, 64u, 255u, 256u, 257u, 511u, 512u, 513u}) {
            if (step >= 64u) check(top - d, step, d % 64u);
            check(d, step, 0u);
            check(d, step, 63u);
        }
    }
    if (g_failures) return 1;
    printf("steps model ok\n");
    return 0;
}
