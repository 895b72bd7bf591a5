// Offsets of the few-row product's normalising forms.  Plain C++: no device code, so that it can be tested without a GPU.
#pragma once

#include <stdint.h>

namespace tsattn {

// Whether every value of `rows` rows can be reached with an unsigned 32-bit byte offset from the first: int32 planes with rows of k
// values, and a float state with rows of state_pitch.  What does not fit is normalised by a launch of its own (64-bit addresses).
// The widest layer served (2^20 values, a feed-forward block of 2^21) fits with 16 rows; a bound on k alone of 2^20 refused it.
constexpr bool few_offsets_fit(int64_t rows, int64_t k, int64_t state_pitch)
{
    constexpr int64_t most = ((int64_t)1 << 32) / 4;
    return k <= most / rows && state_pitch <= most / rows;
}

} // namespace tsattn
