// The words in which the count pass keeps large rectangles' claims for the
// write pass. Plain constexpr functions, the same for the kernels and for host
// code.
#pragma once

#include <cstdint>

namespace mg {

// The count pass keeps each large rectangle's claims, one 64-bit word per
// walk step (the wave's ballot of that step's claims), so the write pass
// replays the steps instead of testing every tile again. A count workgroup
// has kBlockWords words, taken by its rectangles as their walks start; a
// rectangle whose steps no longer fit is walked again by the write pass.
// Its mask word records where its words are: 1 + the first word's index, the
// step count from bit kWordSteps and the walk's rows a step, less one, from
// bit kWordRows (0: not kept).
constexpr int kBlockWords = 1024;
constexpr int kWordSteps = 11, kWordRows = 22;
static_assert(kBlockWords < (1 << kWordSteps), "the first word's index + 1 fits below the steps");
static_assert(kBlockWords < (1 << (kWordRows - kWordSteps)), "the steps fit below the rows");

constexpr uint32_t kept_mask(int first, int nst, int R) {
    return (uint32_t)(first + 1) | ((uint32_t)nst << kWordSteps) |
           ((uint32_t)(R - 1) << kWordRows);
}
constexpr int kept_first(uint32_t m) { return (int)(m & ((1u << kWordSteps) - 1u)) - 1; }
constexpr int kept_steps(uint32_t m) {
    return (int)(m >> kWordSteps & ((1u << (kWordRows - kWordSteps)) - 1u));
}
constexpr int kept_rows(uint32_t m) { return (int)(m >> kWordRows) + 1; }

// Whether the write pass takes up a Gaussian with this count and mask word.
// One that claims nothing has a mask word only if words are kept for it
// (a small rectangle's mask is its claims): it emits nothing, but its run
// must be marked, so that every word up to the last run's end lies in a
// marked run.
constexpr bool write_takes(int count, uint32_t mask) { return count > 0 || mask != 0u; }

}  // namespace mg
