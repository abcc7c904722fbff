// Which row of the raster backward's per-entry sums (S.grad) a lane adds to.
// Plain constexpr functions, the same for the kernel and for host code.
#pragma once

namespace mg {

// Rows of S.grad: colour 3, moments 5, sum dg, and |d uv| where it is asked for.
constexpr int grad_rows(bool abs) { return abs ? 10 : 9; }

// The row that lane row r (0..3) of reduce10_to_rows's q-th result is added
// to. Row r of q0 holds the sum of value {0,2,1,3}[r], of q1 {4,6,5,7}[r], of
// q2 {8,-,9,-}[r], "-" a sum of zeros. q2's zeros, among them value 9 without
// |d uv|, go to a row that exists, where they add nothing: a lane-dependent
// address, which the compiler does not turn into a wave-aggregation loop as it
// does a single lane's.
constexpr int deposit_row(int q, int r, bool abs) {
    return q < 2 ? 4 * q + (r & 1) * 2 + (r >> 1) : abs ? 8 + (r >> 1) : 8 - (r >> 1);
}

// The value of reduce18's sum in a lane, -1 for lanes that deposit nothing.
constexpr int reduce18_slot(int lane) {
    return (lane & 1) ? -1
           : (lane & 2)
               ? ((lane & 0x1C) == 0 ? 8 : -1)
               : 4 * ((lane >> 2) & 1) + 2 * ((lane >> 3) & 1) + ((lane >> 4) & 1);
}

constexpr bool deposits_in_range(bool abs) {
    for (int q = 0; q < 3; ++q)
        for (int r = 0; r < 4; ++r)
            if (deposit_row(q, r, abs) < 0 || deposit_row(q, r, abs) >= grad_rows(abs)) return false;
    // reduce18 sums nine values, without |d uv|.
    for (int lane = 0; lane < 64; ++lane)
        if (reduce18_slot(lane) >= grad_rows(false)) return false;
    return true;
}
static_assert(deposits_in_range(true) && deposits_in_range(false), "every deposit has its row");

}  // namespace mg
