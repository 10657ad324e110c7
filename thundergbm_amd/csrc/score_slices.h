// How the rows of a scoring call are cut into slices (host only).
#pragma once
#include <algorithm>
#include <vector>

namespace tgbm {

// First rows of the slices of n sparse rows, and n: whole rows, as many as `entries` stored values hold, at least `least_rows`
// of them, none fewer at the end either.
inline std::vector<int> score_slices(const int *row_ptr, int n, long entries, int least_rows) {
    std::vector<int> first{0};
    while (first.back() < n) {
        const int r0 = first.back();
        const int *from = row_ptr + r0 + 1, *last = row_ptr + n + 1;
        const long upto = std::min((long)row_ptr[r0] + entries, (long)row_ptr[n]);
        int rows = (int)(std::upper_bound(from, last, (int)upto) - from);
        rows = std::max(rows, least_rows);
        first.push_back(n - r0 - rows < least_rows ? n : r0 + rows);
    }
    return first;
}

}  // namespace tgbm
