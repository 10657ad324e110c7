// Runs of features whose cut points a workgroup holds in LDS while it looks for the bins of their values (host only).
#pragma once
#include <vector>

namespace tgbm {

constexpr int kBinLds = 16384;  // words: a run's cut points, its features' ranges and one more

// First feature of every run, and the end; empty: a feature has too many cut points.
inline std::vector<int> bin_groups(const std::vector<int> &cut_row_ptr) {
    std::vector<int> first{0};
    const int F = (int)cut_row_ptr.size() - 1;
    for (int f = 0; f < F; ++f) {
        const int cuts = cut_row_ptr[(size_t)f + 1] - cut_row_ptr[(size_t)first.back()];
        if (f > first.back() && cuts + (f + 1 - first.back()) + 1 > kBinLds) first.push_back(f);
        if (cut_row_ptr[(size_t)f + 1] - cut_row_ptr[(size_t)f] + 2 > kBinLds) return {};
    }
    first.push_back(F);
    return first;
}

// Are the bins looked for by runs? Every run looks for its first value in every row, so rows have to have some of its values: us by a value's
// own way through the caches and by runs, 50 k x 1810 in 29 runs with 1.1 values a row and run 42 and 140, 3.1 184 and 199, 6.2 354 and
// 213, 60 2581 and 628; 200 k x 400 in 7 with 2.9 142 and 158, 5.7 258 and 186; 20 k x 6000 in 96 with 3.1 264 and 325, 6.2 495 and 387.
constexpr int kBinGroupValues = 4;
inline bool bins_by_groups(long nnz, long rows, int n_groups) { return nnz >= kBinGroupValues * rows * n_groups; }

}  // namespace tgbm
