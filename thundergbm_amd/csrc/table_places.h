// Where the values of the frequent features of the sparse level pass lie (host only).
#pragma once
#include <algorithm>
#include <vector>

namespace tgbm {

constexpr int kSpreadGroup = 4;             // places are counted in groups of as many
constexpr int kSparseTaskValues = 32768;    // stored values per task at most (and places per chunk of a big feature)

// Groups that `values` values in `blocks` row blocks take at most: up to three places are nobody's in every block that has some.
inline long groups_of(long values, int blocks) {
    const long begun = std::min<long>(std::max(1, blocks), values);
    return (values + (kSpreadGroup - 1) * begun + kSpreadGroup - 1) / kSpreadGroup;
}

// Ends of the chunks that a feature's groups [begin, end) are cut into. (Everything is counted in groups: close to 2^31 values, which the
// level pass takes, have more places than an int counts.)
inline std::vector<int> chunk_ends(int begin, int end) {
    constexpr int kChunk = kSparseTaskValues / kSpreadGroup;
    std::vector<int> ends;
    for (int g = begin; g < end; g += kChunk) ends.push_back(std::min(end, g + kChunk));
    return ends;
}

// What a workgroup of the set-up gives their places: up to so many values of a frequent feature, from the begin-th on. (Counted in values
// and not in row blocks: a feature of 10 000 values has some in each of 300 blocks, one of 10 M may have them all in one.)
constexpr int kTableSetupValues = 8192;
struct TablePart {
    int feature;  // among the frequent ones
    int begin;
};
inline void add_table_parts(std::vector<TablePart> &parts, int feature, long values) {
    for (long v = 0; v < values; v += kTableSetupValues) parts.push_back(TablePart{feature, (int)v});
}

}  // namespace tgbm
