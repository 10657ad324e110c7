// Which query groups a workgroup of a ranking round takes (host only).
#pragma once
#include <algorithm>
#include <vector>

namespace tgbm {

// Neighbouring groups share a workgroup where groups have at most kShareMean rows on average: a workgroup's fixed part, some ten trips to the
// caches, is then most of what it does. 1 M rows, depth 4, 20 rounds, ms with a workgroup a group and with shared ones: groups of 1 row
// 13.4, 2.0; 2 9.6, 3.1; 5 5.8, 3.1; 12 4.1, 3.2; 24 3.57, 3.24; 40 3.37, 3.45. (Beyond it the look-ups of a row's group cost more than they save.)
constexpr int kShareMean = 24;
// Rows that groups which share a workgroup have together at most, and rows of the longest group that such workgroups take.
constexpr int kPackRows = 128, kMiddleGroup = 256;

// Rows [begin, end) of a workgroup; group: theirs, or the first of several neighbours'.
struct alignas(16) RankPack {
    int begin, end, group;
};
// `packs`: groups by themselves or, shared, neighbours of at most kPackRows rows together; `wide`: the groups of more than kMiddleGroup rows.
// Groups without rows are in none.
struct RankPacks {
    std::vector<RankPack> packs, wide;
    int most = 0;  // rows of a pack
    bool shared = false;
};
inline RankPacks rank_packs(const std::vector<int> &group) {
    RankPacks out;
    RankPack open{0, 0, 0};  // (end == begin: none)
    long rows = 0;
    for (int r : group) rows += r;
    out.shared = rows <= kShareMean * (long)group.size();
    const auto close = [&] {
        if (open.end > open.begin) out.packs.push_back(open);
        out.most = std::max(out.most, open.end - open.begin);
    };
    int row = 0;
    for (int g = 0; g < (int)group.size(); row += group[g++]) {
        const RankPack own{row, row + group[g], g};
        if (group[g] == 0) continue;
        if (group[g] > kMiddleGroup) {
            out.wide.push_back(own);
        } else if (out.shared && open.end > open.begin && own.begin == open.end && own.end - open.begin <= kPackRows) {
            open.end = own.end;
        } else {
            close();
            open = own;
        }
    }
    close();
    return out;
}

}  // namespace tgbm
