// Query groups of a workgroup (rank_packs.h): every row is in one pack or wide group, packs hold whole groups, shared ones are full.
#include <cstdio>

#include "../../thundergbm_amd/csrc/rank_packs.h"

#define CHECK(c) \
    if (!(c)) { std::printf("line %d: %s (case %d)\n", __LINE__, #c, at); return 1; }

int main() {
    using namespace tgbm;
    const std::vector<std::vector<int>> cases = {
        {}, {0}, {1}, {0, 0, 5, 0}, {64}, {65}, {256}, {257}, {257, 0, 0}, {2048}, {1, 64, 1}, {32, 32, 1}, {100, 29, 64, 0, 256, 3, 257, 0, 4, 2000, 63, 1, 1},
        std::vector<int>(100000, 1), std::vector<int>(5000, 3), std::vector<int>(700, 24), std::vector<int>(700, 25), std::vector<int>(300, 120)};
    int at = 0;
    for (const auto &group : cases) {
        std::vector<int> gptr{0};
        for (int rows : group) gptr.push_back(gptr.back() + rows);
        const RankPacks p = rank_packs(group);
        std::vector<int> seen((size_t)gptr.back(), 0);
        int most = 0;
        for (const std::vector<RankPack> *list : {&p.packs, &p.wide})
            for (const RankPack &k : *list) {
                CHECK(k.begin >= 0 && k.begin < k.end && k.end <= gptr.back());
                for (int r = k.begin; r < k.end; ++r) ++seen[(size_t)r];
                int inside = 0, first = -1;
                for (size_t g = 0; g < group.size(); ++g) {
                    if (group[g] == 0 || gptr[g] < k.begin || gptr[g] >= k.end) continue;
                    if (inside++ == 0) first = (int)g;
                    CHECK(gptr[g + 1] <= k.end && (group[g] > kMiddleGroup) == (list == &p.wide));
                }
                CHECK(inside > 0 && k.group == first);
                CHECK(inside == 1 || (p.shared && list == &p.packs && k.end - k.begin <= kPackRows));
                if (list == &p.packs) most = std::max(most, k.end - k.begin);
            }
        for (int times : seen) CHECK(times == 1);
        CHECK(most == p.most);
        // (two shared packs side by side have more rows than one takes)
        CHECK(p.shared == (gptr.back() <= kShareMean * (long)group.size()));
        CHECK((long)p.packs.size() <= (p.shared ? 2l * gptr.back() / kPackRows + 1 + (long)p.wide.size() : (long)group.size()));
        ++at;
    }
    std::printf("ok\n");
    return 0;
}
