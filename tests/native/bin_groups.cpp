// Runs of features for the search of bins (bin_groups.h): they hold every feature once and in order, fit the LDS and are full; rows of
// few values do not go by them.
#include <cstdio>

#include "../../thundergbm_amd/csrc/bin_groups.h"

#define CHECK(c) \
    if (!(c)) { std::printf("line %d: %s (case %d)\n", __LINE__, #c, at); return 1; }

int main() {
    using namespace tgbm;
    const struct { int features, cuts; } cases[] = {{0, 0}, {1, 1}, {1, 16382}, {700, 255}, {1810, 255}, {20000, 1}, {20000, 0}, {37, 1024}, {3, 16382}, {64, 254}};
    int at = 0;
    for (const auto &c : cases) {
        std::vector<int> ptr{0};
        for (int f = 0; f < c.features; ++f) ptr.push_back(ptr.back() + (f % 7 == 3 ? c.cuts / 2 : c.cuts));
        const std::vector<int> first = bin_groups(ptr);
        CHECK(first.size() >= 2 && first.front() == 0 && first.back() == c.features);
        for (size_t g = 0; g + 1 < first.size(); ++g) {
            const int f0 = first[g], f1 = first[g + 1];
            CHECK(f0 < f1 || c.features == 0);
            CHECK(ptr[f1] - ptr[f0] + (f1 - f0) + 1 <= kBinLds);
            CHECK(f1 == c.features || ptr[f1 + 1] - ptr[f0] + (f1 + 1 - f0) + 1 > kBinLds);
        }
        ++at;
    }
    CHECK(bin_groups({0, 5, 5 + kBinLds}).empty());
    // click data with a dense matrix of bins (203 501 rows of 21 values in 1810 columns), and a full table of the same columns
    CHECK(!bins_by_groups(4174607, 203501, 29));
    CHECK(bins_by_groups(203501l * 1810, 203501, 29));
    std::printf("ok\n");
    return 0;
}
