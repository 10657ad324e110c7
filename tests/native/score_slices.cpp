// The slices of a scoring call (score_slices.h): they cover the rows once and in order, hold the values they are meant for, and
// none has too few rows for the kernel that the whole call is for.
#include <cstdio>
#include <random>

#include "../../thundergbm_amd/csrc/score_slices.h"

#define CHECK(c) \
    if (!(c)) { std::printf("line %d: %s (case %d)\n", __LINE__, #c, at); return 1; }

int main() {
    constexpr int kLeast = 65536;
    std::mt19937 gen(1);
    const struct { int rows, per_row; long entries; int least; } cases[] = {
        {500000, 40, 2 << 20, kLeast}, {500000, 40, 2 << 20, 1}, {65536, 100, 2 << 20, kLeast}, {131071, 60, 2 << 20, kLeast},
        {131072, 60, 2 << 20, kLeast}, {200000, 0, 2 << 20, kLeast}, {1, 5, 1, 1}, {1000, 7, 1, 1}, {70000, 33, 1, kLeast}};
    int at = 0;
    for (const auto &c : cases) {
        for (int ragged = 0; ragged < 2; ++ragged) {
            std::vector<int> ptr{3};  // (values may begin anywhere)
            for (int r = 0; r < c.rows; ++r) {
                const int big = ragged && r % 997 == 5 ? 40 * c.per_row : 0;
                ptr.push_back(ptr.back() + (ragged ? (int)(gen() % (unsigned)(2 * c.per_row + 1)) * (r % 3 != 0) + big : c.per_row));
            }
            const std::vector<int> first = tgbm::score_slices(ptr.data(), c.rows, c.entries, c.least);
            CHECK(first.front() == 0 && first.back() == c.rows);
            for (size_t k = 0; k + 1 < first.size(); ++k) {
                const int rows = first[k + 1] - first[k];
                const long held = ptr[first[k + 1]] - ptr[first[k]];
                CHECK(rows >= c.least);
                CHECK(held <= c.entries || rows < 2 * c.least || rows == 1);
                // (a row more would not have fitted, unless nothing is left)
                CHECK(k + 2 == first.size() || ptr[first[k + 1] + 1] - ptr[first[k]] > c.entries);
            }
        }
        ++at;
    }
    std::printf("ok\n");
    return 0;
}
