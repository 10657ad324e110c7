// Places of the frequent features' values (table_places.h): every feature has room for what it may take, and its chunks cover it
// once and in order, up to 2^31 - 1 values, which the level pass takes.
#include <cstdio>

#include "../../thundergbm_amd/csrc/table_places.h"

#define CHECK(c) \
    if (!(c)) { std::printf("line %d: %s (%ld values, %d features)\n", __LINE__, #c, all, features); return 1; }

int main() {
    using namespace tgbm;
    for (long all : {1l, 5l, 40000l, 3000000l, (1l << 30) - 1, 1l << 30, (1l << 31) - 32768, (1l << 31) - 1})
        for (int features : {1, 3, 128, 500, 20000})
            for (int blocks : {0, 1, 31, 341}) {
                if (blocks > 0 && all >= 1l << 30) continue;  // (such data is not spread)
                long groups = 0;
                for (int f = 0; f < features; ++f) {
                    const long values = all / features + (f < all % features ? 1 : 0);
                    const long next = groups + groups_of(values, blocks);
                    CHECK(next < (1l << 31) && next >= groups);
                    // all blocks but one begin with one value: the most groups that so many values can take
                    const long begun = std::min<long>(std::max(1, blocks), values);
                    const long most = values == 0 ? 0 : begun - 1 + (values - (begun - 1) + kSpreadGroup - 1) / kSpreadGroup;
                    CHECK(next - groups >= most);
                    long at = groups;
                    for (int end : chunk_ends((int)groups, (int)next)) {
                        CHECK(end > at && (end - at) * kSpreadGroup <= kSparseTaskValues);
                        at = end;
                    }
                    CHECK(at == next);
                    groups = next;
                }
            }
    // Parts of the set-up: every value has one, and there are no more of them than features and values call for, however many row blocks
    // there are (an ordinary feature of 10 M rows has a few values in each of 300, one that most rows store has them all in the one
    // "block" of values that are not spread).
    for (long all : {0l, 1l, 8191l, 8192l, 8193l, 12000000l, (1l << 31) - 1})
        for (int features : {1, 7, 15000}) {
            std::vector<TablePart> parts;
            for (int f = 0; f < features; ++f) add_table_parts(parts, f, all / features + (f < all % features ? 1 : 0));
            CHECK((long)parts.size() <= std::min<long>(features, all) + all / kTableSetupValues);
            size_t at = 0;
            for (int f = 0; f < features; ++f)
                for (long v = 0, values = all / features + (f < all % features ? 1 : 0); v < values; v += kTableSetupValues, ++at)
                    CHECK(at < parts.size() && parts[at].feature == f && parts[at].begin == v);
            CHECK(at == parts.size());
        }
    std::printf("ok\n");
    return 0;
}
