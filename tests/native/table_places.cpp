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
    std::printf("ok\n");
    return 0;
}
