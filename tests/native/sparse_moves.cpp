// k_sparse_partition as it stands in sparse_kernels.hip (moves.inc, its text) with its threads one after the other between
// the barriers: a thread then finds everything that the ones before it have stored. Every array checks its indices, and
// LDS that nobody has written may not be read.
#include <algorithm>
#include <condition_variable>
#include <cstdio>
#include <cstdlib>
#include <mutex>
#include <thread>
#include <vector>

using std::max;
using std::min;
static void check(bool ok, const char *what) {
    if (ok) return;
    std::printf("%s\n", what);
    std::fflush(stdout);
    std::_Exit(1);
}

struct Cell {
    int v = 0;
    bool set = false;
    operator int() const {
        check(set, "LDS read that nobody has written");
        return v;
    }
    Cell &operator=(int to) {
        v = to;
        set = true;
        return *this;
    }
};
template <int N>
struct Shared {
    Cell c[N];
    Cell &operator[](int i) {
        check(i >= 0 && i < N, "LDS index");
        return c[i];
    }
};
template <typename T>
struct Array {
    std::vector<T> *v = nullptr;
    T &operator[](size_t i) const {
        check(i < v->size(), "index of a global array");
        return (*v)[i];
    }
    bool operator!=(std::nullptr_t) const { return v != nullptr; }
};
static void atomicAdd(Cell *c, int by) { *c = *c + by; }
static void atomicAdd(int *c, int by) { *c += by; }

struct Node {
    bool splits;
    int split_feature_id;
    unsigned char split_bid;
    bool default_right;
};
typedef Node TreeNode;
static bool node_splits(const Node &nd) { return nd.splits; }
struct TreeBuffers {
    int n;
    Array<Node> nodes;
    Array<unsigned short> nid16;
    Array<unsigned> row_word;
    Array<int> cut_row_ptr, node_rows;
    TreeBuffers for_class(int) const { return *this; }
};
struct CsrBins {
    Array<int> col_of_feature;
    Array<unsigned char> colbin;
    size_t col_stride;
};
static bool csr_goes_right(const CsrBins &, int, int, int, int, bool) { return false; }

constexpr int kSpBlock = 1024, kSparseMaxLevelNodes = 1024, kMissingBin = 255;
constexpr unsigned kRareNodeMask = 0x7ffu;
struct Dim {
    int x, z;
};
static thread_local Dim threadIdx;
static Dim blockIdx{0, 0}, gridDim{1, 1};
static int lane_id() { return threadIdx.x & 63; }
static int __clz(int v) { return __builtin_clz((unsigned)v); }

static std::mutex mutex;
static std::condition_variable turn_changed[kSpBlock];
static int turn = 0, rounds = 0;  // whose turn it is; barriers that all have reached
static void pass_turn(int me, bool barrier) {
    std::unique_lock<std::mutex> lock(mutex);
    const int round = rounds;
    turn = me + 1;
    if (turn == kSpBlock) {
        turn = 0;
        ++rounds;
    }
    turn_changed[turn].notify_one();
    if (barrier) turn_changed[me].wait(lock, [&] { return rounds > round && turn == me; });
}
static void __syncthreads() { pass_turn(threadIdx.x, true); }

#define __global__ static
#define __launch_bounds__(...)
#include "moves.inc"

int main() {
    const int level = 1, n = 4 * kSpBlock - 100;  // the last 100 threads have no fourth row
    std::vector<Node> nodes(7, Node{false, -1, 0, false});
    nodes[1] = Node{true, 0, 3, false};
    nodes[2] = Node{true, 1, 5, true};
    std::vector<unsigned short> nid(n);
    std::vector<unsigned> word(n, 0u);
    std::vector<int> cuts{0, 8, 16}, rows(7, 0), col_of{0, 1};
    std::vector<unsigned char> colbin(2 * n);
    for (int r = 0; r < n; ++r) {
        nid[r] = (unsigned short)(1 + r % 2);
        colbin[r] = (unsigned char)(r % 7);
        colbin[n + r] = (unsigned char)(r % 5 == 0 ? kMissingBin : r % 8);
    }
    TreeBuffers tb{n, {&nodes}, {&nid}, {&word}, {&cuts}, {&rows}};
    CsrBins bins{{&col_of}, {&colbin}, (size_t)n};
    std::vector<std::thread> threads;
    for (int t = 0; t < kSpBlock; ++t)
        threads.emplace_back([&, t] {
            threadIdx = Dim{t, 0};
            {
                std::unique_lock<std::mutex> lock(mutex);
                turn_changed[t].wait(lock, [&] { return turn == t && rounds == 0; });
            }
            k_sparse_partition(tb, bins, level);
            pass_turn(t, false);
        });
    for (std::thread &t : threads) t.join();
    std::vector<int> want(7, 0);
    for (int r = 0; r < n; ++r) {
        const bool second = r % 2 == 1;
        const int b = second ? colbin[n + r] : colbin[r];
        const bool right = b == kMissingBin ? second : b >= (second ? 5 : 3);
        const int to = (second ? 5 : 3) + (right ? 1 : 0);
        check(nid[r] == to && (word[r] & kRareNodeMask) == (unsigned)(to - 3), "a row's node");
        ++want[to];
    }
    check(rows == want, "rows per child");
    return 0;
}
