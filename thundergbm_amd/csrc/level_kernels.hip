// The rows of a level move on to its nodes' children (dense layout): two launches per level. The first picks every node's
// best candidate, applies it to the tree and decides left or right for every row; the second compacts the row lists and
// leaves the next level's sibling pairs. What used to be launches of their own in between - the update of the tree, the
// scan of the items' counts, the plan of the next level - is done again by every workgroup from a few hundred bytes
// that it finds in the L2: a launch costs 4 to 8 us whatever it does, the repeated work well below one.
// 500 k x 28, depth 8: five launches and 23 us a level (update 4.8, count 5.7, plan 5.5, scatter 4.9, gaps) -> two.
// That holds up to 512 nodes. Deeper levels have 16 to 130 KB of plan and more items to repeat it for; they are planned by a
// third launch (TreeBuffers::planned).
#include <algorithm>

#include "device_api.h"
#include "kernel_common.h"
#include "tree_common.h"

namespace tgbm {
namespace {

// A partition work item: kPartChunk rows of one node. The nodes of a level own ceil(rows / kPartChunk) items each, at
// least one (a node without rows still has a split record to fill), numbered node by node.
struct NodeItem {
    int x_in;   // node within the level, -1: there is no such item
    int first;  // first item of the node
    int count;  // items of the node
    int2 seg;
};

// Every wavefront of the workgroup finds the item for itself, without a barrier; the result is the same in all of its lanes.
// PLANNED: TreeBuffers::planned(level), by the launcher (as a branch in here it cost the count launches of the other
// levels 0.4 us each)
template <bool PLANNED>
__device__ __forceinline__ NodeItem locate_item(const TreeBuffers &tb, int level, int item) {
    const int nl = 1 << level, off = nl - 1;
    NodeItem out;
    if (!PLANNED && level == 0) {
        out.count = max(1, (tb.n + kPartChunk - 1) / kPartChunk);
        out.x_in = item < out.count ? 0 : -1;
        out.first = 0;
        out.seg = make_int2(0, tb.n);
        return out;
    }
    out.x_in = -1;
    if (PLANNED) {
        const int *__restrict__ begin = tb.pbegin(level);
        if (item >= __builtin_amdgcn_readfirstlane(begin[nl])) return out;
        out.x_in = find_owner_wave(begin, nl, item);
        out.first = __builtin_amdgcn_readfirstlane(begin[out.x_in]);
        out.count = __builtin_amdgcn_readfirstlane(begin[out.x_in + 1]) - out.first;
        const int2 sg = tb.seg[off + out.x_in];
        out.seg = make_int2(__builtin_amdgcn_readfirstlane(sg.x), __builtin_amdgcn_readfirstlane(sg.y));
        return out;
    }
    constexpr int A = 4;  // 64 nodes each, loaded together
    const int2 *__restrict__ segs = tb.seg + off;
    int carry = 0;
    for (int base = 0; base < nl; base += A * 64) {
        int2 sg[A];
#pragma unroll
        for (int a = 0; a < A; ++a) sg[a] = segs[min(base + a * 64 + lane_id(), nl - 1)];
#pragma unroll
        for (int a = 0; a < A; ++a) {
            if (base + a * 64 >= nl) break;
            const int cnt = base + a * 64 + lane_id() < nl ? max(1, (sg[a].y - sg[a].x + kPartChunk - 1) / kPartChunk) : 0;
            const int inc = wave_scan_i(cnt), ex = carry + inc - cnt;
            const unsigned long long owner = __ballot(item >= ex && item < ex + cnt);
            if (owner != 0ull) {
                const int l = __ffsll((long long)owner) - 1;
                out.x_in = base + a * 64 + l;
                out.first = read_lane(ex, l);
                out.count = read_lane(cnt, l);
                out.seg = make_int2(read_lane(sg[a].x, l), read_lane(sg[a].y, l));
                return out;
            }
            carry += read_lane(inc, 63);
        }
    }
    return out;
}

// What the workgroups of a node need of its best candidate (larger |score|, then the smaller bin index).
struct Picked {
    bool found;  // false: the node has no candidate
    SplitCand c;
};
// Up to so many packs each wavefront looks at all of them: no barrier, no LDS (500 k x 28: the candidates' part of a count
// launch 1.7 -> 0.95 us; of a small level's sixteen wavefronts 2.9 -> 0.65 with 100 packs). Beyond, the workgroup
// shares them out.
constexpr int kWavePacks = 256;
struct PickShared {
    SplitCand cand;
    float abs[16];
    int idx[16];
};
// A lane's candidate where every wavefront looks at all of them, so that its load can be issued ahead of what comes before.
__device__ __forceinline__ SplitCand early_candidate(const TreeBuffers &tb, int x_in) {
    return tb.cand[(size_t)x_in * tb.n_packs + min(lane_id(), tb.n_packs - 1)];
}
// NW: wavefronts of the workgroup, all of whose threads call
template <int NW>
__device__ __forceinline__ Picked pick_candidate(const TreeBuffers &tb, int x_in, bool valid, PickShared &sh, const SplitCand &early) {
    const bool alone = tb.n_packs <= kWavePacks;
    float a_best = -1.f;
    int i_best = 0x7fffffff;
    SplitCand best;
    best.score = 0.f;
    best.index = 0x7fffffff;
    best.miss = best.left = GHPair{0, 0};
    best.feature = best.bin = 0;
    const SplitCand *__restrict__ cand = tb.cand + (size_t)x_in * tb.n_packs;
    auto look = [&](const SplitCand &c, bool in) {
        const float a = fabsf(c.score);
        // (index 0x7fffffff: a wavefront whose features have no bins)
        const bool better = in && c.index != 0x7fffffff && (a > a_best || (a == a_best && c.index < i_best));
        a_best = better ? a : a_best;
        i_best = better ? c.index : i_best;
        best.score = better ? c.score : best.score;
        best.miss.g = better ? c.miss.g : best.miss.g;
        best.miss.h = better ? c.miss.h : best.miss.h;
        best.left.g = better ? c.left.g : best.left.g;
        best.left.h = better ? c.left.h : best.left.h;
        best.feature = better ? c.feature : best.feature;
        best.bin = better ? c.bin : best.bin;
    };
    if (alone) {
        constexpr int U = kWavePacks / 64;
        SplitCand c[U];
        c[0] = early;
#pragma unroll
        for (int u = 1; u < U; ++u)
            if (u * 64 < tb.n_packs) c[u] = cand[min(u * 64 + lane_id(), tb.n_packs - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (u * 64 < tb.n_packs) look(c[u], valid && u * 64 + lane_id() < tb.n_packs);
    } else {
        constexpr int U = 3;  // candidates per thread whose loads are issued together
        for (int p0 = threadIdx.x; p0 - (int)threadIdx.x < tb.n_packs; p0 += U * NW * 64) {
            SplitCand c[U];
#pragma unroll
            for (int u = 0; u < U; ++u) c[u] = cand[min(p0 + u * NW * 64, tb.n_packs - 1)];
#pragma unroll
            for (int u = 0; u < U; ++u) look(c[u], valid && p0 + u * NW * 64 < tb.n_packs);
        }
    }
    best.index = i_best;
    float win;
    int win_idx;
    const int owner = wave_best(a_best, i_best, &win, &win_idx);
    if (!alone) {
        if (lane_id() == 0) {
            sh.abs[wave_id()] = win;
            sh.idx[wave_id()] = win_idx;
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NW; ++i)
            if (sh.abs[i] > win || (sh.abs[i] == win && sh.idx[i] < win_idx)) {
                win = sh.abs[i];
                win_idx = sh.idx[i];
            }
        if (win_idx != 0x7fffffff && a_best == win && i_best == win_idx) sh.cand = best;
        __syncthreads();
        best = sh.cand;
        if (win_idx == 0x7fffffff) best.index = win_idx;
    }
    const int from = alone ? owner : 0;
    Picked out;
    out.found = win_idx != 0x7fffffff;
    out.c.score = read_lane(best.score, from);
    out.c.index = read_lane(best.index, from);
    out.c.miss.g = read_lane(best.miss.g, from);
    out.c.miss.h = read_lane(best.miss.h, from);
    out.c.left.g = read_lane(best.left.g, from);
    out.c.left.h = read_lane(best.left.h, from);
    out.c.feature = read_lane(best.feature, from);
    out.c.bin = read_lane(best.bin, from);
    return out;
}

__device__ __forceinline__ void apply_candidate(const TreeBuffers &tb, int x, int x_in, const TreeNode &node, bool found,
                                                const SplitCand &c, float rt_eps, float lambda) {
    if (!node.is_valid) {
        SplitPoint z{};
        z.nid = -1;
        z.split_fea_id = -1;
        tb.sp[x_in] = z;
    } else if (!found) {
        no_split(tb, x, x_in);
    } else {
        apply_split(tb, x, x_in, node, c, c.feature, c.bin, tb.cut_val[c.index - (c.bin != 0 ? 1 : 0)], rt_eps, lambda);
    }
}

// UPDATE: the nodes' candidates are fresh from the split search; else the tree has been updated already.
// A row goes right if its bin is not below the split bin, or if it has no value of the feature and the default says so
// (hist_tree_builder_single.cu:986-1011).
// MAP: the rows that end here leave their node in tb.nid for k_map_end. 1: those of nodes that do not split. 2 (the last level,
// whose children get no lists): all rows.
template <bool DIRECT, typename BinT, bool UPDATE, bool PLANNED, int MAP = 0>
__global__ __launch_bounds__(kBlock) void k_split_count(TreeBuffers tb_all, DenseBins bins, int level, float rt_eps,
                                                       float lambda) {
    __shared__ int lds[kWaves];
    __shared__ PickShared s_pick;
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int *__restrict__ ridx = tb.list(level);
    const int item = blockIdx.x;
    const NodeItem it = locate_item<PLANNED>(tb, level, item);
    if (it.x_in < 0) return;
    const int x_in = it.x_in, x = (1 << level) - 1 + x_in;
    const int2 sg = it.seg;
    const int pb = sg.x + (item - it.first) * kPartChunk;
    const int pe = min(sg.y, pb + kPartChunk);
    // All row ids first, then all bins, then the decisions, then the stores. Every load is unconditional (positions
    // past the item's end are clamped to its last row), so each phase's loads are issued back to back and a thread's
    // eight gathers are in flight together; a conditional load would make the compiler wait for everything
    // outstanding, the previous store included, before the next one.
    constexpr int R = kPartChunk / kBlock;
    int row[R], b[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int pos = max(min(pb + k * kBlock + (int)threadIdx.x, pe - 1), 0);
        row[k] = DIRECT ? pos : ridx[pos];
    }
    SplitCand early;
    if (UPDATE) early = early_candidate(tb, x_in);
    const TreeNode node = node_of_wave(tb, x);
    Picked best{};
    bool splits, dr = false;
    int f = 0, sbid = 0;
    if (UPDATE) {
        best = pick_candidate<kWaves>(tb, x_in, node.is_valid, s_pick, early);
        splits = best.found && fabsf(best.c.score) > rt_eps;
        if (splits) {
            f = best.c.feature;
            // (the byte that the model keeps, unless the features have more than 255 bins)
            sbid = tb.split_bin != nullptr ? best.c.bin : (int)(unsigned char)best.c.bin;
            dr = best.c.score < 0;
        }
    } else {
        splits = node_splits(node);
        if (splits) {
            f = node.split_feature_id;
            sbid = tb.split_bin != nullptr ? tb.split_bin[x] : (int)node.split_bid;
            dr = node.default_right;
        }
    }
    // (the tree's own stores come last: nothing of this workgroup waits for them)
    auto update = [&] {
        if (UPDATE && item == it.first && threadIdx.x == 0) apply_candidate(tb, x, x_in, node, best.found, best.c, rt_eps, lambda);
    };
    if (!splits) {
        if (MAP != 2 && threadIdx.x == 0) tb.pitem_nleft[item] = 0;
        if (MAP != 0)
#pragma unroll
            for (int k = 0; k < R; ++k)
                if (pb + k * kBlock + (int)threadIdx.x < pe) tb.nid[row[k]] = x;
        update();
        return;
    }
    // A stored bin outside [lo, lo + span) means that the row has no value of the feature: the missing sentinel, or
    // (a feature that shares its column with others, DenseBins::feat_col) a bin of another feature of the bundle.
    int c = f, lo = 0, span = sizeof(BinT) == 2 ? kMissingBin16 : kMissingBin;
    if (sizeof(BinT) == 1 && bins.feat_col != nullptr) {
        c = bins.feat_col[f];
        lo = bins.feat_lo[f];
        span = tb.cut_row_ptr[f + 1] - tb.cut_row_ptr[f];
    }
    const BinT *column = reinterpret_cast<const BinT *>(bins.col) + (size_t)c * bins.col_stride;
    int nleft = 0;
#pragma unroll
    for (int k = 0; k < R; ++k) b[k] = column[row[k]];
    unsigned rights = 0;
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int t = b[k] - lo;
        const bool right = ((unsigned)t >= (unsigned)span) ? dr : (t >= sbid);
        if (MAP == 2) {
            if (pb + k * kBlock + (int)threadIdx.x < pe) tb.nid[row[k]] = 2 * x + (right ? 2 : 1);
            continue;
        }
        rights |= (right ? 1u : 0u) << k;
        if (pb + k * kBlock + (int)threadIdx.x < pe) nleft += right ? 0 : 1;
    }
    if (MAP == 2) {
        update();
        return;
    }
    // the decisions of a thread's eight rows as one byte (k_split_scatter gives the same rows to the same thread)
    static_assert(R <= 8, "a byte per thread holds the decisions of its rows");
    tb.goes_right[(size_t)item * kBlock + threadIdx.x] = (uint8_t)rights;
    const int tot = block_sum(nleft, lds);
    if (threadIdx.x == 0) tb.pitem_nleft[item] = tot;
    update();
}

// Sums of kPartGroup items' counts, a wavefront per group. 100 M x 6, depth 8: with every count of the node in every item
// 11.1 ms a tree, with the groups 9.8; 20 M x 8: 2.09 and 2.04, 10 M x 28: 1.274 and 1.278 (as atomics of k_split_count, whose
// sums share cache lines, 1.36).
__global__ __launch_bounds__(kBlock) void k_split_groups(TreeBuffers tb_all, int items) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int g = blockIdx.x * kWaves + wave_id(), item = g * kPartGroup + lane_id();
    static_assert(kPartGroup == 64, "a lane per item");
    if (g * kPartGroup >= items) return;
    const int sum = wave_sum_i(item < items ? tb.pitem_nleft[item] : 0);
    if (lane_id() == 0) tb.pitem_loff[g] = sum;
}

// Stable two-way compaction of a work item's rows into the children's segments with wavefront ballots and popcounts;
// where the item's rows go follows from the counts of its node's items, which the workgroup adds up itself (a node of
// 10 M rows has 4 883 of them: 20 KB from the L2). That is a square of the rows: from kPartGroupRows on a node of many
// items is added up by groups (k_split_groups). Every node's first item also leaves the children's segments and the
// pair of the next level: the child with fewer rows is built from them (ties: the left one, as
// hist_tree_builder_single.cu:466-467), the other one comes from subtraction. (Moving the gradient pairs along with the
// row ids was measured: it makes the histogram's gradient reads sequential but costs more here than it saves there.)
template <bool DIRECT, bool GROUPS, bool PLANNED>
__global__ __launch_bounds__(kBlock) void k_split_scatter(TreeBuffers tb_all, int level) {
    __shared__ int s_sum[2][kWaves];
    __shared__ int s_cnt[kPartChunk / kBlock][2][kWaves];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int *__restrict__ ridx_cur = tb.list(level);
    int *__restrict__ ridx_next = tb.list(level + 1);
    const int item = blockIdx.x;
    const NodeItem it = locate_item<PLANNED>(tb, level, item);
    if (it.x_in < 0) return;
    const int x_in = it.x_in, x = (1 << level) - 1 + x_in;
    const int2 sg = it.seg;
    const int mine = item - it.first;  // of the node's items
    const int pb = sg.x + mine * kPartChunk;
    const int pe = min(sg.y, pb + kPartChunk);
    const int lane = lane_id(), w = wave_id();
    const TreeNode nd = node_of_wave(tb, x);
    const bool splits = node_splits(nd);
    const int lch = nd.lch_index, rch = nd.rch_index;
    // all loads of the item first (unconditional, clamped positions), then one barrier for the sums of the node's counts
    // and the wavefront counts of all eight steps, then all stores
    constexpr int R = kPartChunk / kBlock;
    int row[R];
    const unsigned rights = tb.goes_right[(size_t)item * kBlock + threadIdx.x];  // bit k: the thread's k-th row goes right
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int pos = max(min(pb + k * kBlock + (int)threadIdx.x, pe - 1), 0);
        row[k] = DIRECT ? pos : ridx_cur[pos];
    }
    int before = 0, total = 0;
    if (!GROUPS || it.count <= kBlock) {
        for (int t = threadIdx.x; t < it.count; t += kBlock) {
            const int c = tb.pitem_nleft[it.first + t];
            total += c;
            before += t < mine ? c : 0;
        }
    } else {
        const int items_end = it.first + it.count;
        const int g0 = (it.first + kPartGroup - 1) / kPartGroup, g1 = items_end / kPartGroup;  // (g1 > g0: 257 items at least)
        const int own = item / kPartGroup, part = threadIdx.x / kPartGroup, t = threadIdx.x % kPartGroup;
        // the first 64 threads: items before group g0, then those from group g1 on, then those of a group of the item's own
        const int from = part == 0 ? it.first : (part == 1 ? g1 : own) * kPartGroup;
        const int to = part == 0 ? g0 * kPartGroup : part == 1 ? items_end : part == 2 && own >= g0 && own < g1 ? item : from;
        if (from + t < to) {
            const int c = tb.pitem_nleft[from + t];
            total = part < 2 ? c : 0;
            before = from + t < item ? c : 0;
        }
        const int *__restrict__ groups = tb.pitem_loff;
        for (int g = g0 + threadIdx.x; g < g1; g += kBlock) {
            const int c = groups[g];
            total += c;
            before += g < own ? c : 0;
        }
    }
    before = wave_sum_i(before);
    total = wave_sum_i(total);
    if (lane == 0) {
        s_sum[0][w] = before;
        s_sum[1][w] = total;
    }
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const bool valid = pb + k * kBlock + (int)threadIdx.x < pe;
        const bool right = (rights >> k) & 1u;
        const unsigned long long mL = __ballot(valid && !right), mR = __ballot(valid && right);
        if (lane == 0) {
            s_cnt[k][0][w] = __popcll(mL);
            s_cnt[k][1][w] = __popcll(mR);
        }
    }
    __syncthreads();
    before = total = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) {
        before += s_sum[0][i];
        total += s_sum[1][i];
    }
    if (mine == 0 && threadIdx.x == 0) {
        const bool singles = tb.singles(level + 1);
        const int nleft = splits ? total : 0, nright = (sg.y - sg.x) - nleft;
        const int2 left = splits ? make_int2(sg.x, sg.x + nleft) : make_int2(0, 0);
        const int2 right = splits ? make_int2(sg.x + nleft, sg.y) : make_int2(0, 0);
        tb.node_nleft[x_in] = nleft;
        tb.seg[lch] = left;
        tb.seg[rch] = right;
        if (singles) {
            // no parent histograms below this level (the arena is smaller than the level): every child of a split node is
            // built from its own rows, and the "pairs" of the next level are its single nodes
            tb.hpair_built[2 * x_in] = splits ? lch : -1;
            tb.hpair_built[2 * x_in + 1] = splits ? rch : -1;
            tb.hpair_plan[2 * x_in] = make_int4(splits ? lch : -1, left.x, left.y, 0);
            tb.hpair_plan[2 * x_in + 1] = make_int4(splits ? rch : -1, right.x, right.y, 0);
        } else {
            const bool build_left = nleft <= nright;
            const int built = splits ? (build_left ? lch : rch) : -1;
            const int2 bs = build_left ? left : right;
            tb.hpair_built[x_in] = built;
            tb.hpair_plan[x_in] = make_int4(built, bs.x, bs.y, 0);
        }
    }
    if (!splits) return;
    int left_base = sg.x + before;
    int right_base = sg.x + total + ((pb - sg.x) - before);
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const bool valid = pb + k * kBlock + (int)threadIdx.x < pe;
        const bool right = (rights >> k) & 1u;
        const unsigned long long mL = __ballot(valid && !right), mR = __ballot(valid && right);
        int bL = 0, bR = 0, tL = 0, tR = 0;
#pragma unroll
        for (int i = 0; i < kWaves; ++i) {
            const int cl = s_cnt[k][0][i], cr = s_cnt[k][1][i];
            if (i < w) {
                bL += cl;
                bR += cr;
            }
            tL += cl;
            tR += cr;
        }
        if (valid) {
            const int dest = right ? right_base + bR + lanes_below(mR) : left_base + bL + lanes_below(mL);
            ridx_next[dest] = row[k];
        }
        left_base += tL;
        right_base += tR;
    }
}

// The plan of a level of many nodes: its histogram work items (hpair_begin, ctl) and its nodes' partition items (pbegin), by
// one workgroup. A thread has consecutive nodes, so that one scan serves them all.
// 500 k x 28, depth 14: planned by every wavefront instead, the histogram launches of 512, 1024, 2048 and 4096 pairs took 25,
// 55, 148 and 478 us and the partition of as many nodes twice 7, 12, 19 and 31.
constexpr int kPlanBlock = 1024;
__global__ __launch_bounds__(kPlanBlock) void k_plan_level(TreeBuffers tb_all, int level, int n_pairs) {
    constexpr int NW = kPlanBlock / 64;
    __shared__ int lds[NW];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int nl = 1 << level, off = nl - 1;
    const int pairs_each = (n_pairs + kPlanBlock - 1) / kPlanBlock, p0 = min(n_pairs, (int)threadIdx.x * pairs_each);
    const int p1 = min(n_pairs, p0 + pairs_each);
    int rows = 0, built = 0;
    for (int p = p0; p < p1; ++p) {
        const int4 q = tb.hpair_plan[p];
        rows += q.x >= 0 ? q.z - q.y : 0;
        built += q.x >= 0 ? 1 : 0;
    }
    int total, n_built, n_items;
    block_excl_scan<NW>(rows, lds, &total);
    block_excl_scan<NW>(built, lds, &n_built);
    const int chunk = hist_chunk(tb, total, n_built);
    auto hist_items = [&](int p) {
        const int4 q = tb.hpair_plan[p];
        return q.x >= 0 ? (q.z - q.y + chunk - 1) / chunk : 0;
    };
    int items = 0;
    for (int p = p0; p < p1; ++p) items += hist_items(p);
    int at = block_excl_scan<NW>(items, lds, &n_items);
    for (int p = p0; p < p1; ++p) {
        tb.hpair_begin[p] = at;
        at += hist_items(p);
    }
    const int nodes_each = (nl + kPlanBlock - 1) / kPlanBlock, x0 = min(nl, (int)threadIdx.x * nodes_each);
    const int x1 = min(nl, x0 + nodes_each);
    auto part_items = [&](int x) {
        const int2 sg = tb.seg[off + x];
        return max(1, (sg.y - sg.x + kPartChunk - 1) / kPartChunk);
    };
    int n_part;
    items = 0;
    for (int x = x0; x < x1; ++x) items += part_items(x);
    at = block_excl_scan<NW>(items, lds, &n_part);
    int *__restrict__ pbegin = tb.pbegin(level);
    for (int x = x0; x < x1; ++x) {
        pbegin[x] = at;
        at += part_items(x);
    }
    if (threadIdx.x == 0) {
        tb.hpair_begin[n_pairs] = n_items;
        pbegin[nl] = n_part;
        tb.ctl[level] = LevelCtl{chunk, n_items, n_part, total};
    }
}

// Few rows (kSmallRows): a level in one launch instead of count, scatter, histogram and merge, which take 5 to 7 us each with
// nothing to do. A workgroup owns a node and a feature block: it picks the node's split, decides for every row, lays the
// children's lists down and adds up the histogram of the child with fewer rows, whose list it has in LDS, right at the
// tree's scales; the split search derives the sibling (k_eval_split<true>). Up to kSplitHistGroups workgroups share a block's
// columns (1605 x 60, depth 6: 0.105 -> 0.101 ms a tree; 16 k x 30, depth 8: 0.214 -> 0.178). Every workgroup of a node repeats
// the split, the first one stores it. The children's rows are also marked in the row -> node map, from which the end of the tree is read
// (k_map_end). Bound by its chain of dependent steps: candidates -> bins of the rows -> lists -> bins and pairs -> LDS.
// The sums are those of k_hist_dense, whose work items count at a scale that hangs on the node's rows only.
constexpr int kSmallWaves = kSmallBlock / 64;
constexpr size_t kSmallSearchBytes = sizeof(longlong2) * kEvalPackBins * kSmallWaves;
constexpr int kSmallSteps = kSmallRows / kSmallBlock;
static_assert(kSmallRowsWide <= 8 * kSmallBlock, "the steps that 16-bit bins have code for");
static_assert(kSmallRows / 2 <= kHistFlushRows, "the built child's packed sums are never drained");
static_assert(kSmallRows <= 1 << 16 && kSmallWaves == 16 && kSmallSteps % 4 == 0, "16-bit row ids, the counts of four steps per wavefront");

// 64-bit words of the histogram and of the built child's row ids (an even number: what follows is read as 16 bytes)
__host__ __device__ inline int small_words(int n, int lds_bins) { return (lds_bins + ((n / 2 + 1) * 2 + 7) / 8 + 1) / 2 * 2; }
// SEARCH: the workgroup has the built child's histogram of its columns whole, so it also derives the sibling's and searches both,
// a column and child per wavefront, into the other one of two candidate arrays (the node's own are still being read). For parts
// of up to 16 columns, so that a wavefront searches once or twice; wider ones leave it to a launch that spreads it over the chip.
// A level of 1605 x 119: 12.3 us instead of 7.5 and 7.0 in two launches; ms a tree: 1605 x 60, depth 6 0.0983 -> 0.0845, 4 k x 100
// 0.1146 -> 0.1012, 8 k x 4, depth 8 0.1326 -> 0.1160, 6 k one-hot of 5 classes 0.1320 -> 0.1183, 2 k x 600 (few levels) 0.1506 -> 0.1475.
struct SmallSearch {
    SplitCand *cand = nullptr;  // of the next level, a slot per column
    int slots = 0;
    float mcw = 0;
    bool store = false;  // the children's histograms are parents again
};
template <int LPR, bool BIN16, int STEPS, bool SEARCH>
__global__ __launch_bounds__(kSmallBlock) void k_small_level(TreeBuffers tb_all, DenseBins bins, const GHPair *__restrict__ gh,
                                                            int level, float rt_eps, float lambda, int log_split, int lds_bins,
                                                            SmallSearch search) {
    extern __shared__ __attribute__((aligned(16))) unsigned long long lds[];  // the block's histogram, then the built child's row ids
    __shared__ PickShared s_pick;
    __shared__ int s_left[STEPS * kSmallWaves];  // rows that go left, per step and wavefront
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    unsigned short *s_rows = reinterpret_cast<unsigned short *>(lds + lds_bins);
    const int fb = blockIdx.x >> log_split, part = blockIdx.x & ((1 << log_split) - 1), x_in = blockIdx.y, x = (1 << level) - 1 + x_in;
    const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
    // (all that follows from the node alone is requested at once)
    const SplitCand early = early_candidate(tb, x_in);
    const int2 sg = level == 0 ? make_int2(0, tb.n) : tb.seg[x];
    const TreeNode node = node_of_wave(tb, x);
    const QuantCtl quant = *tb.quant;
    constexpr int RPS = kSmallBlock / LPR, FPL = BIN16 ? 2 : 4, COLS = LPR * FPL, U = 8;
    const int q = threadIdx.x % LPR, rsub = threadIdx.x / LPR;
    // the part's columns and bins
    const int *__restrict__ col_off = tb.feat_lds_off + ((fb << log_split) + part) * COLS;
    const int blk0 = tb.blk_bin_begin[fb], off0 = col_off[0];
    const int bin0 = blk0 + off0, nb = (part + 1 == 1 << log_split ? tb.blk_bin_begin[fb + 1] - blk0 : col_off[COLS]) - off0;
    const int o0 = col_off[q * FPL] - off0, o1 = col_off[q * FPL + 1] - off0;
    const int o2 = BIN16 ? 0 : col_off[q * FPL + 2] - off0, o3 = BIN16 ? 0 : col_off[q * FPL + 3] - off0;
    const int row_shift = log_split + (LPR == 1 ? 2 : LPR == 2 ? 3 : LPR == 4 ? 4 : LPR == 8 ? 5 : 6);
    const int len = sg.y - sg.x, steps = (len + kSmallBlock - 1) / kSmallBlock;
    const int *__restrict__ ridx = tb.list(level);
    int row[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
        row[k] = 0;
        if (k < steps) {
            const int pos = min(sg.x + k * kSmallBlock + (int)threadIdx.x, sg.y - 1);
            row[k] = level == 0 ? pos : ridx[pos];
        }
    }
    // SEARCH: the wavefront's column and the first child that it searches (0: the built one, 1: its sibling)
    static_assert(!SEARCH || (COLS <= kSmallWaves && !BIN16), "a column per wavefront");
    const int my_col = w % COLS, my_child = w / COLS;
    const int c0 = SEARCH ? col_off[my_col] - off0 : 0;
    const int c1 = SEARCH ? (part + 1 == 1 << log_split && my_col + 1 == COLS ? nb : col_off[my_col + 1] - off0) : 0;
    longlong2 parent[4];
    PackMeta meta;
    if constexpr (SEARCH) {
        meta.load(tb, bin0 + c0, bin0 + c1);
#pragma unroll
        for (int j = 0; j < 4; ++j) parent[j] = tb.hist(level)[(size_t)x_in * tb.n_bins + max(0, bin0 + min(c0 + lane * 4 + j, c1 - 1))];
    }
    for (int i = threadIdx.x; i < nb; i += kSmallBlock) lds[i] = 0ull;
    const Picked best = pick_candidate<kSmallWaves>(tb, x_in, node.is_valid, s_pick, early);
    const bool splits = best.found && fabsf(best.c.score) > rt_eps;
    const bool first = blockIdx.x == 0 && threadIdx.x == 0;
    if (!splits) {
        if (first) {
            tb.node_nleft[x_in] = 0;
            if (node.lch_index >= 0) tb.seg[node.lch_index] = tb.seg[node.rch_index] = make_int2(0, 0);
            tb.hpair_built[x_in] = -1;
            apply_candidate(tb, x, x_in, node, best.found, best.c, rt_eps, lambda);
        }
        return;
    }
    const int f = best.c.feature;
    const int sbid = tb.split_bin != nullptr ? best.c.bin : (int)(unsigned char)best.c.bin;
    const bool dr = best.c.score < 0;
    int c = f, lo = 0, span = BIN16 ? kMissingBin16 : kMissingBin;
    if (!BIN16 && bins.feat_col != nullptr) {  // (see k_split_count)
        c = bins.feat_col[f];
        lo = bins.feat_lo[f];
        span = tb.cut_row_ptr[f + 1] - tb.cut_row_ptr[f];
    }
    const uint8_t *column = bins.col + (size_t)c * bins.col_stride * (BIN16 ? 2 : 1);
    int b[STEPS];
#pragma unroll
    for (int k = 0; k < STEPS; ++k)
        if (k < steps) b[k] = BIN16 ? (int)reinterpret_cast<const uint16_t *>(column)[row[k]] : (int)column[row[k]];
    unsigned long long left_mask[STEPS];  // (wave-uniform)
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
        left_mask[k] = 0;
        if (k < steps) {
            const int t = b[k] - lo;
            const bool right = ((unsigned)t >= (unsigned)span) ? dr : (t >= sbid);
            left_mask[k] = __ballot(!right && k * kSmallBlock + (int)threadIdx.x < len);
        }
        if (lane == 0) s_left[k * kSmallWaves + w] = __popcll(left_mask[k]);
    }
    __syncthreads();
    // lefts before every (step, wavefront), and of all: by every wavefront for itself, four steps at a time
    int upto[(STEPS + 3) / 4], nleft = 0;
#pragma unroll
    for (int k = 0; k < (STEPS + 3) / 4; ++k) {
        upto[k] = 0;
        if (k * 4 < steps) {
            const int own = k * 64 + lane < STEPS * kSmallWaves ? s_left[k * 64 + lane] : 0;
            const int inc = wave_scan_i(own);
            upto[k] = nleft + inc - own;
            nleft += read_lane(inc, 63);
        }
    }
    const int nright = len - nleft;
    // the child with fewer rows is built from them (ties: the left one, as hist_tree_builder_single.cu:466-467)
    const bool build_left = nleft <= nright;
    const int m = build_left ? nleft : nright;
    int *__restrict__ ridx_next = tb.list(level + 1);
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
        const int i = k * kSmallBlock + (int)threadIdx.x;
        const int before = read_lane(upto[k / 4], k % 4 * kSmallWaves + w);  // (out here: the lane that is read may have no row)
        if (k < steps && i < len) {
            const int lefts = before + lanes_below(left_mask[k]);
            const bool left = (left_mask[k] >> lane & 1ull) != 0;
            const int at = left ? lefts : i - lefts;  // in the child's list
            if (left == build_left) s_rows[at] = (unsigned short)row[k];
            if (blockIdx.x == 0) {
                ridx_next[sg.x + (left ? at : nleft + at)] = row[k];
                tb.nid[row[k]] = left ? node.lch_index : node.rch_index;
            }
        }
    }
    __syncthreads();
    const int h_bits = quant.h_bits;
    const int rows = max(1, min(m, quant.flush_rows));
    const int shift_g = item_shift(quant.gq_max, rows, 63 - h_bits), shift_h = quant.h_integer ? 0 : item_shift(quant.hq_max, rows, h_bits);
    const float scale_g = ldexpf(quant.scale_g, -shift_g), scale_h = ldexpf(quant.scale_h, -shift_h);
    const bool word_lane = bins.gh_lane >= 0 && part * LPR + q == bins.gh_lane;
    const uint8_t *blk = bins.data + (size_t)fb * bins.block_stride;
    for (int base = 0; base < m; base += RPS * U) {
        unsigned pk[U];
        GHPair s[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned r = s_rows[min(base + rsub + u * RPS, m - 1)];
            pk[u] = *reinterpret_cast<const unsigned *>(blk + ((r << row_shift) + (unsigned)(part * LPR + q) * 4));
            s[u] = gh[r];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u * RPS >= m) break;  // (uniform)
            const unsigned v = base + rsub + u * RPS < m && !word_lane ? pk[u] : 0xffffffffu;
            add_row<BIN16>(lds, v, s[u], scale_g, scale_h, h_bits, o0, o1, o2, o3);
        }
    }
    __syncthreads();
    const int built = build_left ? node.lch_index : node.rch_index;
    const unsigned long long h_mask = (1ull << h_bits) - 1ull;
    auto unpacked = [&](unsigned long long t) {
        const unsigned long long low = t & h_mask;
        return make_longlong2(((long long)(t - low) >> h_bits) << shift_g, (long long)low << shift_h);
    };
    if constexpr (!SEARCH) {
        longlong2 *out = tb.hist(level + 1) + (size_t)(built - ((2 << level) - 1)) * tb.n_bins + bin0;
        for (int i = threadIdx.x; i < nb; i += kSmallBlock) out[i] = unpacked(lds[i]);
    } else if (const int column = ((fb << log_split) + part) * COLS + my_col; column < search.slots) {
        // the children's sums as apply_split computes them
        GHPair ls = best.c.bin != 0 ? best.c.left : GHPair{0, 0};
        if (!(best.c.score < 0)) {
            ls.g += best.c.miss.g;
            ls.h += best.c.miss.h;
        }
        const GHPair rs{node.sum_gh_pair.g - ls.g, node.sum_gh_pair.h - ls.h};
        longlong2 *s_v = reinterpret_cast<longlong2 *>(lds + small_words(tb.n, lds_bins)) + w * kEvalPackBins;
        TreeBuffers next = tb;
        next.cand = search.cand + (size_t)blockIdx.z * tb.max_level_nodes * search.slots;
        next.n_packs = search.slots;
        for (int child = my_child; child < 2; child += kSmallWaves / COLS) {
            const bool left = build_left == (child == 0);
            const int x_child = 2 * x_in + (left ? 0 : 1);
            longlong2 *out = tb.hist(level + 1) + (size_t)x_child * tb.n_bins + bin0;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int b = c0 + lane * 4 + j;
                longlong2 v = make_longlong2(0, 0);
                if (b < c1) {
                    v = unpacked(lds[b]);
                    if (child == 1) v = make_longlong2(parent[j].x - v.x, parent[j].y - v.y);
                    if (search.store) out[b] = v;
                }
                s_v[lane * 4 + j] = v;
            }
            wave_lds_sync();
            search_pack(next, meta, s_v, x_child, column, true, bin0 + c0, bin0 + c1, left ? ls : rs, quant.inv_g, quant.inv_h, search.mcw, lambda);
            wave_lds_sync();
        }
    }
    if (first) {
        tb.node_nleft[x_in] = nleft;
        tb.seg[node.lch_index] = make_int2(sg.x, sg.x + nleft);
        tb.seg[node.rch_index] = make_int2(sg.x + nleft, sg.y);
        tb.hpair_built[x_in] = built;
        atomicAdd(&tb.ctl[level + 1].n_hitems, 1);
        atomicAdd(&tb.ctl[level + 1].rows_built, m);
        apply_candidate(tb, x, x_in, node, best.found, best.c, rt_eps, lambda);
    }
}

// A run of a node's rows: run / kPartChunk consecutive partition items of it, at least one run for every node.
struct NodeRun {
    int x_in;        // node within the level, -1: there is no such run
    int first, count;  // runs of the node, numbered node by node
    int pitem, pitems;  // its partition items
    int2 seg;
};
__device__ __forceinline__ NodeRun locate_run(const TreeBuffers &tb, int level, int item, int run) {
    const int nl = 1 << level;
    const int2 *__restrict__ segs = tb.seg + (nl - 1);
    NodeRun out;
    out.x_in = -1;
    if (level == 0) {
        out.first = out.pitem = 0;
        out.count = max(1, (tb.n + run - 1) / run);
        out.pitems = max(1, (tb.n + kPartChunk - 1) / kPartChunk);
        out.seg = make_int2(0, tb.n);
        if (item < out.count) out.x_in = 0;
        return out;
    }
    constexpr int A = 4;  // 64 nodes each, loaded together
    int carry = 0, pcarry = 0;
    for (int base = 0; base < nl; base += A * 64) {
        int2 sg[A];
#pragma unroll
        for (int a = 0; a < A; ++a) sg[a] = segs[min(base + a * 64 + lane_id(), nl - 1)];
#pragma unroll
        for (int a = 0; a < A; ++a) {
            if (base + a * 64 >= nl) break;
            const bool in = base + a * 64 + lane_id() < nl;
            const int rows = sg[a].y - sg[a].x;
            const int cnt = in ? max(1, (rows + run - 1) / run) : 0, pcnt = in ? max(1, (rows + kPartChunk - 1) / kPartChunk) : 0;
            const int inc = wave_scan_i(cnt), ex = carry + inc - cnt, pinc = wave_scan_i(pcnt);
            const unsigned long long owner = __ballot(item >= ex && item < ex + cnt);
            if (owner != 0ull) {
                const int l = __ffsll((long long)owner) - 1;
                out.x_in = base + a * 64 + l;
                out.first = read_lane(ex, l);
                out.count = read_lane(cnt, l);
                out.pitem = pcarry + read_lane(pinc - pcnt, l);
                out.pitems = read_lane(pcnt, l);
                out.seg = make_int2(read_lane(sg[a].x, l), read_lane(sg[a].y, l));
                return out;
            }
            carry += read_lane(inc, 63);
            pcarry += read_lane(pinc, 63);
        }
    }
    return out;
}

// Moderately many rows (split_hist_plan): k_split_scatter and the next level's k_hist_dense in one launch. A workgroup owns a
// run of S partition items of a node and a feature block. The counts of the node's items tell it where the run's rows go and
// which child has fewer rows; those of them that go there meet in LDS, and their histogram is a work item of the next level,
// stored packed at the child's own scale (item_shift), so its sums are k_hist_dense's whatever the items. The first block
// stores the lists. Bound by its chain of dependent steps - segments, decisions with rows and counts, lists, records - and by
// the LDS, which adds about 8 pairs a nanosecond and CU to random bins: 1000 rows x 28 in 3.5 us.
// 500 k x 28: 9.5 us with 1 item, where scatter, gap and histogram (which looks for its pair and fetches the row ids again) took
// 13.3; a tree of depth 8 0.281 -> 0.266 ms (0.263 and 0.261 without and with the write-through; 900 k x 28 0.296 and 0.290).
// Measured and not kept: every row's addend rounded once, by a thread of its own, and passed on through LDS (the LDS is what it
// waits for: 4.6 -> 6.1 us in that part); the decisions taken here as well, the runs of a node telling each other their counts
// through agent-scope atomics (a launch less, but 245 workgroups that look at 245 words each: a tree 0.32 instead of 0.27 ms).
constexpr int kRunWaves = kHistBlock / 64;
constexpr int kRunHalves = kPartChunk / kHistBlock;  // rows of a partition item per thread
static_assert(kSplitHistMost * kPartChunk <= kHistFlushRows, "a run's packed sums are never drained");
static_assert(kRunHalves == 2 && kBlock * 8 == kPartChunk, "the mapping of k_split_count's decision bytes");
template <int LPR, bool BIN16, bool GHW, int S>
__global__ __launch_bounds__(kHistBlock) __attribute__((amdgpu_waves_per_eu(8)))
void k_split_hist(TreeBuffers tb_all, DenseBins bins, const GHPair *__restrict__ gh, int level, int log_split, int lds_bins) {
    constexpr int R = S * kRunHalves;  // rows per thread
    constexpr int E = R * kRunWaves;   // counts of the run: one per round and wavefront
    extern __shared__ unsigned long long lds[];  // the histogram, then the rows to add up
    __shared__ int s_cnt[E < 64 ? 64 : E];
    __shared__ int s_sum[2][kRunWaves];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    int *s_rows = reinterpret_cast<int *>(lds + lds_bins);
    const int fb = blockIdx.x >> log_split, part = blockIdx.x & ((1 << log_split) - 1), item = blockIdx.y;
    const NodeRun it = locate_run(tb, level, item, S * kPartChunk);
    if (it.x_in < 0) return;
    // the part's columns and bins
    constexpr int FPL = BIN16 ? 2 : 4, COLS = LPR * FPL;
    const int *__restrict__ col_off = tb.feat_lds_off + ((fb << log_split) + part) * COLS;
    const int blk0 = tb.blk_bin_begin[fb], off0 = col_off[0];
    const int bin0 = blk0 + off0, nb = (part + 1 == 1 << log_split ? tb.blk_bin_begin[fb + 1] - blk0 : col_off[COLS]) - off0;
    const int nl = 1 << level, x_in = it.x_in, x = nl - 1 + x_in;
    const int2 sg = it.seg;
    const int mine = item - it.first;  // of the node's runs
    const int pb = sg.x + mine * (S * kPartChunk);
    const int pe = min(sg.y, pb + S * kPartChunk);
    const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
    const int *__restrict__ ridx = tb.list(level);
    const TreeNode nd = node_of_wave(tb, x);
    const bool splits = node_splits(nd);
    const int lch = nd.lch_index, rch = nd.rch_index;
    int row[R];
    unsigned rights[S];
#pragma unroll
    for (int k = 0; k < S; ++k)
        rights[k] = tb.goes_right[(size_t)(it.pitem + min(mine * S + k, it.pitems - 1)) * kBlock + threadIdx.x % kBlock];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int pos = max(min(pb + k * kHistBlock + (int)threadIdx.x, pe - 1), 0);
        row[k] = level == 0 ? pos : ridx[pos];
    }
    static_assert(kSplitHistRows / kPartChunk <= kHistBlock, "a partition item of the node per thread");
    int total = tb.pitem_nleft[it.pitem + min((int)threadIdx.x, it.pitems - 1)];
    if ((int)threadIdx.x >= it.pitems) total = 0;
    int before = (int)threadIdx.x < mine * S ? total : 0;
    const QuantCtl quant = *tb.quant;
    for (int i = threadIdx.x; i < nb; i += kHistBlock) lds[i] = 0ull;
    before = wave_sum_i(before);
    total = wave_sum_i(total);
    if (lane == 0) {
        s_sum[0][w] = before;
        s_sum[1][w] = total;
    }
    unsigned long long left_mask[R];  // (wave-uniform)
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const bool valid = pb + k * kHistBlock + (int)threadIdx.x < pe;
        // (k_split_count's thread t decides for the rows t, t + 256, ... of a partition item, bit by bit)
        const bool right = rights[k / kRunHalves] >> (k % kRunHalves * (8 / kRunHalves) + threadIdx.x / kBlock) & 1u;
        left_mask[k] = __ballot(valid && !right);
        if (lane == 0) s_cnt[k * kRunWaves + w] = __popcll(left_mask[k]);
    }
    __syncthreads();
    before = wave_sum_i(lane < kRunWaves ? s_sum[0][lane % kRunWaves] : 0);
    total = wave_sum_i(lane < kRunWaves ? s_sum[1][lane % kRunWaves] : 0);
    const int nleft = splits ? total : 0, nright = (sg.y - sg.x) - nleft;
    // the child with fewer rows is built from them (ties: the left one, as hist_tree_builder_single.cu:466-467)
    const bool build_left = nleft <= nright;
    const int built = splits ? (build_left ? lch : rch) : -1;
    if (blockIdx.x == 0 && mine == 0 && threadIdx.x == 0) {
        tb.node_nleft[x_in] = nleft;
        tb.seg[lch] = splits ? make_int2(sg.x, sg.x + nleft) : make_int2(0, 0);
        tb.seg[rch] = splits ? make_int2(sg.x + nleft, sg.y) : make_int2(0, 0);
        tb.hpair_built[x_in] = built;
        tb.hpair_begin[x_in] = it.first;
        if (x_in == nl - 1) tb.hpair_begin[nl] = it.first + it.count;
        if (splits) {
            atomicAdd(&tb.ctl[level + 1].n_hitems, it.count);
            atomicAdd(&tb.ctl[level + 1].rows_built, min(nleft, nright));
        }
    }
    if (!splits) return;
    // lefts of the run before every (round, wavefront)
    int sum[E > 64 ? E / 64 : 1], upto[E > 64 ? E / 64 : 1], lefts = 0;
#pragma unroll
    for (int q = 0; q < (E > 64 ? E / 64 : 1); ++q) {
        sum[q] = q * 64 + lane < E ? s_cnt[q * 64 + lane] : 0;
        const int inc = wave_scan_i(sum[q]);
        upto[q] = lefts + inc - sum[q];
        lefts += read_lane(inc, 63);
    }
    const int m = build_left ? lefts : pe - pb - lefts;  // rows of the run to add up
    int *__restrict__ ridx_next = tb.list(level + 1);
    const int left_base = sg.x + before, right_base = sg.x + total + ((pb - sg.x) - before);
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int i = k * kHistBlock + (int)threadIdx.x;
        const int e = k * kRunWaves;
        const int l = read_lane(upto[e / 64], e % 64 + w) + lanes_below(left_mask[k]);  // lefts before row i
        const bool left = (left_mask[k] >> lane & 1ull) != 0;
        if (pb + i < pe) {
            const int at = left ? l : i - l;
            if (left == build_left) s_rows[at] = row[k];
            if (blockIdx.x == 0) ridx_next[left ? left_base + at : right_base + at] = row[k];
        }
    }
    __syncthreads();
    // The rows in batches: a batch's loads are issued together, the first ones before the scales are worked out.
    constexpr int RPS = kHistBlock / LPR, U = LPR >= 16 ? 8 : 4;
    const int q = threadIdx.x % LPR, rsub = threadIdx.x / LPR;
    const int row_shift = log_split + (LPR == 1 ? 2 : LPR == 2 ? 3 : LPR == 4 ? 4 : LPR == 8 ? 5 : 6);
    const uint8_t *blk = bins.data + (size_t)fb * bins.block_stride;
    unsigned pk[U];
    GHPair s[U];  // (GHW: the word, in the first slot)
    auto load_rows = [&](int base) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u * RPS >= m) break;  // (uniform)
            const unsigned r = (unsigned)s_rows[min(base + rsub + u * RPS, m - 1)];
            const uint8_t *record = blk + (r << row_shift);
            pk[u] = *reinterpret_cast<const unsigned *>(record + (unsigned)(part * LPR + q) * 4);
            if (GHW) s[u].g = __uint_as_float(*reinterpret_cast<const unsigned *>(record + (unsigned)bins.gh_lane * 4));
            else s[u] = *reinterpret_cast<const GHPair *>(reinterpret_cast<const char *>(gh) + r * 8u);
        }
    };
    if (m > 0) load_rows(0);
    const int h_bits = quant.h_bits;
    const int rows = max(1, min(min(nleft, nright), quant.flush_rows));
    const int shift_g = item_shift(quant.gq_max, rows, 63 - h_bits), shift_h = quant.h_integer ? 0 : item_shift(quant.hq_max, rows, h_bits);
    if (blockIdx.x == 0 && threadIdx.x == 0) tb.hitem_shift[item] = make_int2(shift_g, shift_h);
    const float scale_g = ldexpf(quant.scale_g, -shift_g), scale_h = ldexpf(quant.scale_h, -shift_h);
    const int o0 = col_off[q * FPL] - off0, o1 = col_off[q * FPL + 1] - off0;
    const int o2 = BIN16 ? 0 : col_off[q * FPL + 2] - off0, o3 = BIN16 ? 0 : col_off[q * FPL + 3] - off0;
    const bool word_lane = bins.gh_lane >= 0 && part * LPR + q == bins.gh_lane;
    for (int base = 0; base < m; base += RPS * U) {
        if (base > 0) load_rows(base);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (base + u * RPS >= m) break;  // (uniform)
            const GHPair sv = GHW ? pair_from_word(bins.gh_objective, __float_as_uint(s[u].g)) : s[u];
            const unsigned v = base + rsub + u * RPS < m && !word_lane ? pk[u] : 0xffffffffu;
            add_row<BIN16>(lds, v, sv, scale_g, scale_h, h_bits, o0, o1, o2, o3);
        }
    }
    __syncthreads();
    unsigned long long *out = reinterpret_cast<unsigned long long *>(tb.partial) + (size_t)item * tb.n_bins + bin0;
    // (written through: what the launch leaves in the L2s is written back when it ends, and everything waits for that)
    for (int i = threadIdx.x; i < nb; i += kHistBlock) __hip_atomic_store(&out[i], lds[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

}  // namespace

static int most_partition_items(const TreeBuffers &tb, int level) {
    return level == 0 ? std::max(1, (tb.n + kPartChunk - 1) / kPartChunk) : tb.n / kPartChunk + (1 << level);
}

static size_t split_hist_lds(int lds_bins, int run) { return (size_t)lds_bins * 8 + (size_t)run * 4; }

int split_hist_run(const TreeBuffers &tb, int n_class) {
    if (tb.n >= kSplitHistRows || tb.depth > kSmallDepth || tb.planned(tb.depth - 1)) return 0;
    auto stored = [&](int run) { return (size_t)((tb.n + run - 1) / run) * tb.n_bins * 8 * n_class; };
    if (tb.n < kSplitHistOneRows && stored(kPartChunk) <= kSplitHistOneBytes) return kPartChunk;
    for (int run = 2 * kPartChunk; run <= kSplitHistMost * kPartChunk; run *= 2)
        if (stored(run) <= kSplitHistBytes) return run;
    return 0;
}

SplitHistPlan split_hist_plan(const TreeBuffers &tb, const DenseBins &bins, const int *part_bins, int n_class) {
    SplitHistPlan plan;
    for (int run = split_hist_run(tb, n_class); run > 0 && run <= kSplitHistMost * kPartChunk; run *= 2) {
        const long runs = (tb.n + run - 1) / run;
        int parts = 0;  // (log2)
        while (4 << (parts + 1) <= bins.W * bins.bin_bytes && (runs * bins.n_blocks * n_class << (parts + 1)) <= kSplitHistGroups) ++parts;
        if (split_hist_lds(part_bins[parts], run) + 4096 > kLdsBytes) continue;
        plan.run = run;
        plan.log_split = parts;
        plan.lds_bins = part_bins[parts];
        plan.walk = n_class > 1 && (long)tb.n * n_class >= kWalkRows && bins.n_blocks == 1 && bins.bin_bytes == 1 && bins.W <= 32 && tb.split_bin == nullptr;
        return plan;
    }
    return plan;
}

template <int LPR, bool BIN16, bool GHW, int S>
static void split_hist_launch(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level, const SplitHistPlan &plan,
                              int n_class) {
    constexpr int run = S * kPartChunk;
    const size_t lds = split_hist_lds(plan.lds_bins, run);
    static LdsOptIn opt_in;
    if (lds > 48 * 1024) opt_in({reinterpret_cast<const void *>(&k_split_hist<LPR, BIN16, GHW, S>)});
    const dim3 grid(bins.n_blocks << plan.log_split, level == 0 ? (tb.n + run - 1) / run : tb.n / run + (1 << level), n_class);
    k_split_hist<LPR, BIN16, GHW, S><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, level, plan.log_split, plan.lds_bins);
}

template <int LPR, bool BIN16, bool GHW>
static void split_hist_run_launch(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level,
                                  const SplitHistPlan &plan, int n_class) {
    if (plan.run == kPartChunk) split_hist_launch<LPR, BIN16, GHW, 1>(s, tb, bins, gh, level, plan, n_class);
    else if (plan.run == 2 * kPartChunk) split_hist_launch<LPR, BIN16, GHW, 2>(s, tb, bins, gh, level, plan, n_class);
    else if (plan.run == 4 * kPartChunk) split_hist_launch<LPR, BIN16, GHW, 4>(s, tb, bins, gh, level, plan, n_class);
    else fatal("runs of %d rows", plan.run);
}

void launch_partition_hist(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level, const SplitHistPlan &plan,
                           float rt_eps, float lambda, int n_class) {
    const dim3 items(most_partition_items(tb, level), 1, n_class);
    const bool last = level == tb.depth - 1;
    if (plan.walk) {  // (bytes)
        if (last) return launch_best_update(s, tb, level, rt_eps, lambda, n_class);
        if (level == 0) k_split_count<true, uint8_t, true, false><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda);
        else k_split_count<false, uint8_t, true, false><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda);
    }
#define TGBM_SPLIT_MAP(T)                                                                                                          \
    if (last && level == 0) k_split_count<true, T, true, false, 2><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda);       \
    else if (last) k_split_count<false, T, true, false, 2><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda);               \
    else if (level == 0) k_split_count<true, T, true, false, 1><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda);          \
    else k_split_count<false, T, true, false, 1><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda)
    else if (bins.bin_bytes == 2) { TGBM_SPLIT_MAP(uint16_t); }
    else { TGBM_SPLIT_MAP(uint8_t); }
#undef TGBM_SPLIT_MAP
    if (last) return;
    const bool words = bins.gh_lane >= 0 && bins.gh_fresh;
#define TGBM_SPLIT_HIST(LPR)                                                                                        \
    if (bins.bin_bytes == 2) split_hist_run_launch<LPR, true, false>(s, tb, bins, gh, level, plan, n_class);          \
    else if (words) split_hist_run_launch<LPR, false, true>(s, tb, bins, gh, level, plan, n_class);                  \
    else split_hist_run_launch<LPR, false, false>(s, tb, bins, gh, level, plan, n_class);                             \
    break
    switch (bins.W * bins.bin_bytes >> plan.log_split) {  // bytes per row of a part
        case 4: TGBM_SPLIT_HIST(1);
        case 8: TGBM_SPLIT_HIST(2);
        case 16: TGBM_SPLIT_HIST(4);
        case 32: TGBM_SPLIT_HIST(8);
        case 64: TGBM_SPLIT_HIST(16);
        default: fatal("unsupported dense block width %d x %d bytes", bins.W, bins.bin_bytes);
    }
#undef TGBM_SPLIT_HIST
}

void launch_partition_dense(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, int level, bool update,
                            float rt_eps, float lambda, int n_class) {
    if (level == tb.depth - 1) return;  // the last level's children never get row lists (see k_tree_end)
    const int most = most_partition_items(tb, level);
    const dim3 items(most, 1, n_class);
    const bool planned = tb.planned(level);
#define TGBM_SPLIT_COUNT(D, T, U, P) k_split_count<D, T, U, P><<<items, kBlock, 0, s>>>(tb, bins, level, rt_eps, lambda)
#define TGBM_SPLIT_COUNT_LEVEL(T, U)                           \
    if (level == 0) TGBM_SPLIT_COUNT(true, T, U, false);       \
    else if (planned) TGBM_SPLIT_COUNT(false, T, U, true);     \
    else TGBM_SPLIT_COUNT(false, T, U, false)
    if (bins.bin_bytes == 2) {
        if (update) { TGBM_SPLIT_COUNT_LEVEL(uint16_t, true); }
        else { TGBM_SPLIT_COUNT_LEVEL(uint16_t, false); }
    } else {
        if (update) { TGBM_SPLIT_COUNT_LEVEL(uint8_t, true); }
        else { TGBM_SPLIT_COUNT_LEVEL(uint8_t, false); }
    }
#undef TGBM_SPLIT_COUNT_LEVEL
#undef TGBM_SPLIT_COUNT
    const bool groups = tb.n >= kPartGroupRows;
    if (groups) k_split_groups<<<dim3((most + kPartGroup * kWaves - 1) / (kPartGroup * kWaves), 1, n_class), kBlock, 0, s>>>(tb, most);
#define TGBM_SPLIT_SCATTER(G)                                                      \
    if (level == 0) k_split_scatter<true, G, false><<<items, kBlock, 0, s>>>(tb, level);   \
    else if (planned) k_split_scatter<false, G, true><<<items, kBlock, 0, s>>>(tb, level); \
    else k_split_scatter<false, G, false><<<items, kBlock, 0, s>>>(tb, level)
    if (groups) { TGBM_SPLIT_SCATTER(true); }
    else { TGBM_SPLIT_SCATTER(false); }
#undef TGBM_SPLIT_SCATTER
    if (tb.planned(level + 1)) k_plan_level<<<dim3(1, 1, n_class), kPlanBlock, 0, s>>>(tb, level + 1, tb.n_hpairs(level + 1));
}

static size_t small_lds(const TreeBuffers &tb, int lds_bins) { return (size_t)small_words(tb.n, lds_bins) * 8; }

bool small_levels_fit(const TreeBuffers &tb) {
    return tb.n <= kSmallRows && tb.depth <= kSmallDepth && small_lds(tb, tb.max_block_bins) + 4096 <= kLdsBytes;
}

struct SmallLaunch {
    int level, log_split, lds_bins, n_class;
    float rt_eps, lambda;
    SmallSearch search;  // cand nullptr: none
};

template <int LPR, bool BIN16, int STEPS, bool SEARCH>
static void small_level_launch(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, const SmallLaunch &l) {
    const size_t lds = small_lds(tb, l.lds_bins) + (SEARCH ? kSmallSearchBytes : 0);
    static LdsOptIn opt_in;
    if (lds > 48 * 1024)  // (with the kernel's own tables more than the default window)
        opt_in({reinterpret_cast<const void *>(&k_small_level<LPR, BIN16, STEPS, SEARCH>)});
    k_small_level<LPR, BIN16, STEPS, SEARCH><<<dim3(bins.n_blocks << l.log_split, 1 << l.level, l.n_class), kSmallBlock, lds, s>>>(
        tb, bins, gh, l.level, l.rt_eps, l.lambda, l.log_split, l.lds_bins, l.search);
}

// (the code of steps that no node of the data can have is not only skipped but left out, see k_small_level)
template <int LPR, bool BIN16, bool SEARCH>
static void small_level_steps(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, const SmallLaunch &l) {
    const int steps = (tb.n + kSmallBlock - 1) / kSmallBlock;
    if (steps <= 2) small_level_launch<LPR, BIN16, 2, SEARCH>(s, tb, bins, gh, l);
    else if (steps <= 4) small_level_launch<LPR, BIN16, 4, SEARCH>(s, tb, bins, gh, l);
    else if (steps <= 8) small_level_launch<LPR, BIN16, 8, SEARCH>(s, tb, bins, gh, l);
    else if constexpr (!BIN16) small_level_launch<LPR, BIN16, kSmallSteps, SEARCH>(s, tb, bins, gh, l);
    else fatal("%d rows of 16-bit bins", tb.n);
}

bool launch_small_level(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level, float rt_eps,
                        float lambda, const int *part_bins, int n_class, SplitCand *next_cand, float mcw) {
    if (level == tb.depth - 1) return false;
    // (up to a workgroup per CU a block's columns are shared out, see kSplitHistGroups)
    SmallLaunch l{level, 0, 0, n_class, rt_eps, lambda, {}};
    while (4 << (l.log_split + 1) <= bins.W * bins.bin_bytes && ((long)bins.n_blocks * n_class << (level + l.log_split + 1)) <= kSplitHistGroups) ++l.log_split;
    l.lds_bins = part_bins[l.log_split];
    const int row_bytes = bins.W * bins.bin_bytes >> l.log_split;  // of a part
    const bool search = next_cand != nullptr && bins.bin_bytes == 1 && row_bytes <= kSmallWaves &&
                        small_lds(tb, l.lds_bins) + kSmallSearchBytes + 8192 <= kLdsBytes;
    if (search) l.search = SmallSearch{next_cand, bins.n_cols, mcw, level + 1 < tb.depth - 1};
#define TGBM_SMALL_LEVEL(LPR)                                                                        \
    if (bins.bin_bytes == 2) small_level_steps<LPR, true, false>(s, tb, bins, gh, l);                \
    else if (LPR <= 4 && search) small_level_steps<LPR, false, (LPR <= 4)>(s, tb, bins, gh, l);      \
    else small_level_steps<LPR, false, false>(s, tb, bins, gh, l);                                   \
    break
    switch (row_bytes) {
        case 4: TGBM_SMALL_LEVEL(1);
        case 8: TGBM_SMALL_LEVEL(2);
        case 16: TGBM_SMALL_LEVEL(4);
        case 32: TGBM_SMALL_LEVEL(8);
        case 64: TGBM_SMALL_LEVEL(16);
        default: fatal("unsupported dense block width %d x %d bytes", bins.W, bins.bin_bytes);
    }
#undef TGBM_SMALL_LEVEL
    return search;
}

}  // namespace tgbm
