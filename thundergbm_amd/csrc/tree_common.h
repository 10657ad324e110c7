// What the tree-building kernel sources share: workgroup scans and sums, the record of a node's split, the plan of a
// level's histogram work items.
#pragma once
#include "device_api.h"
#include "kernel_common.h"

namespace tgbm {
namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;
constexpr int kHistMinChunk = 1024;
constexpr int kHistBlock = 1024;      // threads per histogram workgroup (they share one LDS histogram)

// Exclusive scan of one int per thread over a block of NW wavefronts; lds needs NW ints.
template <int NW = kWaves>
__device__ int block_excl_scan(int v, int *lds, int *total) {
    int lane = lane_id(), w = wave_id();
    const int inc = wave_scan_i(v);
    if (lane == 63) lds[w] = inc;
    __syncthreads();
    int base = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        int c = lds[i];
        if (i < w) base += c;
        tot += c;
    }
    *total = tot;
    __syncthreads();
    return base + inc - v;
}

__device__ int block_sum(int v, int *lds) {
    v = wave_sum_i(v);
    if (lane_id() == 0) lds[wave_id()] = v;
    __syncthreads();
    int tot = 0;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) tot += lds[i];
    __syncthreads();
    return tot;
}

__device__ __forceinline__ float wave_sum_f(float v) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) v += __shfl_xor(v, d);
    return v;
}

// A node's record for a whole wavefront, by words: its flags as bytes, which scalar loads do not have, were a vector load that
// the wavefront waited for in front of its rows' (k_small_level of 10 k x 8 14.0 -> 13.85 us, of 1605 x 119 11.9 -> 11.7).
__device__ __forceinline__ TreeNode node_of_wave(const TreeBuffers &tb, int x) {
    typedef int __attribute__((may_alias)) Word;
    static_assert(sizeof(TreeNode) == 48 && offsetof(TreeNode, lch_index) == 4 && offsetof(TreeNode, split_feature_id) == 24 &&
                      offsetof(TreeNode, is_leaf) == 34 && offsetof(TreeNode, is_valid) == 35 && offsetof(TreeNode, is_pruned) == 36,
                  "TreeNode layout");
    const Word *__restrict__ w = reinterpret_cast<const Word *>(tb.nodes + x);
    TreeNode node;
    node.final_id = w[0];
    node.lch_index = w[1];
    node.rch_index = w[2];
    node.parent_index = w[3];
    node.gain = __int_as_float(w[4]);
    node.base_weight = __int_as_float(w[5]);
    node.split_feature_id = w[6];
    node.split_value = __int_as_float(w[7]);
    const unsigned flags = (unsigned)w[8];
    node.split_bid = (unsigned char)flags;
    node.default_right = (flags >> 8 & 0xffu) != 0;
    node.is_leaf = (flags >> 16 & 0xffu) != 0;
    node.is_valid = flags >> 24 != 0;
    node.is_pruned = (w[9] & 0xff) != 0;
    node.sum_gh_pair = GHPair{__int_as_float(w[10]), __int_as_float(w[11])};
    return node;
}

// Node x (x_in within its level) stays a leaf: none of its candidates can split it, or it has none.
__device__ __forceinline__ void no_split(const TreeBuffers &tb, int x, int x_in) {
    SplitPoint z{};
    z.nid = x;
    z.split_fea_id = -1;
    TreeNode &node = tb.nodes[x];
    const int lch = node.lch_index, rch = node.rch_index;
    tb.sp[x_in] = z;
    node.is_leaf = true;
    tb.nodes[lch].is_valid = false;
    tb.nodes[rch].is_valid = false;
}

// The split record of node x from its best candidate c (the split feature and the candidate's bin within it), applied to
// the tree: hist_tree_builder_single.cu:365-389 and update_tree, :860-899. `node` is a copy that was loaded before: a
// load that follows a store waits for the store to reach memory, so everything is read first and written last.
// fval: cut_val[c.index - 1], or cut_val[c.index] for the first bin of a feature
__device__ __forceinline__ void apply_split(const TreeBuffers &tb, int x, int x_in, TreeNode node, const SplitCand &c,
                                            int f, int bin, float fval, float rt_eps, float lambda) {
    SplitPoint s{};
    s.split_fea_id = f;
    s.nid = x;
    s.gain = fabsf(c.score);
    s.split_bid = (int)(unsigned char)bin;
    s.fea_missing_gh = c.miss;
    s.default_right = c.score < 0;
    s.best_index = c.index;
    if (bin != 0) {
        s.lch_sum_gh = c.left;
        s.fval = fval;
    } else {
        s.lch_sum_gh = GHPair{0, 0};
        s.fval = (float)((double)(fval - fabsf(fval)) - 1e-5);
    }
    TreeNode &out = tb.nodes[x];
    TreeNode &l = tb.nodes[node.lch_index];
    TreeNode &r = tb.nodes[node.rch_index];
    if (s.gain > rt_eps) {
        GHPair ls = s.lch_sum_gh;
        if (!s.default_right) {
            ls.g += s.fea_missing_gh.g;
            ls.h += s.fea_missing_gh.h;
        }
        GHPair rs{node.sum_gh_pair.g - ls.g, node.sum_gh_pair.h - ls.h};
        const float lw = -ls.g / (ls.h + lambda), rw = -rs.g / (rs.h + lambda);
        out.gain = s.gain;
        out.split_feature_id = f;
        out.split_value = s.fval;
        out.split_bid = (unsigned char)s.split_bid;
        out.default_right = s.default_right != 0;
        if (tb.split_bin != nullptr) tb.split_bin[x] = bin;
        l.is_valid = true;
        r.is_valid = true;
        l.sum_gh_pair = ls;
        r.sum_gh_pair = rs;
        l.base_weight = lw;
        r.base_weight = rw;
    } else {
        out.is_leaf = true;
        l.is_valid = false;
        r.is_valid = false;
    }
    tb.sp[x_in] = s;
}

// Rows per histogram work item of a level that builds n_built nodes of `total` rows. Every built node adds up to one
// partly filled item: the items are sized so that their number stays within target_hitems (= the workgroups the chip
// holds at once; one more would run as a second round).
__device__ __forceinline__ int hist_chunk(const TreeBuffers &tb, int total, int n_built) {
    const int room = max(tb.target_hitems / 4, tb.target_hitems - n_built);
    const int chunk = (total + room - 1) / room;
    return max(kHistMinChunk, (chunk + 255) / 256 * 256);
}

// The owner of `item` among n >= 1 owners whose items begin at begin[0] = 0, ..., begin[n] (item < begin[n]; owners may be
// empty), found by a wavefront in steps of 64. The same in every lane.
__device__ __forceinline__ int find_owner_wave(const int *__restrict__ begin, int n, int item) {
    const int lane = lane_id();
    int lo = 0;
    while (n > 1) {
        const int step = (n + 63) >> 6;
        const bool upto = lane * step < n && begin[lo + lane * step] <= item;
        const int at = (__popcll(__ballot(upto)) - 1) * step;
        lo += at;
        n = min(step, n - at);
    }
    return __builtin_amdgcn_readfirstlane(lo);
}

// Histogram work items of a level, planned from its pairs (hpair_plan) by whoever needs them: every wavefront of the asking
// workgroup does the same few steps, so nothing waits at a barrier and no launch is needed. The steps grow with the
// pairs, for each of the items that grow with them too; levels of more than kUnplannedPairs pairs are planned by one
// launch (k_plan_level) and looked up here.
struct HistPlan {
    int pair = -1;  // the pair that `item` belongs to, -1: there is no such item
    int built = 0, chunk = 0, first_item = 0;
    int item0 = 0;  // first item of the pairs that the launch serves (TreeBuffers::hpair_lo)
    int2 seg = make_int2(0, 0);
};
// publish (wave-uniform): also store the plan of a level that nobody has planned - hpair_begin and ctl[level] -, for
// k_hist_merge and the profile
__device__ __forceinline__ HistPlan plan_hist_item(const TreeBuffers &tb, int n_pairs, int item, bool publish, int level) {
    const int lane = lane_id();
    HistPlan out;  // (the same in every lane: scalar registers)
    if (tb.planned(level)) {
        const LevelCtl ctl = tb.ctl[level];
        if (item >= __builtin_amdgcn_readfirstlane(ctl.n_hitems)) return out;
        out.pair = find_owner_wave(tb.hpair_begin, n_pairs, item);
        const int4 q = tb.hpair_plan[out.pair];
        out.built = __builtin_amdgcn_readfirstlane(q.x);
        out.seg = make_int2(__builtin_amdgcn_readfirstlane(q.y), __builtin_amdgcn_readfirstlane(q.z));
        out.chunk = __builtin_amdgcn_readfirstlane(ctl.hchunk);
        out.first_item = __builtin_amdgcn_readfirstlane(tb.hpair_begin[out.pair]);
        out.item0 = __builtin_amdgcn_readfirstlane(tb.hpair_begin[tb.hpair_lo(level)]);
        return out;
    }
    int4 mine = make_int4(-1, 0, 0, 0);
    if (lane < n_pairs) mine = tb.hpair_plan[lane];
    int total = 0, n_built = 0;
    for (int p0 = 0; p0 < n_pairs; p0 += 64) {
        const int4 q = p0 == 0 ? mine : (p0 + lane < n_pairs ? tb.hpair_plan[p0 + lane] : make_int4(-1, 0, 0, 0));
        total += q.x >= 0 ? q.z - q.y : 0;
        n_built += q.x >= 0 ? 1 : 0;
    }
    total = wave_sum_i(total);
    n_built = wave_sum_i(n_built);
    const int chunk = hist_chunk(tb, total, n_built);
    out.chunk = chunk;
    int carry = 0;
    for (int p0 = 0; p0 < n_pairs; p0 += 64) {
        const int4 q = p0 == 0 ? mine : (p0 + lane < n_pairs ? tb.hpair_plan[p0 + lane] : make_int4(-1, 0, 0, 0));
        const int cnt = q.x >= 0 ? (q.z - q.y + chunk - 1) / chunk : 0;
        const int inc = wave_scan_i(cnt);
        const int ex = carry + inc - cnt;
        const int lo = tb.hpair_lo(level);
        if (lo >= p0 && lo < p0 + 64) out.item0 = read_lane(ex, lo - p0);
        if (publish && p0 + lane < n_pairs) tb.hpair_begin[p0 + lane] = ex;
        const unsigned long long owner = __ballot(item >= ex && item < ex + cnt);
        if (owner != 0ull) {
            const int l = __ffsll((long long)owner) - 1;
            out.pair = p0 + l;
            out.built = read_lane(q.x, l);
            out.seg = make_int2(read_lane(q.y, l), read_lane(q.z, l));
            out.first_item = read_lane(ex, l);
        }
        carry += read_lane(inc, 63);
    }
    if (publish && lane == 0) {
        tb.hpair_begin[n_pairs] = carry;
        tb.ctl[level] = LevelCtl{chunk, carry, 0, total};
    }
    return out;
}

// What a lane's columns of a row (v: two bins of 16 bits or four of 8) add to their bins in LDS: exact products (the scales are
// powers of two), rounded once to the nearest integer, the hessian's in the low h_bits. Its integer is below 2^32, and the
// gradient's below 2^31 where the hessian has 32 bits (item_shift: rows * the largest fit the field), so these are converted
// in 32 bits and lie side by side; only whole-number hessians leave the gradient more. With both through doubles and 64-bit
// shifts the root launch of 10 M x 28 was bound by vector instructions: 150 -> 141 us, which is its bytes at the rate of a copy
// (320 MB read, 320 written, 40 of words).
template <bool BIN16>
__device__ __forceinline__ void add_row(unsigned long long *lds, unsigned v, GHPair p, float scale_g, float scale_h, int h_bits, int o0, int o1,
                                        int o2, int o3) {
    const unsigned hq = (unsigned)rintf(fmaxf(p.h, 0.f) * scale_h);
    unsigned long long add;
    if (h_bits == 32) add = (unsigned long long)(unsigned)(int)rintf(p.g * scale_g) << 32 | hq;
    else add = ((unsigned long long)round_to_ll(p.g * scale_g) << h_bits) + hq;
    if (BIN16) {
        const unsigned b0 = v & 0xffff, b1 = v >> 16;
        if (b0 != kMissingBin16) atomicAdd(lds + o0 + b0, add);
        if (b1 != kMissingBin16) atomicAdd(lds + o1 + b1, add);
    } else {
        const unsigned b0 = v & 0xff, b1 = (v >> 8) & 0xff, b2 = (v >> 16) & 0xff, b3 = v >> 24;
        if (b0 != kMissingBin) atomicAdd(lds + o0 + b0, add);
        if (b1 != kMissingBin) atomicAdd(lds + o1 + b1, add);
        if (b2 != kMissingBin) atomicAdd(lds + o2 + b2, add);
        if (b3 != kMissingBin) atomicAdd(lds + o3 + b3, add);
    }
}

// The value that the last of the LPR lanes of a row holds, in every lane of the row (LPR = 4, 8 or 16 consecutive
// lanes): a DPP broadcast inside the 16-lane row of the wavefront, no trip through the LDS crossbar.
template <int LPR>
__device__ __forceinline__ unsigned last_lane_of_row(unsigned v) {
    if (LPR == 4) return (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0xff, 0xf, 0xf, true);  // quad_perm:[3,3,3,3]
    const unsigned hi = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x15f, 0xf, 0xf, true);  // row_newbcast:15
    if (LPR == 16) return hi;
    const unsigned lo = (unsigned)__builtin_amdgcn_mov_dpp((int)v, 0x157, 0xf, 0xf, true);  // row_newbcast:7
    return (threadIdx.x & 8u) ? hi : lo;
}

// What a wavefront has stored in LDS is there for its other lanes (the accesses of a wavefront stay in order).
__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// What search_pack needs of a lane's four bins, loaded early so that nothing waits for it there.
struct PackMeta {
    unsigned meta[4];  // TreeBuffers::bin_meta: one word per bin instead of the chain bin -> feature -> feature's bin range
    bool ignored[4];
    __device__ __forceinline__ void load(const TreeBuffers &tb, int b_begin, int b_end) {
#pragma unroll
        for (int j = 0; j < 4; ++j) meta[j] = tb.bin_meta[max(0, min(b_begin + lane_id() * 4 + j, b_end - 1))];
#pragma unroll
        for (int j = 0; j < 4; ++j)
            ignored[j] = tb.ignored != nullptr && tb.ignored[tb.cut_fid[max(0, min(b_begin + lane_id() * 4 + j, b_end - 1))]] != 0;
    }
};

// The search of one pack of one node, by one wavefront: s_v holds the pack's bins (kEvalPackBins entries, overwritten). A lane has
// four consecutive bins. The sums below a bin within its feature are differences of plain prefix sums, exact in integers. A
// pack of one feature, the usual one with 255 bins, has them without a detour through LDS, and its missing sum once.
// A wavefront takes 2.1 ns for an instruction that depends on the one before whatever else the CU does, and deep levels keep
// the vector ALUs busy, so the code is short before all: no branches, about 650 instructions instead of the
// 1000 of a segmented scan with them (10 k x 8 0.123 -> 0.119 ms a tree, 500 k x 28 0.254 -> 0.249, 50 k x 700 0.269 -> 0.263).
__device__ __forceinline__ void search_pack(const TreeBuffers &tb, const PackMeta &pm, longlong2 *s_v, int x_in, int pack, bool active,
                                            int b_begin, int b_end, GHPair S, double inv_g, double inv_h, float mcw, float lambda) {
#pragma clang fp contract(off)
    const int lane = lane_id(), nb = b_end - b_begin, at = lane * 4;
    // (read here, all of them: read where one of four is picked below, the record would be looked up by its index, in scratch memory)
    unsigned word[4];
    bool ignored[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        word[j] = pm.meta[j];
        ignored[j] = pm.ignored[j];
    }
    long long exg[4], exh[4];
    long long g = 0, h = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const longlong2 v = s_v[at + j];
        exg[j] = g;
        exh[j] = h;
        g += at + j < nb ? v.x : 0;
        h += at + j < nb ? v.y : 0;
    }
    long long upg = g, uph = h;
    wave_scan_pair(upg, uph);
    const long long allg = read_lane_ll(upg, 63), allh = read_lane_ll(uph, 63);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        exg[j] += upg - g;
        exh[j] += uph - h;
    }
    const float fterm = (S.g * S.g) / (S.h + lambda);
    auto missing = [&](long long tg, long long th) {
        return GHPair{S.g - scaled_float(tg, inv_g), S.h - scaled_float(th, inv_h)};
    };
    GHPair m[4];
    const bool one_feature = read_lane((int)(word[0] & 0xffu), 0) + 1 >= nb;
    if (one_feature) {
        m[0] = missing(allg, allh);
        m[1] = m[2] = m[3] = m[0];
    } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) s_v[at + j] = make_longlong2(exg[j], exh[j]);
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // (past the pack's end the words of its last bin repeat: clamped, nobody looks at the result)
            const int head = max(0, at + j - (int)(word[j] >> 8 & 0xffu)), end = min(at + j + (int)(word[j] & 0xffu) + 1, nb);
            const longlong2 below = s_v[head], upto = s_v[min(end, kEvalPackBins - 1)];
            m[j] = missing((end == nb ? allg : upto.x) - below.x, (end == nb ? allh : upto.y) - below.y);
            exg[j] -= below.x;
            exh[j] -= below.y;
        }
    }
    float score[4], best = -1.f;
    GHPair left[4];
    int which = 0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        left[j] = GHPair{scaled_float(exg[j], inv_g), scaled_float(exh[j], inv_h)};
        const float gr = split_gain_select(S, fterm, left[j], mcw, lambda);
        const float gl = split_gain_select(S, fterm, GHPair{left[j].g + m[j].g, left[j].h + m[j].h}, mcw, lambda);
        score[j] = gl > gr ? gl : -gr;
        score[j] = ignored[j] ? 0.f : score[j];  // column sampling: hist_tree_builder_single.cu:304 / :663
        const float a = at + j < nb ? fabsf(score[j]) : -1.f;
        which = a > best ? j : which;
        best = fmaxf(best, a);
    }
    // wavefront arg-max: larger |score| wins, ties go to the smaller bin index, which is the first lane's: lanes hold ascending
    // bins. The lane that holds the winner writes its candidate itself (without any candidate every lane holds the initial
    // one and the first lane writes the empty record).
    const unsigned long long owners = __ballot(best == wave_max_f(best));
    if (active && lane == __ffsll((long long)owners) - 1) {
        const bool none = best < 0.f;
        unsigned meta = word[0];
        SplitCand c;
        c.score = score[0];
        c.left = left[0];
        c.miss = m[0];
#pragma unroll
        for (int j = 1; j < 4; ++j)
            if (which == j) {
                c.score = score[j];
                c.left = left[j];
                c.miss = m[j];
                meta = word[j];
            }
        c.index = b_begin + at + which;
        c.feature = (int)(meta >> 16);
        c.bin = (int)(meta >> 8 & 0xffu);
        if (none) {
            c.score = 0.f;
            c.index = 0x7fffffff;
            c.miss = c.left = GHPair{0, 0};
            c.feature = c.bin = 0;
        }
        tb.cand[(size_t)x_in * tb.n_packs + pack] = c;
    }
}

}  // namespace
}  // namespace tgbm
