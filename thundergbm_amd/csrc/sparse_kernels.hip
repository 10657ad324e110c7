// Sparse layout, level pass: histogram build and split search of one tree level in a single pass over the
// bin-major copy of the stored values (sorted by global bin id, rows ascending inside a bin).
//
// The reference (hist_tree_builder_single.cu:203-216, :485-505, :257-350, :614-752) keeps one histogram of all
// cut points per node and scans every bin of every node. With 100 000 features that is ~100 MB per node of which a
// deep node touches a few percent. Here a workgroup owns a run of features: it adds the fixed-point gradient pair
// of every stored value to an LDS table cell (bin, node of the value's row), then searches the tables of its
// features for the best candidate of every node (same prefix sums, missing-value term, gain formula and tie rule as
// the dense split search) and hands one candidate per node to k_best_update. Nothing per-node lives in HBM, nothing
// has to be zeroed or subtracted, and a (feature, node) pair without stored values costs one look at its cells.
// Sums are 64-bit integers at the tree's scales: exact, so the candidates are the very numbers a per-node histogram
// would give.
#include <algorithm>
#include <cstdlib>

#include "device_api.h"
#include "kernel_common.h"
#include "rare_bound.h"

namespace tgbm {
namespace {

constexpr int kSpBlock = 1024;
constexpr int kSpWaves = kSpBlock / 64;

struct SegResult {
    float win;     // |score| of the segment's best candidate, -1: none
    int win_idx;   // its global bin index
    float score;   // owner lane only: signed score, missing sums, left sums
    GHPair miss, left;
    bool owner;
};

// Upper estimate of a gain from the hardware reciprocal (1 ulp) instead of divisions; -1: the weight gate closes
__device__ __forceinline__ float gain_estimate(GHPair f, float fterm, GHPair l, float mcw, float lambda) {
    const GHPair r{f.g - l.g, f.h - l.h};
    if (!(l.h >= mcw && r.h >= mcw)) return -1.f;
    const float a = l.g * l.g * __builtin_amdgcn_rcpf(l.h + lambda), b = r.g * r.g * __builtin_amdgcn_rcpf(r.h + lambda);
    return (a + b - fterm) + (a + b + fabsf(fterm)) * 0x1p-18f;  // + 2^-18 of the terms: far above the roundings
}

// Best candidate of one (feature, node) segment; one wavefront, lane l looks at ceil(kf / 64) consecutive bins of the
// feature's kf <= 256 bins. The arithmetic is that of k_eval_split: exact integer prefix sums,
// missing = node sum - feature total, gain with the missing rows sent right and left
// (hist_tree_builder_single.cu:300-323), largest |gain| wins, ties go to the smaller bin index (:330-335).
// `force`: evaluate even when the segment holds no value (the feature owning global bin 0: when no candidate of a
// node has a positive gain the arg-max of the reference ends on bin 0).
// `floor`: the best gain that the node has seen; a segment none of whose candidates reaches it by their estimates has no result.
// A wavefront takes 2.1 ns for an instruction that depends on the one before, so the code has no branches but the ones that
// all lanes take alike. BPL: most bins of a lane. TRY: with the estimates.
template <int BPL, bool TRY>
__device__ __forceinline__ SegResult eval_segment(const longlong2 *cells, int kf, int gbin0, GHPair S, double inv_g, double inv_h,
                                                  float mcw, float lambda, bool ignored, bool force, float floor) {
#pragma clang fp contract(off)
    const int lane = lane_id();
    const int bpl = BPL == 1 ? 1 : (kf + 63) >> 6;  // bins per lane: 1 for the usual <= 64 bins, so that every lane has a candidate
    long long exg[BPL], exh[BPL], rung = 0, runh = 0;
#pragma unroll
    for (int j = 0; j < BPL; ++j) {
        exg[j] = rung;
        exh[j] = runh;
        if (j >= bpl) break;
        const int b = lane * bpl + j;
        const longlong2 v = cells[min(b, kf - 1)];
        rung += b < kf ? v.x : 0;
        runh += b < kf ? v.y : 0;
    }
    long long upg = rung, uph = runh;
    wave_scan_pair(upg, uph);
    const long long totg = read_lane_ll(upg, 63), toth = read_lane_ll(uph, 63);
    SegResult r;
    r.win = -1.f;
    r.win_idx = 0x7fffffff;
    r.owner = false;
    r.score = 0.f;
    r.miss = r.left = GHPair{0, 0};
    if (!force && totg == 0 && toth == 0) return r;
    const long long carryg = upg - rung, carryh = uph - runh;  // exclusive prefix of the lane
    const GHPair m{S.g - scaled_float(totg, inv_g), S.h - scaled_float(toth, inv_h)};
    if (TRY && !force) {
        const float about = S.g * S.g * __builtin_amdgcn_rcpf(S.h + lambda);
        float most = -1.f;
#pragma unroll
        for (int j = 0; j < BPL; ++j) {
            if (j >= bpl) break;
            const GHPair l{scaled_float(carryg + exg[j], inv_g), scaled_float(carryh + exh[j], inv_h)};
            const float e = fmaxf(gain_estimate(S, about, l, mcw, lambda), gain_estimate(S, about, GHPair{l.g + m.g, l.h + m.h}, mcw, lambda));
            most = lane * bpl + j < kf ? fmaxf(most, e) : most;
        }
        if (!__any(most >= floor)) return r;
    }
    const float fterm = (S.g * S.g) / (S.h + lambda);
    float best = -1.f, best_score = 0.f;
    int which = 0;
    GHPair best_left{0, 0};
#pragma unroll
    for (int j = 0; j < BPL; ++j) {
        if (j >= bpl) break;
        const int b = lane * bpl + j;
        const GHPair l{scaled_float(carryg + exg[j], inv_g), scaled_float(carryh + exh[j], inv_h)};
        const float gr = split_gain_select(S, fterm, l, mcw, lambda);
        const float gl = split_gain_select(S, fterm, GHPair{l.g + m.g, l.h + m.h}, mcw, lambda);
        const float score = ignored ? 0.f : (gl > gr ? gl : -gr);  // column sampling: hist_tree_builder_single.cu:304 / :663
        const float a = b < kf ? fabsf(score) : -1.f;
        const bool better = a > best;
        which = better ? j : which;
        best_score = better ? score : best_score;
        best_left.g = better ? l.g : best_left.g;
        best_left.h = better ? l.h : best_left.h;
        best = better ? a : best;
    }
    // (lanes hold ascending bins: among equal gains the first lane's is the smallest)
    const float win = wave_max_f(best);
    const int first = __ffsll((long long)__ballot(best == win)) - 1;
    r.win = win;
    r.win_idx = win < 0.f ? 0x7fffffff : read_lane(gbin0 + lane * bpl + which, first);
    r.owner = lane == first && best >= 0.f;
    r.score = best_score;
    r.miss = m;
    r.left = best_left;
    return r;
}

// key that orders candidates like the reference's arg-max: larger |gain| first, then the smaller bin index
__device__ __forceinline__ unsigned long long cand_key(float abs_gain, int index) {
    return ((unsigned long long)__float_as_uint(abs_gain) << 32) | (unsigned long long)(0xffffffffu - (unsigned)index);
}
__device__ __forceinline__ int key_index(unsigned long long key) { return (int)(0xffffffffu - (unsigned)key); }

constexpr int kSpKept = 256;  // segments of a batch whose results are kept (what the LDS has left beside the largest tables)
struct SpShared {
    float kept[kSpKept][5];  // score, missing and left sums
    GHPair S[kSparseMaxLevelNodes];              // node sums of the level
    unsigned long long key[kSparseMaxLevelNodes];  // best candidate of every node over the task's features so far
    unsigned char ok[kSparseMaxLevelNodes];        // node is valid
    int fbin[kSparseBatchFeatures + 2];            // first bin (relative to the batch) of every feature of the batch
    int ctl[8];  // batch: first feature, end feature, first bin, bins, node range begin, nodes in range, first group, end group
};
// (a launch asks for n_cells <= kSparseCells of LDS beside these)
static_assert(sizeof(SpShared) + kSparseCells * sizeof(longlong2) <= kLdsBytes, "the largest tables' LDS");

// Level-wide state every task starts from: node sums and validity into LDS, and the best keys that other tasks have published:
// a node whose best candidate is another task's by now needs no record of this one's.
__device__ void sp_begin(const TreeBuffers &tb, SpShared &sh, int level) {
    const int nl = 1 << level, off = nl - 1;
    for (int x = threadIdx.x; x < nl; x += kSpBlock) {
        const TreeNode &nd = tb.nodes[off + x];
        sh.S[x] = nd.sum_gh_pair;
        sh.ok[x] = nd.is_valid ? 1 : 0;
        sh.key[x] = __hip_atomic_load(&tb.best_key[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// End of a task: its best key of every node competes with the other tasks' (the record already sits in the task's
// candidate slot, where k_best_update finds it through the winning bin's feature).
__device__ void sp_publish(const TreeBuffers &tb, SpShared &sh, int level) {
    const int nl = 1 << level;
    __syncthreads();
    for (int x = threadIdx.x; x < nl; x += kSpBlock) {
        const unsigned long long k = sh.key[x];
        if (k != 0ull && k > __hip_atomic_load(&tb.best_key[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
            atomicMax(&tb.best_key[x], k);
    }
}

// Split search over the tables of one batch: features [fa, fa + nf) x nodes [n0, n0 + nn) of the level, cells at
// (node - n0) * bins + (bin - bin0): the bins of a (feature, node) segment lie next to each other. Phase 1 raises every node's key; after a barrier the wavefronts whose segment holds
// a node's current best write that candidate's details to the task's slot (a later batch with a better candidate
// overwrites them), kept from phase 1 or, past kSpKept segments, worked out again. `dump`: also store the cells into the level's per-node histograms.
template <int BPL, bool DEEP>
__device__ void sp_search_batch(const TreeBuffers &tb, SpShared &sh, const longlong2 *cells, int level, int fa, int nf,
                                int bin0, int n0, int nn, int cand_slot, float mcw, float lambda, longlong2 *dump) {
    const int w = threadIdx.x >> 6, lane = lane_id();
    const double inv_g = tb.quant->inv_g, inv_h = tb.quant->inv_h;
    const int n_seg = nf * nn;
    const int bins = sh.fbin[nf];
    for (int seg = w; seg < n_seg; seg += kSpWaves) {
        const int fi = seg / nn, x = seg - fi * nn;
        const int node = n0 + x;
        if (!sh.ok[node]) continue;
        const int b0 = sh.fbin[fi], kf = sh.fbin[fi + 1] - b0;
        if (kf <= 0) continue;
        const bool ign = tb.ignored != nullptr && tb.ignored[fa + fi] != 0;
        const SegResult r = eval_segment<BPL, DEEP>(cells + (size_t)x * bins + b0, kf, bin0 + b0, sh.S[node], inv_g, inv_h, mcw, lambda, ign,
                                              bin0 + b0 == 0, __uint_as_float((unsigned)(sh.key[node] >> 32)));
        if (r.win >= 0.f && lane == 0) atomicMax(&sh.key[node], cand_key(r.win, r.win_idx));
        if (DEEP && seg < kSpKept && r.owner) {
            sh.kept[seg][0] = r.score;
            sh.kept[seg][1] = r.miss.g;
            sh.kept[seg][2] = r.miss.h;
            sh.kept[seg][3] = r.left.g;
            sh.kept[seg][4] = r.left.h;
        }
    }
    __syncthreads();
    for (int x = w; x < nn; x += kSpWaves) {
        const int node = n0 + x;
        const unsigned long long key = sh.key[node];
        if (key == 0ull) continue;
        const int idx = key_index(key);
        if (idx < bin0 || idx >= bin0 + bins) continue;  // the node's best comes from an earlier batch
        // the feature of that bin: last feature of the batch whose first bin is <= idx - bin0
        int lo = 0, hi = nf;
        while (hi - lo > 1) {
            const int mid = (lo + hi) >> 1;
            if (sh.fbin[mid] <= idx - bin0) lo = mid; else hi = mid;
        }
        SplitCand c;
        c.index = idx;
        c.feature = c.bin = 0;
        const int seg = lo * nn + x;
        if (DEEP && seg < kSpKept) {
            c.score = sh.kept[seg][0];
            c.miss = GHPair{sh.kept[seg][1], sh.kept[seg][2]};
            c.left = GHPair{sh.kept[seg][3], sh.kept[seg][4]};
            if (lane == 0) tb.cand[(size_t)node * tb.n_packs + cand_slot] = c;
            continue;
        }
        const int b0 = sh.fbin[lo], kf = sh.fbin[lo + 1] - b0;
        const bool ign = tb.ignored != nullptr && tb.ignored[fa + lo] != 0;
        const SegResult r = eval_segment<BPL, DEEP>(cells + (size_t)x * bins + b0, kf, bin0 + b0, sh.S[node], inv_g, inv_h, mcw, lambda, ign, true, 0.f);
        if (r.owner && r.win_idx == idx) {
            c.score = r.score;
            c.miss = r.miss;
            c.left = r.left;
            tb.cand[(size_t)node * tb.n_packs + cand_slot] = c;
        }
    }
    if (dump != nullptr) {
        const int total = bins * nn;
        for (int c = threadIdx.x; c < total; c += kSpBlock) {
            const int x = c / bins, b = c - x * bins;
            dump[(size_t)(n0 + x) * tb.n_bins + bin0 + b] = cells[c];
        }
    }
}

// One task = a run of whole features (batched so that their tables fit the LDS) or one chunk of a big feature (its
// table goes to the partial buffer, k_sparse_big adds the chunks up and searches them).
// Added up in 33 us at levels 0 to 3 for the 15 M values of the frequent features of 1 M x 100 k (7 bytes each: the pair's word, the
// bin, the node), 72 where the nodes are looked up (5 M lines of the L2) and 78 with 8 bytes more a value: waits for loads, the LDS
// is busy for 14 of them, the vector units for 24. At deep levels the search comes on top, 63 us at level 7: issue of its
// instructions with a workgroup on a CU. It took 119 us, with winners' segments searched again for their records, without the
// estimates, and with chunks before the tasks that search.
// DEEP: one workgroup on a CU, for its registers (more than 64 bins) or its table (from level 4 on); else two, without the estimates and
// kept records, for which 64 registers are too few (33 -> 45 us at level 1).
// NODES: kRootNode (level 0): every row is in the one node; the pairs are looked up there and left in table_gh for the levels below (a
// launch of its own before: 130 us and 67 at 1 M rows, together 113), unless k_sparse_spread has (kRootWords). kSpreadNodes: the rows'
// nodes have been brought to the values, too. kRowNodes: they are looked up. WORDS: the rows' gradient words instead of their pairs, half the bytes; the
// pairs that they stand for have the same bits.
enum { kRootNode, kRootWords, kRowNodes, kSpreadNodes };
template <int NODES, bool WORDS, int BPL, bool DEEP>
__global__ __launch_bounds__(kSpBlock, DEEP ? 4 : 8) void k_sparse_level(TreeBuffers tb_all, SparsePass sp, const GHPair *__restrict__ gh,
                                                                            int level, float mcw, float lambda, int dump_hist,
                                                                            int n_cells) {
    extern __shared__ longlong2 cells[];  // [n_cells]
    __shared__ SpShared sh;
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    const SparseTask task = sp.tasks[blockIdx.x];
    const int nl = 1 << level, off = nl - 1;
    const unsigned short *__restrict__ nid16 = tb.nid16;
    const int *__restrict__ crp = tb.cut_row_ptr;
    const float scale_g = tb.quant->scale_g, scale_h = tb.quant->scale_h;
    // (in units of a group of places)
    const size_t set = (size_t)blockIdx.z * (sp.n_table_places / kSpreadGroup);
    const bool copied = sp.table_gh != nullptr;
    const unsigned *__restrict__ nodes =
        reinterpret_cast<const unsigned *>(sp.value_node + (size_t)blockIdx.z * (sp.n_rare_places + sp.n_table_places) + sp.n_rare_places);
    const int task_bin0 = crp[task.f_begin];
    sp_begin(tb, sh, level);
    longlong2 *dump = (dump_hist && task.cand_slot >= 0) ? tb.hist(level) : nullptr;
    longlong2 *partial = task.partial_slot >= 0
                             ? sp.partial + ((size_t)blockIdx.z * sp.n_partial_slots + task.partial_slot) * sp.partial_stride
                             : nullptr;
    int f = task.f_begin;
    while (f < task.f_end) {
        __syncthreads();
        if (threadIdx.x == 0) {
            // next batch: as many whole features as fit with all nodes of the level, or one feature with a node range
            int kf = crp[f + 1] - crp[f];
            int fb = f + 1, nn = nl;
            if ((long)kf * nl <= n_cells) {
                int total = kf;
                while (fb < task.f_end && fb - f < kSparseBatchFeatures) {
                    const int k = crp[fb + 1] - crp[fb];
                    if ((long)(total + k) * nl > n_cells) break;
                    total += k;
                    ++fb;
                }
                kf = total;
            } else {
                nn = n_cells / kf;
            }
            sh.ctl[0] = f;
            sh.ctl[1] = fb;
            sh.ctl[2] = crp[f];
            sh.ctl[3] = kf;
            sh.ctl[5] = nn;
            sh.ctl[6] = max(task.g_begin, sp.table_first[f]);
            sh.ctl[7] = min(task.g_end, sp.table_first[fb]);
        }
        __syncthreads();
        const int fa = sh.ctl[0], fb = sh.ctl[1], bin0 = sh.ctl[2], nbins = sh.ctl[3], nn_max = sh.ctl[5];
        const int g0 = sh.ctl[6], g1 = sh.ctl[7];
        const int nf = fb - fa;
        for (int i = threadIdx.x; i <= nf; i += kSpBlock) sh.fbin[i] = crp[fa + i] - bin0;
        for (int n0 = 0; n0 < nl; n0 += nn_max) {
            const int nn = min(nn_max, nl - n0);
            const int n_cells = nbins * nn;
            __syncthreads();
            for (int c = threadIdx.x; c < n_cells; c += kSpBlock) cells[c] = make_longlong2(0, 0);
            __syncthreads();
            // accumulate: a thread takes two groups of places at a time, one where 64 registers have to do (every load is unconditional -
            // past the end the last group repeats and is skipped below -, so that a stage's loads are issued together instead of one after
            // the other)
            constexpr int U = DEEP ? 2 : 1, V = kSpreadGroup;
            static_assert(V == 4, "a group's loads");
            const int bin_shift = bin0 - task_bin0;
            for (int q0 = g0 + (int)threadIdx.x; q0 < g1; q0 += kSpBlock * U) {
                unsigned long long bin4[U];
                unsigned node4[U];       // (kSpreadNodes)
                int x[U][V];             // (kRowNodes)
                float g[U][V], h[U][V];  // (WORDS: g the word)
                int row[U][V];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const int q = min(q0 + u * kSpBlock, g1 - 1);
                    bin4[u] = __builtin_nontemporal_load(reinterpret_cast<const unsigned long long *>(sp.table_bin) + q);
                    if (NODES == kSpreadNodes) node4[u] = __builtin_nontemporal_load(nodes + q);
                    if ((NODES != kSpreadNodes && NODES != kRootWords) || !copied) {
                        const int4 r4 = reinterpret_cast<const int4 *>(sp.table_row)[q];
                        row[u][0] = r4.x, row[u][1] = r4.y, row[u][2] = r4.z, row[u][3] = r4.w;
                    }
                    if (NODES != kRootNode && copied) {
                        if (WORDS) {
                            const uint4 w4 = reinterpret_cast<const uint4 *>(sp.table_gh)[q];
                            g[u][0] = __uint_as_float(w4.x), g[u][1] = __uint_as_float(w4.y), g[u][2] = __uint_as_float(w4.z), g[u][3] = __uint_as_float(w4.w);
                        } else {
                            const float4 a = reinterpret_cast<const float4 *>(sp.table_gh)[2 * (set + q)], b = reinterpret_cast<const float4 *>(sp.table_gh)[2 * (set + q) + 1];
                            g[u][0] = a.x, h[u][0] = a.y, g[u][1] = a.z, h[u][1] = a.w;
                            g[u][2] = b.x, h[u][2] = b.y, g[u][3] = b.z, h[u][3] = b.w;
                        }
                    }
                }
                if (NODES == kRowNodes) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
#pragma unroll
                        for (int k = 0; k < V; ++k) x[u][k] = (int)nid16[row[u][k]] - off - n0;
                    }
                }
                if (NODES == kRootNode || !copied) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
#pragma unroll
                        for (int k = 0; k < V; ++k) {
                            if (WORDS) {
                                g[u][k] = __uint_as_float(sp.gh_words[row[u][k]]);
                            } else {
                                const GHPair s = gh[row[u][k]];
                                g[u][k] = s.g;
                                h[u][k] = s.h;
                            }
                        }
                    }
                }
                if (NODES == kRootNode && copied) {
#pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const int q = q0 + u * kSpBlock;
                        if (q >= g1) continue;
                        if (WORDS) {
                            reinterpret_cast<float4 *>(sp.table_gh)[q] = make_float4(g[u][0], g[u][1], g[u][2], g[u][3]);
                        } else {
                            reinterpret_cast<float4 *>(sp.table_gh)[2 * (set + q)] = make_float4(g[u][0], h[u][0], g[u][1], h[u][1]);
                            reinterpret_cast<float4 *>(sp.table_gh)[2 * (set + q) + 1] = make_float4(g[u][2], h[u][2], g[u][3], h[u][3]);
                        }
                    }
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
#pragma unroll
                    for (int k = 0; k < V; ++k) {
                        const int bin = (int)(bin4[u] >> 16 * k & 0xffffu), of = (int)(node4[u] >> 8 * k & 0xffu);
                        const int at = NODES == kRootNode || NODES == kRootWords ? 0 : NODES == kRowNodes ? x[u][k] : of == 0xff ? -1 : of - n0;
                        if (q0 + u * kSpBlock < g1 && (unsigned)at < (unsigned)nn && bin != (int)kTableEmpty) {
                            const GHPair p = WORDS ? pair_from_word(sp.gh_objective, __float_as_uint(g[u][k])) : GHPair{g[u][k], h[u][k]};
                            const long long gq = round_to_ll(p.g * scale_g), hq = round_to_ll(p.h * scale_h);
                            unsigned long long *cell = reinterpret_cast<unsigned long long *>(cells + at * nbins + (bin - bin_shift));
                            atomicAdd(cell, (unsigned long long)gq);
                            atomicAdd(cell + 1, (unsigned long long)hq);
                        }
                    }
                }
            }
            __syncthreads();
            if (partial != nullptr) {
                // (node, bin) cells of the whole level, this node range's part
                for (int c = threadIdx.x; c < n_cells; c += kSpBlock) {
                    const int xx = c / nbins, b = c - xx * nbins;
                    partial[(size_t)(n0 + xx) * nbins + b] = cells[c];
                }
            } else {
                sp_search_batch<BPL, DEEP>(tb, sh, cells, level, fa, nf, bin0, n0, nn, task.cand_slot, mcw, lambda, dump);
            }
        }
        f = fb;
    }
    if (partial == nullptr) sp_publish(tb, sh, level);
}

// A big feature: the tables of its chunks are added up (node range by node range) and searched.
template <int BPL>
__global__ __launch_bounds__(kSpBlock) void k_sparse_big(TreeBuffers tb_all, SparsePass sp, int level, float mcw,
                                                        float lambda, int dump_hist, int n_cells) {
    extern __shared__ longlong2 cells[];
    __shared__ SpShared sh;
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const SparseBig big = sp.big[blockIdx.x];
    const int nl = 1 << level;
    const int f = big.feature;
    const int bin0 = tb.cut_row_ptr[f], kf = tb.cut_row_ptr[f + 1] - bin0;
    sp_begin(tb, sh, level);
    if (threadIdx.x == 0) {
        sh.fbin[0] = 0;
        sh.fbin[1] = kf;
    }
    const longlong2 *base = sp.partial + (size_t)blockIdx.z * sp.n_partial_slots * sp.partial_stride;
    longlong2 *dump = dump_hist ? tb.hist(level) : nullptr;
    // the level's nodes are shared out over gridDim.y workgroups (a feature of many chunks would otherwise add up
    // megabytes of tables in one workgroup)
    const int per = (nl + (int)gridDim.y - 1) / (int)gridDim.y;
    const int ny0 = min(nl, (int)blockIdx.y * per), ny1 = min(nl, ny0 + per);
    const int nn_max = (long)kf * per <= n_cells ? per : n_cells / kf;
    for (int n0 = ny0; n0 < ny1; n0 += nn_max) {
        const int nn = min(nn_max, ny1 - n0);
        const int n_cells = kf * nn;
        __syncthreads();
        // (few cells: the chunks are shared out over the threads that are left, whose sums meet in the cells)
        const int parts = max(1, min(kSpBlock / n_cells, (big.slot_end - big.slot_begin) / 4));
        if (parts > 1) {
            for (int c = threadIdx.x; c < n_cells; c += kSpBlock) cells[c] = make_longlong2(0, 0);
            __syncthreads();
        }
        for (int i = threadIdx.x; i < n_cells * parts; i += kSpBlock) {
            const int part = i / n_cells, c = i - part * n_cells;
            long long g = 0, h = 0;
#pragma unroll 8
            for (int slot = big.slot_begin + part; slot < big.slot_end; slot += parts) {
                const longlong2 v = base[(size_t)slot * sp.partial_stride + (size_t)n0 * kf + c];
                g += v.x;
                h += v.y;
            }
            if (parts == 1) {
                cells[c] = make_longlong2(g, h);
            } else {
                atomicAdd(reinterpret_cast<unsigned long long *>(cells + c), (unsigned long long)g);
                atomicAdd(reinterpret_cast<unsigned long long *>(cells + c) + 1, (unsigned long long)h);
            }
        }
        __syncthreads();
        sp_search_batch<BPL, true>(tb, sh, cells, level, f, 1, bin0, n0, nn, big.cand_slot, mcw, lambda, dump);
    }
    sp_publish(tb, sh, level);
}

// ------------------------------------------------------------------------------------ rare features
// Features with few stored values: nearly none of their candidates can win a node (1 M rows x 100 k
// features: fewer than 20 of 23 M a level pass a reciprocal estimate of their gain), so the pass first finds the few
// (feature, node) runs that could and searches only those.
//
// The filter. A candidate of a run splits off a subset A of the run's values - a prefix in the order of their bins when
// the missing rows go right, a suffix when they go left. One word per row holds its node and g and h in ten-bit units of
// the tree's largest. The values of a feature are cut into groups of neighbours in bin order (as many as the cells
// allow: 64 at the root, one where the level has more (feature, node) runs than that), and every (feature, node, group)
// has a cell in LDS that adds up its positive and its negative g, its h and its values. A prefix that ends inside a
// group is the sum of the groups before it and some of that group's values, which bounds A.g from both sides and A.h
// from both sides, hence the gain. A run all of whose bounds stay below the best gain its node has seen so far - the table
// tasks of the level have published theirs - loses whatever its order is. The margins cover the float roundings of the
// missing-value arithmetic, a few ulps of the node's sums. (Bounds without groups or signs leave most runs of the later
// trees, whose best gains are small.)
//
// What is left is collected over the tiles of a group (k_sparse_rare_search), sorted by (feature, node, bin) and searched by one segmented scan:
// candidates exist only where the left sum changes - the feature's first bin (left side empty) and the bin after every bin
// that holds a value; the bins in between repeat the previous candidate's gain and lose the tie on the smaller index - so
// the result is what the scan of a complete (bin, node) table gives.
//
// Where every value looks its row's word up, that is what bounds it: a request for a 128-byte line of the L2 each, 127 us a level for
// 18.8 M values of 1 M rows, 361 for twice the values of 2 M rows, whose words are more than an L2. On many values the rows' nodes
// are therefore brought to them first (k_sparse_spread), and the filter takes 47: 30 of them its vector instructions, 25 the
// LDS. A bound is some 70 instructions: a run's sums alone exclude most runs before their groups are looked at, and at deep levels
// only runs that weigh enough are looked at, gathered from all threads (67 us without both). The tiles of a group are strided over
// the features, whose frequencies often fall with their index.
constexpr int kRareV = kRareTile / kRareBlock;
constexpr int kRareWaves = kRareBlock / 64;
constexpr int kRareCells = 3072;  // (with them two workgroups fit a CU)
constexpr int kRareMaxGroups = 64;
// LDS position of position i: one element of padding after every 32, so that the lanes of a wavefront that each own
// eight consecutive positions do not meet in a bank
constexpr int kRareLds = kRareTile + kRareTile / 32;
__device__ __forceinline__ int rare_phys(int i) { return i + (i >> 5); }

// (the tree's largest as an integer too: rounded, a small one can exceed its product with the scale)
__device__ __forceinline__ unsigned rare_row_word(unsigned node, GHPair s, const QuantCtl &q) {
    return rare_word(node, (float)round_to_ll(s.g * q.scale_g), (float)round_to_ll(s.h * q.scale_h),
                     (float)round_to_ll(q.gq_max), (float)round_to_ll(q.hq_max));
}
static_assert(kRareTile * 1023 < 1 << 22 && kRareTile < 1 << 13, "fields of a cell");

// No part of `part` that weighs the least leaves the rest of its node as much (rare_hopeless says the same of `part` alone).
__device__ __forceinline__ bool rare_too_light(RareCell part, float node_h, RareBound u) {
    const RareCell none{0, 0};
    const RareRange r = rare_range(none, part, u);
    return r.h_max + node_h * 0x1p-21f < u.mcw;
}

// No candidate that splits off all of `whole` and some of the values of `part` reaches the gain `floor`.
__device__ __forceinline__ bool rare_hopeless(RareCell whole, RareCell part, GHPair S, float P, float floor, RareBound u) {
    const RareRange r = rare_range(whole, part, u);
    // (the candidates' sums are differences of floats)
    const float eg = (fabsf(S.g) + fabsf(r.g_max) + fabsf(r.g_min)) * 0x1p-21f, eh = S.h * 0x1p-21f;
    const float h_min = r.h_min - eh, h_max = r.h_max + eh;
    if (h_max < u.mcw || S.h - h_min + eh < u.mcw) return true;  // one of the sides weighs too little
    const float a = fmaxf(fabsf(r.g_max), fabsf(r.g_min)) + eg, b = fmaxf(fabsf(S.g - r.g_max), fabsf(S.g - r.g_min)) + eg;
    const float t = a * a * __builtin_amdgcn_rcpf(fmaxf(u.mcw, h_min) + u.lambda) +
                    b * b * __builtin_amdgcn_rcpf(fmaxf(u.mcw, S.h - h_max) + u.lambda);
    return (t - P) + (t + fabsf(P)) * 0x1p-18f < floor;
}

// The runs of a tile with at least two groups per (feature, node): a thread takes four cells that follow each other, a run
// is a part of a thread's cells or the cells of up to sixteen neighbouring lanes. open(): the run may hold a winner. The groups
// are looked at only where some of the wavefront's runs may win by their sums alone.
template <typename MayWin, typename Open>
__device__ __forceinline__ void rare_check_cells(const unsigned long long *cell_g, const unsigned *cell_h, int cells,
                                                 int log_groups, const MayWin &may_win, const Open &open) {
    constexpr int V = 4;
    const int groups = 1 << log_groups, lanes = groups / V;  // lanes of a run (0: several runs per thread)
#pragma unroll 1
    for (int i0 = (int)threadIdx.x * V; __any(i0 < cells); i0 += kRareBlock * V) {
        RareCell upto[V], carry{0, 0}, run{0, 0};
#pragma unroll
        for (int j = 0; j < V; ++j) {
            const RareCell c = i0 + j < cells ? RareCell{cell_g[i0 + j], cell_h[i0 + j]} : RareCell{0, 0};
            run = (j & (groups - 1)) == 0 ? c : run + c;
            upto[j] = run;
        }
        RareCell total = run;
        if (lanes > 1) {
            for (int d = 1; d < lanes; d <<= 1) {
                const RareCell o{(unsigned long long)shfl_up_ll((long long)total.g, d), (unsigned)__shfl_up((int)total.h, d)};
                if ((lane_id() & (lanes - 1)) >= d) total = total + o;
            }
            carry = total - run;
            const int last = lane_id() | (lanes - 1);
            total.g = (unsigned long long)(unsigned)__shfl((int)(unsigned)total.g, last) |
                      (unsigned long long)(unsigned)__shfl((int)(total.g >> 32), last) << 32;
            total.h = (unsigned)__shfl((int)total.h, last);
        }
        const RareCell none{0, 0};
        bool hope = total.g != 0 && may_win((i0 + V - 1) >> log_groups, none, groups == 2 ? upto[V - 1] : total, none);
        if (groups == 2) hope = hope || (upto[1].g != 0 && may_win(i0 >> log_groups, none, upto[1], none));
        if (!__any(hope)) continue;
#pragma unroll
        for (int j = 0; j < V; ++j) {
            if (groups == 2) total = upto[j | 1];
            const RareCell before = (j & (groups - 1)) == 0 ? carry : carry + upto[j > 0 ? j - 1 : 0];
            const RareCell own = carry + upto[j] - before;
            if (own.g != 0 && may_win((i0 + j) >> log_groups, before, own, total - before - own)) open((i0 + j) >> log_groups);
        }
    }
}

struct RareSum {
    long long g, h;
    int n;
};
__device__ __forceinline__ RareSum operator+(RareSum a, RareSum b) { return {a.g + b.g, a.h + b.h, a.n + b.n}; }

struct RareScan {
    RareSum sum;
    int flag;  // a run starts in one of the lanes summed up
    template <int CTRL, int ROWS>
    __device__ __forceinline__ void at() {
        const RareSum o{dpp_ll<CTRL, ROWS>(sum.g), dpp_ll<CTRL, ROWS>(sum.h), dpp_i<CTRL, ROWS>(0, sum.n)};
        const int of = dpp_i<CTRL, ROWS>(0, flag);
        if (!flag) sum = o + sum;
        flag |= of;
    }
};

// Inclusive segmented scan (thread t owns positions t * V ..): v[j] becomes the sum from the start of its run
// (head = a run starts here) up to j. Two barriers.
template <int V>
__device__ void rare_block_scan(RareSum (&v)[V], const bool (&head)[V], RareSum *s_agg, int *s_flag) {
    const int lane = lane_id(), w = wave_id();
    RareSum run{0, 0, 0};
    bool any = false;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        run = head[j] ? v[j] : run + v[j];
        any = any || head[j];
        v[j] = run;
    }
    RareScan scan{run, any ? 1 : 0};
    wave_scan_steps(scan);
    RareSum carry{dpp_ll<kDppWaveShr1>(scan.sum.g), dpp_ll<kDppWaveShr1>(scan.sum.h), dpp_i<kDppWaveShr1>(0, scan.sum.n)};
    const int cflag = dpp_i<kDppWaveShr1>(0, scan.flag);  // (nothing in lane 0)
    if (lane == 63) {
        s_agg[w] = scan.sum;
        s_flag[w] = scan.flag;
    }
    __syncthreads();
    RareSum before{0, 0, 0};
    for (int u = 0; u < w; ++u) before = s_flag[u] ? s_agg[u] : before + s_agg[u];
    if (!cflag) carry = before + carry;
    bool open = true;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        open = open && !head[j];
        if (open) v[j] = carry + v[j];
    }
    __syncthreads();
}

// split_gain with the node's own term (f.g^2 / (f.h + lambda), the same for every candidate of the node) taken from
// a table: the same operations in the same order, hence the same bits
__device__ __forceinline__ float rare_gain(GHPair f, float fterm, GHPair l, float mcw, float lambda) {
#pragma clang fp contract(off)
    const GHPair r{f.g - l.g, f.h - l.h};
    float gain = 0.f;
    if (l.h >= mcw && r.h >= mcw) gain = (l.g * l.g) / (l.h + lambda) + (r.g * r.g) / (r.h + lambda) - fterm;
    return fmaxf(0.f, gain);
}

// Signed score of a candidate (> 0: missing values go left), hist_tree_builder_single.cu:300-323. `floor`: the
// largest |score| the candidate's node has seen so far; a candidate whose estimate stays below it cannot become the
// node's best and is not evaluated (0 = no candidate).
__device__ __forceinline__ float rare_score(GHPair S, float fterm, GHPair m, GHPair l, float mcw, float lambda, float floor) {
#pragma clang fp contract(off)
    const GHPair l2{l.g + m.g, l.h + m.h};
    const float er = gain_estimate(S, fterm, l, mcw, lambda), el = gain_estimate(S, fterm, l2, mcw, lambda);
    if (fmaxf(er, el) < floor) return 0.f;
    const float gr = rare_gain(S, fterm, l, mcw, lambda);
    const float gl = rare_gain(S, fterm, l2, mcw, lambda);
    return (gl > gr) ? gl : -gr;
}

// A value that passed the filter: tile of the group (4 bits), feature in the tile (11), node (10), bin (8), row (31)
__device__ __forceinline__ unsigned long long rare_item(int tile, unsigned key, unsigned node, int row) {
    const unsigned long long feature = (unsigned)tile << 11 | key >> kRareFeatShift;
    return ((feature << 10 | node) << 8 | (key & 0xffu)) << 31 | (unsigned)row;
}
__device__ __forceinline__ unsigned rare_run(unsigned long long item) { return (unsigned)(item >> 39); }  // feature and node
__device__ __forceinline__ int rare_node(unsigned long long item) { return (int)(item >> 39) & 0x3ff; }
__device__ __forceinline__ int rare_bin(unsigned long long item) { return (int)(item >> 31) & 0xff; }

struct RareFilter {
    unsigned long long g[kRareCells];
    unsigned h[kRareCells];
    unsigned long long open[kRareCells / 64];  // runs of the tile that may hold a winner
    unsigned short look[kRareBlock];           // runs of one group that weigh enough
    int looks, any, passed;
};
struct RareShared {
    unsigned long long item[kRareLds];
    GHPair gh[kRareLds];
    RareSum agg[kRareWaves];
    int flag[kRareWaves];
    int meta[kRareGroupTiles];  // first entry of the tiles' features in rare_meta
};

// Sorts the n <= kRareTile collected items. A compare-exchange over at most 64 positions stays inside the 128 items
// that a wavefront owns, so only the wider ones need a barrier.
__device__ void rare_sort(unsigned long long *item, int n) {
    int size = 128;
    while (size < n) size *= 2;
    for (int i = n + threadIdx.x; i < size; i += kRareBlock) item[rare_phys(i)] = ~0ull;
    __syncthreads();
    for (int k = 2; k <= size; k *= 2) {
        for (int j = k / 2; j > 0; j /= 2) {
            for (int i = threadIdx.x; i < size / 2; i += kRareBlock) {
                const int a = ((i & ~(j - 1)) << 1) | (i & (j - 1));
                const int pa = rare_phys(a), pb = rare_phys(a | j);
                const unsigned long long x = item[pa], y = item[pb];
                if ((x > y) == ((a & k) == 0)) {
                    item[pa] = y;
                    item[pb] = x;
                }
            }
            if (j > 64 || (j == 1 && k >= 128)) __syncthreads();
            else __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
    }
}

// What the search needs of a node: per node of the level its best key (8 bytes), its sums (8) and its own gain term (4).
struct RareNodes {
    unsigned long long *best;
    GHPair *S;
    float *P;
    __device__ RareNodes(unsigned char *lds, int nl)
        : best(reinterpret_cast<unsigned long long *>(lds)), S(reinterpret_cast<GHPair *>(best + nl)),
          P(reinterpret_cast<float *>(S + nl)) {}
    __device__ void load(const TreeBuffers &tb, int nl, float lambda) {
#pragma clang fp contract(off)
        for (int x = threadIdx.x; x < nl; x += kRareBlock) {
            const GHPair s = tb.nodes[nl - 1 + x].sum_gh_pair;
            best[x] = __hip_atomic_load(&tb.best_key[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            S[x] = s;
            P[x] = (s.g * s.g) / (s.h + lambda);
        }
    }
    __device__ float floor(int x) const { return __uint_as_float((unsigned)(best[x] >> 32)); }
};

// Searches the n <= V * kRareBlock collected values, V consecutive ones per thread, and clears the way for the next ones.
template <int V>
__device__ void rare_search(const TreeBuffers &tb, const SparsePass &sp, RareShared &sh, const RareNodes &node,
                            const GHPair *__restrict__ gh, int n, int slot, float mcw, float lambda) {
#pragma clang fp contract(off)
    rare_sort(sh.item, n);
    for (int p = threadIdx.x; p < n; p += kRareBlock)
        sh.gh[rare_phys(p)] = gh[(int)((unsigned)sh.item[rare_phys(p)] & 0x7fffffffu)];
    __syncthreads();
    const float scale_g = tb.quant->scale_g, scale_h = tb.quant->scale_h;
    const double inv_g = tb.quant->inv_g, inv_h = tb.quant->inv_h;
    const int i0 = threadIdx.x * V;
    static_assert(32 % V == 0, "a thread's positions must not straddle a padding element");
    const int pb = rare_phys(i0);  // rare_phys(i0 + j) = pb + j: a thread's positions share one padding count
    unsigned long long it[V];
    RareSum fs[V];
    bool head[V], tail[V], last_of_bin[V];
    const unsigned long long before = (i0 > 0 && i0 - 1 < n) ? sh.item[rare_phys(i0 - 1)] : ~0ull;
    const unsigned long long after = i0 + V < n ? sh.item[rare_phys(i0 + V)] : ~0ull;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const bool in = i0 + j < n;
        it[j] = in ? sh.item[pb + j] : ~0ull;
        fs[j] = RareSum{0, 0, 0};
        if (in) {
            const GHPair s = sh.gh[pb + j];
            fs[j] = RareSum{round_to_ll(s.g * scale_g), round_to_ll(s.h * scale_h), 1};
        }
    }
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const int p = i0 + j;
        const bool in = p < n;
        const unsigned long long prev = j == 0 ? before : it[j > 0 ? j - 1 : 0];
        const unsigned long long next = j == V - 1 ? after : it[j < V - 1 ? j + 1 : 0];
        head[j] = in && (p == 0 || rare_run(prev) != rare_run(it[j]));
        tail[j] = in && (p + 1 == n || rare_run(next) != rare_run(it[j]));
        last_of_bin[j] = in && (p + 1 == n || (next >> 31) != (it[j] >> 31));
    }
    // (the scan's barriers: every thread has read its pairs, their place takes the run totals)
    rare_block_scan(fs, head, sh.agg, sh.flag);
    // the last value of a run holds the run's sums = the feature's total in the node: as floats to the run's start
    GHPair left[V];
    int start[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        left[j] = GHPair{(float)((double)fs[j].g * inv_g), (float)((double)fs[j].h * inv_h)};
        start[j] = rare_phys(max(0, i0 + j - fs[j].n + 1));
        if (tail[j]) sh.gh[start[j]] = left[j];
    }
    __syncthreads();
    // candidates raise the node's key in LDS, then the winners publish. A candidate without gain never competes: the
    // node's candidate at global bin 0 (a table feature's) has at least its key.
    float sc_head[V], sc_bin[V];
#pragma unroll
    for (int j = 0; j < V; ++j) {
        sc_head[j] = sc_bin[j] = 0.f;
        if (!(head[j] || last_of_bin[j])) continue;
        const unsigned long long item = sh.item[pb + j];
        const int x = rare_node(item), lb = rare_bin(item);
        const int2 meta = sp.rare_meta[sh.meta[(int)(item >> 60)] + ((int)(item >> 49) & 0x7ff)];
        const GHPair tot = sh.gh[start[j]];
        const GHPair S = node.S[x];
        const float P = node.P[x];
        const GHPair mm{S.g - tot.g, S.h - tot.h};
        const float floor = node.floor(x);
        if (head[j]) {
            sc_head[j] = rare_score(S, P, mm, GHPair{0, 0}, mcw, lambda, floor);
            if (sc_head[j] != 0.f) atomicMax(&node.best[x], cand_key(fabsf(sc_head[j]), meta.x));
        }
        if (last_of_bin[j] && lb < meta.y - 1) {
            sc_bin[j] = rare_score(S, P, mm, left[j], mcw, lambda, floor);
            if (sc_bin[j] != 0.f) atomicMax(&node.best[x], cand_key(fabsf(sc_bin[j]), meta.x + lb + 1));
        }
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < V; ++j) {
        if (sc_head[j] == 0.f && sc_bin[j] == 0.f) continue;
        const unsigned long long item = sh.item[pb + j];
        const int x = rare_node(item), lb = rare_bin(item);
        const int fbegin = sp.rare_meta[sh.meta[(int)(item >> 60)] + ((int)(item >> 49) & 0x7ff)].x;
        const unsigned long long best = node.best[x];
        const bool win_head = sc_head[j] != 0.f && best == cand_key(fabsf(sc_head[j]), fbegin);
        const bool win_bin = sc_bin[j] != 0.f && best == cand_key(fabsf(sc_bin[j]), fbegin + lb + 1);
        if (!(win_head || win_bin)) continue;
        // the group's best of the node: worth publishing only if it beats what other groups have published so far
        if (best <= __hip_atomic_load(&tb.best_key[x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) continue;
        const GHPair S = node.S[x], tot = sh.gh[start[j]];
        SplitCand o;
        o.miss = GHPair{S.g - tot.g, S.h - tot.h};
        o.feature = o.bin = 0;
        if (win_head) {
            o.score = sc_head[j];
            o.index = fbegin;
            o.left = GHPair{0, 0};  // the first bin records an empty left side (hist_tree_builder_single.cu:378)
        } else {
            o.score = sc_bin[j];
            o.index = fbegin + lb + 1;
            o.left = left[j];
        }
        tb.cand[(size_t)x * tb.n_packs + slot] = o;
        atomicMax(&tb.best_key[x], best);
    }
    __syncthreads();
}

// Brings what the rows of the values hold to the values' places: a row block's part in LDS, looked up there. Fetched by
// the filter itself a look-up is a request for a whole line of the L2, whatever it takes of it.
// kBringCodes: the rows' words, with the value's feature in the node's place, to the rare values, once per tree; kBringPairs: the rows'
// gradient words to the table values, once per tree; kBringNodes: the rows' nodes of a level to all of them. Bound by its traffic: 4
// bytes a node (2 the row in its block, 1 the place, 1 the node), 36 M values in 33.5 us, 4.3 TB/s (37 with the groups of a step
// fetched when it begins). Blocks of 32 768 rows: their words still fit the LDS, and a tile of
// 4096 values has some 130 of a block next to each other at 1 M rows.
enum { kBringCodes, kBringPairs, kBringNodes };
template <int WHAT>
__global__ __launch_bounds__(1024) void k_sparse_spread(TreeBuffers tb_all, SparsePass sp, int level) {
    extern __shared__ unsigned spread_dyn[];  // [kSpreadRows] words, or as many bytes
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int r0 = (int)blockIdx.y << kSpreadLogRows, rows = min(kSpreadRows, tb.n - r0);
    const unsigned *__restrict__ begin = sp.spread_begin + (size_t)blockIdx.y * sp.n_lists;
    const unsigned g0 = begin[WHAT == kBringPairs ? sp.n_rare_tasks : 0], g1 = begin[WHAT == kBringCodes ? sp.n_rare_tasks : sp.n_lists];
    const unsigned per = (g1 - g0 + gridDim.x - 1) / gridDim.x;
    const unsigned first = g0 + blockIdx.x * per, end = min(g1, first + per);
    if (first >= end) return;
    constexpr int U = WHAT == kBringNodes ? 4 : 2;
    // (the groups of the next step are on their way while this one's are looked up; past the end the last group once more, with the
    // same result)
    uint2 next_row[U];
    unsigned next_place[U];
    const auto fetch = [&](unsigned i) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned g = min(i + u * 1024, end - 1);
            next_row[u] = reinterpret_cast<const uint2 *>(sp.spread_row)[g];
            next_place[u] = sp.spread_place[g];
        }
    };
    fetch(first + threadIdx.x);
    if (WHAT == kBringNodes) {
        const unsigned off = (1u << level) - 1u;
        const unsigned *__restrict__ pairs = reinterpret_cast<const unsigned *>(tb.nid16 + r0);
        unsigned short *out = reinterpret_cast<unsigned short *>(spread_dyn);
        const int n_pairs = (rows + 1) / 2;
        constexpr int L = kSpreadRows / 2 / 1024;
        unsigned v[L];
#pragma unroll
        for (int l = 0; l < L; ++l) v[l] = pairs[min(l * 1024 + (int)threadIdx.x, n_pairs - 1)];
#pragma unroll
        for (int l = 0; l < L; ++l) {
            const unsigned a = v[l] & 0xffffu, b = v[l] >> 16;
            out[l * 1024 + threadIdx.x] = (unsigned short)((a >= off ? a - off : 0xffu) | (b >= off ? (b - off) & 0xffu : 0xffu) << 8);
        }
    } else {
        const unsigned *__restrict__ words = WHAT == kBringCodes ? tb.row_word : sp.gh_words;
#pragma unroll 8
        for (int r = threadIdx.x; r < rows; r += 1024) spread_dyn[r] = WHAT == kBringCodes ? words[r0 + r] & ~kRareNodeMask : words[r0 + r];
    }
    __syncthreads();
    for (unsigned i = first + threadIdx.x; i < end; i += 1024 * U) {
        uint2 row[U];
        unsigned place[U];
#pragma unroll
        for (int u = 0; u < U; ++u) row[u] = next_row[u], place[u] = next_place[u];
        fetch(i + 1024 * U);
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const unsigned a = row[u].x & 0xffffu, b = row[u].x >> 16, c = row[u].y & 0xffffu, d = row[u].y >> 16;
            if (WHAT == kBringCodes) {
                const uint4 key = reinterpret_cast<const uint4 *>(sp.rare_key)[place[u]];
                const auto code = [&](unsigned r, unsigned k) { return k == kRareEmpty ? kRareEmpty : spread_dyn[r] | k >> kRareFeatShift; };
                reinterpret_cast<uint4 *>(sp.rare_code + (size_t)blockIdx.z * sp.n_rare_places)[place[u]] =
                    make_uint4(code(a, key.x), code(b, key.y), code(c, key.z), code(d, key.w));
            } else if (WHAT == kBringPairs) {
                reinterpret_cast<uint4 *>(sp.table_gh)[place[u] - (unsigned)(sp.n_rare_places / kSpreadGroup)] =
                    make_uint4(spread_dyn[a], spread_dyn[b], spread_dyn[c], spread_dyn[d]);
            } else {
                const uint8_t *nodes = reinterpret_cast<const uint8_t *>(spread_dyn);
                reinterpret_cast<unsigned *>(sp.value_node + (size_t)blockIdx.z * (sp.n_rare_places + sp.n_table_places))[place[u]] =
                    (unsigned)nodes[a] | (unsigned)nodes[b] << 8 | (unsigned)nodes[c] << 16 | (unsigned)nodes[d] << 24;
            }
        }
    }
}

// One workgroup per tile: the values of the runs that may hold a winner go to the tile's part of rare_item.
// SPREAD: the rows' words and nodes have been brought to the values (k_sparse_spread), which stream in groups of four places.
template <bool DUMP, bool SPREAD>
__global__ __launch_bounds__(kRareBlock, 8) void k_sparse_rare_filter(TreeBuffers tb_all, SparsePass sp,
                                                                     const GHPair *__restrict__ gh, int level, float mcw,
                                                                     float lambda) {
    extern __shared__ __attribute__((aligned(16))) unsigned char rare_dyn[];
    __shared__ RareFilter sh;
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    const int nl = 1 << level;
    const RareTask task = sp.rare_tasks[blockIdx.x];
    const int places = sp.rare_places[blockIdx.x];
    const unsigned *__restrict__ keys = sp.rare_key + task.v_begin;
    const int *__restrict__ rows = sp.rare_row + task.v_begin;
    const unsigned *__restrict__ words = tb.row_word;
    // k-th place of a thread
    const auto place = [&](int k) {
        return SPREAD ? ((k / kSpreadGroup) * kRareBlock + (int)threadIdx.x) * kSpreadGroup + k % kSpreadGroup : k * kRareBlock + (int)threadIdx.x;
    };
    // word: of the row, in place of its node the value's feature (below); node: of the level; group: sixty-fourth of the
    // feature's values. (Places past the end repeat the last ones, so that all loads are issued at once.)
    unsigned word[kRareV], node_of[kRareV], group_of[kRareV];
    if (SPREAD) {
        static_assert(kRareV % kSpreadGroup == 0 && kSpreadGroup == 4, "a thread's places are whole groups");
        const size_t first = (size_t)blockIdx.z * sp.n_rare_places + task.v_begin;
        const size_t first_node = (size_t)blockIdx.z * (sp.n_rare_places + sp.n_table_places) + task.v_begin;
        const uint4 *__restrict__ codes = reinterpret_cast<const uint4 *>(sp.rare_code + first);
        const unsigned *__restrict__ nodes = reinterpret_cast<const unsigned *>(sp.value_node + first_node);
        const unsigned *__restrict__ groups = reinterpret_cast<const unsigned *>(sp.rare_group + task.v_begin);
        uint4 c[kRareV / 4];
        unsigned x[kRareV / 4], g[kRareV / 4];
#pragma unroll
        for (int j = 0; j < kRareV / 4; ++j) {
            const int q = min(j * kRareBlock + (int)threadIdx.x, places / kSpreadGroup - 1);
            c[j] = codes[q];
            x[j] = level > 0 ? nodes[q] : 0u;
            g[j] = groups[q];
        }
#pragma unroll
        for (int k = 0; k < kRareV; ++k) {
            word[k] = k % 4 == 0 ? c[k / 4].x : k % 4 == 1 ? c[k / 4].y : k % 4 == 2 ? c[k / 4].z : c[k / 4].w;
            node_of[k] = x[k / 4] >> 8 * (k % 4) & 0xffu;
            group_of[k] = g[k / 4] >> 8 * (k % 4) & 0xffu;
            if (word[k] == kRareEmpty || node_of[k] == 0xffu) node_of[k] = kRareNodeMask;
        }
    } else {
        unsigned key[kRareV];
        int row[kRareV];
#pragma unroll
        for (int k = 0; k < kRareV; ++k) {
            const int q = min(place(k), places - 1);
            // (streamed past the caches: the words stay in the L2s)
            row[k] = __builtin_nontemporal_load(rows + q);
            key[k] = __builtin_nontemporal_load(keys + q);
        }
#pragma unroll
        for (int k = 0; k < kRareV; ++k) word[k] = words[row[k]];
#pragma unroll
        for (int k = 0; k < kRareV; ++k) {
            node_of[k] = key[k] == kRareEmpty ? kRareNodeMask : word[k] & kRareNodeMask;
            group_of[k] = key[k] >> 8 & 0x3fu;
            word[k] = (word[k] & ~kRareNodeMask) | key[k] >> kRareFeatShift;
        }
    }
    int log_groups = 0;
    while (2 << log_groups <= kRareMaxGroups && task.n_feat * nl << (log_groups + 1) <= kRareCells) ++log_groups;
    const bool folded = task.n_feat * nl > kRareCells;  // (more runs than cells: two runs that meet in one only loosen the bound)
    const int cells = folded ? kRareCells : task.n_feat * nl << log_groups;
    for (int c = threadIdx.x; c < cells; c += kRareBlock) {
        sh.g[c] = 0ull;
        sh.h[c] = 0u;
    }
    if (threadIdx.x < kRareCells / 64) sh.open[threadIdx.x] = 0ull;
    if (threadIdx.x == 0) sh.looks = sh.any = sh.passed = 0;
    RareNodes node(rare_dyn, nl);
    node.load(tb, nl, lambda);
    const RareBound unit{(float)round_to_ll(tb.quant->gq_max) * tb.quant->inv_g / kRareSteps,
                         (float)round_to_ll(tb.quant->hq_max) * tb.quant->inv_h / kRareSteps, mcw, lambda};
    __syncthreads();
    int cell[kRareV];  // -1: the value takes no part
#pragma unroll
    for (int k = 0; k < kRareV; ++k) {
        const unsigned x = node_of[k];
        const int feature = (int)(word[k] & kRareNodeMask);
        const bool on = place(k) < places && x != kRareNodeMask;
        unsigned at = (unsigned)feature << (level + log_groups) | x << log_groups | group_of[k] >> (6 - log_groups);
        if (folded) at %= (unsigned)kRareCells;
        cell[k] = on ? (int)at : -1;
        if (tb.ignored != nullptr && on && tb.ignored[sp.rare_fid[task.meta_begin + feature]] != 0)
            cell[k] = -1;  // column sampling: all scores are 0 (hist_tree_builder_single.cu:304 / :663)
        if (cell[k] >= 0) {
            atomicAdd(&sh.g[cell[k]], rare_addend(word[k]));
            atomicAdd(&sh.h[cell[k]], word[k] >> 22);
        }
        if (DUMP && on) {
            // stage-wise inspection: the per-node histograms of the level (zeroed before the launch) get the values
            const GHPair s = gh[rows[place(k)]];
            const size_t b = (size_t)x * tb.n_bins + sp.rare_meta[task.meta_begin + feature].x + (keys[place(k)] & 0xffu);
            unsigned long long *out = reinterpret_cast<unsigned long long *>(tb.hist(level) + b);
            atomicAdd(out, (unsigned long long)round_to_ll(s.g * tb.quant->scale_g));
            atomicAdd(out + 1, (unsigned long long)round_to_ll(s.h * tb.quant->scale_h));
        }
    }
    __syncthreads();
    const auto hopeless = [&](int x, RareCell whole, RareCell part) {
        return rare_hopeless(whole, part, node.S[x], node.P[x], node.floor(x), unit);
    };
    const auto open = [&](int run) {
        atomicOr(reinterpret_cast<unsigned *>(sh.open) + (run >> 5), 1u << (run & 31));
        sh.any = 1;
    };
    const auto look_at = [&](int c) {
        if (!hopeless(c & (nl - 1), RareCell{0, 0}, RareCell{sh.g[c], sh.h[c]})) open(c);
    };
    if (log_groups > 0) {
        rare_check_cells(
            sh.g, sh.h, cells, log_groups,
            [&](int run, RareCell before, RareCell own, RareCell after) {
                const int x = run & (nl - 1);
                return !hopeless(x, before, own) || !hopeless(x, after, own);
            },
            open);
    } else {
        // A bound takes some 70 instructions and few runs of deep levels weigh enough to split off: those are listed first, one for
        // every thread (with four workgroups on a CU there is no room for more; what does not fit is looked at at once).
        static_assert(kRareCells % kSparseMaxLevelNodes == 0 && kRareCells % kRareBlock == 0, "a cell's node");
#pragma unroll
        for (int i = 0; i < kRareCells / kRareBlock; ++i) {
            const int c = i * kRareBlock + (int)threadIdx.x;
            bool look = c < cells;
            if (look) {
                const RareCell cell{sh.g[c], sh.h[c]};
                look = cell.g != 0 && !rare_too_light(cell, node.S[c & (nl - 1)].h, unit);
            }
            const unsigned long long who = __ballot(look);
            if (who == 0) continue;
            int at = lane_id() == 0 ? atomicAdd(&sh.looks, __popcll(who)) : 0;
            at = read_lane(at, 0) + lanes_below(who);
            if (!look) continue;
            if (at < kRareBlock) sh.look[at] = (unsigned short)c;
            else look_at(c);
        }
        __syncthreads();
        if ((int)threadIdx.x < sh.looks) look_at(sh.look[threadIdx.x]);
    }
    __syncthreads();
    if (sh.any == 0) {  // (the tile's, after the barrier)
        if (threadIdx.x == 0) sp.rare_passed[(size_t)blockIdx.z * sp.n_rare_tasks + blockIdx.x] = 0;
        return;
    }
    unsigned pass = 0;
#pragma unroll
    for (int k = 0; k < kRareV; ++k) {
        if (cell[k] < 0) continue;
        const int run = cell[k] >> log_groups;
        if (reinterpret_cast<const unsigned *>(sh.open)[run >> 5] >> (run & 31) & 1u) pass |= 1u << k;
    }
    if (__any(pass != 0)) {
        // (few values pass: they are read again)
        int at = pass != 0 ? atomicAdd(&sh.passed, __popc(pass)) : 0;
        unsigned long long *out = sp.rare_item + (size_t)blockIdx.z * sp.n_rare_places + task.v_begin;
        const uint8_t *__restrict__ nodes =
            SPREAD ? sp.value_node + (size_t)blockIdx.z * (sp.n_rare_places + sp.n_table_places) + task.v_begin : nullptr;
        for (unsigned left = pass; left != 0; left &= left - 1) {
            const int q = place(__ffs(left) - 1);
            const unsigned x = !SPREAD ? words[rows[q]] & kRareNodeMask : level > 0 ? (unsigned)nodes[q] : 0u;
            out[at++] = rare_item((int)(blockIdx.x / (unsigned)sp.n_rare_groups), keys[q], x, rows[q]);
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) sp.rare_passed[(size_t)blockIdx.z * sp.n_rare_tasks + blockIdx.x] = sh.passed;
}

// One workgroup = the tiles blockIdx.x, blockIdx.x + gridDim.x, ... (at most kRareGroupTiles).
__global__ __launch_bounds__(kRareBlock, 4) void k_sparse_rare_search(TreeBuffers tb_all, SparsePass sp,
                                                                     const GHPair *__restrict__ gh, int level, float mcw,
                                                                     float lambda) {
    extern __shared__ __attribute__((aligned(16))) unsigned char rare_dyn[];
    __shared__ RareShared sh;
    __shared__ int s_passed[kRareGroupTiles];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    if (threadIdx.x < kRareGroupTiles) {
        const int tile = (int)blockIdx.x + (int)threadIdx.x * (int)gridDim.x;
        const bool in = tile < sp.n_rare_tasks;
        s_passed[threadIdx.x] = in ? sp.rare_passed[(size_t)blockIdx.z * sp.n_rare_tasks + tile] : 0;
        sh.meta[threadIdx.x] = in ? sp.rare_tasks[tile].meta_begin : 0;
    }
    __syncthreads();
    int all = 0;
    for (int j = 0; j < kRareGroupTiles; ++j) all += s_passed[j];
    if (all == 0) return;
    RareNodes node(rare_dyn, 1 << level);
    node.load(tb, 1 << level, lambda);
    const int slot = sp.rare_slot + (int)blockIdx.x;
    int filled = 0;
    for (int j = 0; j <= kRareGroupTiles; ++j) {
        const int passed = j < kRareGroupTiles ? s_passed[j] : 0;
        if (filled > 0 && (j == kRareGroupTiles || filled + passed > kRareTile)) {
            // (a value per thread instead of eight: a shorter chain, 22 -> 17 us on 512 values)
            if (filled <= kRareBlock) rare_search<1>(tb, sp, sh, node, gh, filled, slot, mcw, lambda);
            else rare_search<kRareV>(tb, sp, sh, node, gh, filled, slot, mcw, lambda);
            filled = 0;
        }
        if (passed == 0) continue;
        const unsigned long long *__restrict__ in =
            sp.rare_item + (size_t)blockIdx.z * sp.n_rare_places + sp.rare_tasks[(int)blockIdx.x + j * (int)gridDim.x].v_begin;
        for (int q = threadIdx.x; q < passed; q += kRareBlock) sh.item[rare_phys(filled + q)] = in[q];
        filled += passed;
        __syncthreads();
    }
}

// Row -> node update of a level (update_ins2node_id, hist_tree_builder_single.cu:908-1020): a row whose node was
// split moves to the left or right child by the reference's rule (binary search of the row's ascending bin ids for
// one inside the split feature's range; none = missing -> default direction). Rows per child are counted on the way.
// Bound by its chain of loads: the nodes' splits are looked up once per workgroup, then a row takes two steps - its node, its
// byte of the split feature's column -, four rows of a thread at a time. At levels of few nodes the lanes count in copies of the
// counters (all lanes of a wavefront on two counters are taken one by one). 1 M rows: 17.5 -> 10.4 us at level 0, 33 -> 17.4 at level 7.
constexpr int kMoveRows = 4;
__global__ __launch_bounds__(kSpBlock) void k_sparse_partition(TreeBuffers tb_all, CsrBins bins, int level) {
    constexpr int kCounters = 2 * kSparseMaxLevelNodes;
    enum { STAYS = -2, SEARCH = -1 };
    __shared__ int cnt[kCounters];
    __shared__ int s_col[kSparseMaxLevelNodes];    // column of the split feature, SEARCH: it has none, STAYS: no split
    __shared__ int s_split[kSparseMaxLevelNodes];  // split bin * 2 + default direction
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int nl = 1 << level, off = nl - 1, log_copies = min(6, 31 - __clz(kCounters >> (level + 1)));
    const int copy = lane_id() & ((1 << log_copies) - 1);
    for (int i = threadIdx.x; i < 2 * nl << log_copies; i += kSpBlock) cnt[i] = 0;
    for (int x = threadIdx.x; x < nl; x += kSpBlock) {
        const TreeNode &nd = tb.nodes[off + x];
        const bool splits = node_splits(nd);
        s_col[x] = !splits ? (int)STAYS : bins.col_of_feature != nullptr ? max((int)SEARCH, bins.col_of_feature[nd.split_feature_id]) : (int)SEARCH;
        s_split[x] = splits ? (int)nd.split_bid * 2 + (nd.default_right ? 1 : 0) : 0;
    }
    __syncthreads();
    for (int base = blockIdx.x * (kSpBlock * kMoveRows); base < tb.n; base += gridDim.x * (kSpBlock * kMoveRows)) {
        int node[kMoveRows], col[kMoveRows], bin[kMoveRows];
        unsigned word[kMoveRows];
#pragma unroll
        for (int k = 0; k < kMoveRows; ++k) {
            const int r = min(base + k * kSpBlock + (int)threadIdx.x, tb.n - 1);
            node[k] = tb.nid16[r];
            word[k] = tb.row_word != nullptr ? tb.row_word[r] : 0u;
        }
#pragma unroll
        for (int k = 0; k < kMoveRows; ++k) {
            const int r = base + k * kSpBlock + (int)threadIdx.x;
            // (a row past the end stays: the last row's node, which was loaded in its place, is a child's by now if the thread that
            // has that row was faster. Other rows stay in leaves of earlier levels.)
            col[k] = r < tb.n && node[k] >= off ? s_col[node[k] - off] : (int)STAYS;
            bin[k] = col[k] >= 0 ? (int)bins.colbin[(size_t)col[k] * bins.col_stride + r] : 0;
        }
#pragma unroll
        for (int k = 0; k < kMoveRows; ++k) {
            const int r = base + k * kSpBlock + (int)threadIdx.x;
            if (r >= tb.n) continue;
            int child = (int)kRareNodeMask;  // of the next level; all ones: the row stays
            if (col[k] != STAYS) {
                const int x = node[k] - off, split = s_split[x];
                // a frequent feature: the row's local bin id is one byte away (same rule: missing -> default
                // direction, else right iff the bin is not below the split bin)
                bool right = bin[k] == kMissingBin ? (split & 1) != 0 : bin[k] >= split >> 1;
                if (col[k] == SEARCH) {
                    const int f = tb.nodes[node[k]].split_feature_id, cb = tb.cut_row_ptr[f], ce = tb.cut_row_ptr[f + 1];
                    right = csr_goes_right(bins, r, cb, ce, cb + (split >> 1), (split & 1) != 0);
                }
                child = 2 * x + (right ? 1 : 0);
                tb.nid16[r] = (unsigned short)(2 * off + 1 + child);  // (children of node x: 2 x + 1, 2 x + 2)
                atomicAdd(&cnt[(child << log_copies) + copy], 1);
            }
            if (tb.row_word != nullptr) tb.row_word[r] = (word[k] & ~kRareNodeMask) | (unsigned)child;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 2 * nl; i += kSpBlock) {
        int rows = 0;
        for (int c = 0; c < 1 << log_copies; ++c) rows += cnt[(i << log_copies) + c];
        if (rows != 0) atomicAdd(&tb.node_rows[2 * off + 1 + i], rows);  // children of level node x: 2 (off + x) + 1, + 2
    }
}

// The rows' words of a tree, every row in the root.
__global__ __launch_bounds__(256) void k_sparse_row_words(TreeBuffers tb_all, const GHPair *__restrict__ gh) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    const QuantCtl q = *tb.quant;
    for (int r = blockIdx.x * 256 + threadIdx.x; r < tb.n; r += gridDim.x * 256) tb.row_word[r] = rare_row_word(0u, gh[r], q);
}

__global__ __launch_bounds__(256) void k_sparse_cols(long nnz, const int *__restrict__ csc_bin,
                                                    const int *__restrict__ csc_row, const int *__restrict__ cut_fid,
                                                    const int *__restrict__ cut_row_ptr,
                                                    const int *__restrict__ col_of_feature, uint8_t *__restrict__ colbin,
                                                    size_t col_stride) {
    for (long e = (long)blockIdx.x * 256 + threadIdx.x; e < nnz; e += (long)gridDim.x * 256) {
        const int b = csc_bin[e];
        const int f = cut_fid[b];
        const int c = col_of_feature[f];
        if (c >= 0) colbin[(size_t)c * col_stride + csc_row[e]] = (uint8_t)(b - cut_row_ptr[f]);
    }
}

// First value of a table feature (positions [v0, v1) of the bin-major copy, rows ascend) whose row is not before `row`.
__device__ __forceinline__ int first_value_of(const int *__restrict__ rows, int v0, int v1, long row) {
    while (v0 < v1) {
        const int mid = v0 + (v1 - v0) / 2;
        if (rows[mid] < row) v0 = mid + 1;
        else v1 = mid;
    }
    return v0;
}

__global__ __launch_bounds__(256) void k_table_count(SparsePass sp, CsrBins bins, unsigned *__restrict__ count) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= sp.n_table_features) return;
    const int f = sp.table_features[i], v0 = sp.feat_val_begin[f], v1 = sp.feat_val_begin[f + 1];
    const long r0 = (long)blockIdx.y << kSpreadLogRows;
    const int m = first_value_of(bins.csc_row, v0, v1, r0 + kSpreadRows) - first_value_of(bins.csc_row, v0, v1, r0);
    count[(size_t)blockIdx.y * sp.n_lists + sp.n_rare_tasks + i] = (unsigned)(m + kSpreadGroup - 1) / kSpreadGroup;
}

// Places of a part of a table feature's values (not spread: one row block is all rows). What is left of its places after the last block's is
// nobody's. Bound by its chain: the blocks' first values are searched side by side, the groups of the blocks before are added up by all
// threads, then a value finds its place in LDS. Set-ups with a workgroup per feature and block instead, each of whose threads added up the
// blocks before: 4 M rows and 10 000 such features 28.0 ms against 16.2, 8 M and 15 000 129 against 67, 12 M rows of values that are not
// spread, which had one workgroup a feature, 67 against 27.
__global__ __launch_bounds__(256) void k_table_setup(SparsePass sp, CsrBins bins, const TablePart *__restrict__ parts,
                                                    const int *__restrict__ task_bin0, int *__restrict__ row,
                                                    unsigned short *__restrict__ table_bin, unsigned short *__restrict__ spread_row,
                                                    unsigned *__restrict__ spread_place) {
    // of the blocks that the part has values of: first value, first group, first group in the block's own list
    __shared__ int s_value[kSpreadBlocks + 1], s_group[kSpreadBlocks + 1];
    __shared__ unsigned s_list[kSpreadBlocks];
    __shared__ int s_before;
    const TablePart part = parts[blockIdx.x];
    const int i = part.feature, f = sp.table_features[i], begin = sp.feat_val_begin[f], end = sp.feat_val_begin[f + 1];
    const int v0 = begin + part.begin, count = min(kTableSetupValues, end - v0);
    const bool spread = sp.n_spread > 0;
    const int b0 = spread ? bins.csc_row[v0] >> kSpreadLogRows : 0, n_blocks = spread ? (bins.csc_row[v0 + count - 1] >> kSpreadLogRows) - b0 + 1 : 1;
    if (threadIdx.x == 0) s_before = sp.table_first[f];
    __syncthreads();
    if (spread) {
        const unsigned *lists = sp.spread_begin + sp.n_rare_tasks + i;
        int before = 0;
        for (int b = threadIdx.x; b < b0; b += 256) before += (int)(lists[(size_t)b * sp.n_lists + 1] - lists[(size_t)b * sp.n_lists]);
        if (before != 0) atomicAdd(&s_before, before);
        for (int k = threadIdx.x; k <= n_blocks; k += 256)
            s_value[k] = first_value_of(bins.csc_row, begin, end, (long)(b0 + k) << kSpreadLogRows);
        for (int k = threadIdx.x; k < n_blocks; k += 256) {
            const unsigned *at = lists + (size_t)(b0 + k) * sp.n_lists;
            s_list[k] = at[0];
            s_group[k + 1] = (int)(at[1] - at[0]);
        }
    } else if (threadIdx.x == 0) {
        s_value[0] = begin;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        s_group[0] = s_before;
        for (int k = 0; spread && k < n_blocks; ++k) s_group[k + 1] += s_group[k];
    }
    __syncthreads();
    for (int a = threadIdx.x; a < count; a += 256) {
        const int r = bins.csc_row[v0 + a], k = spread ? (r >> kSpreadLogRows) - b0 : 0, in_block = v0 + a - s_value[k];
        const size_t at = (size_t)s_group[k] * kSpreadGroup + in_block;
        row[at] = r;
        table_bin[at] = (unsigned short)(bins.csc_bin[v0 + a] - task_bin0[i]);
        if (spread) {
            spread_row[(size_t)s_list[k] * kSpreadGroup + in_block] = (unsigned short)(r & (kSpreadRows - 1));
            if (in_block % kSpreadGroup == 0) spread_place[s_list[k] + in_block / kSpreadGroup] = (unsigned)((sp.n_rare_places + at) / kSpreadGroup);
        }
    }
    // nobody's places behind the blocks whose last value is the part's, and behind the feature's last block
    for (int k = threadIdx.x; spread && k < n_blocks; k += 256) {
        if (s_value[k + 1] - v0 > count) continue;  // (the last block: a later part has its end)
        const unsigned wide = (unsigned)(s_group[k + 1] - s_group[k]) * kSpreadGroup;
        for (unsigned a = (unsigned)(s_value[k + 1] - s_value[k]); a < wide; ++a) {
            row[(size_t)s_group[k] * kSpreadGroup + a] = 0;
            table_bin[(size_t)s_group[k] * kSpreadGroup + a] = (unsigned short)kTableEmpty;
            spread_row[(size_t)s_list[k] * kSpreadGroup + a] = 0;
        }
    }
    if (v0 + count != end) return;
    const size_t used = spread ? (size_t)s_group[n_blocks] * kSpreadGroup : (size_t)s_group[0] * kSpreadGroup + (size_t)(end - begin);
    for (size_t at = used + threadIdx.x; at < (size_t)sp.table_first[f + 1] * kSpreadGroup; at += 256) {
        row[at] = 0;
        table_bin[at] = (unsigned short)kTableEmpty;
    }
}

// table_first from the table features' groups. The others' are not read, and the host does not make them: 2 M features of three values
// 57.7 ms a call with one tree while it did, 43.0 without (49.3 before their values were spread).
__global__ __launch_bounds__(256) void k_table_first(int n_table, const int *__restrict__ table_features, const int *__restrict__ first,
                                                     int *__restrict__ table_first) {
    const int i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n_table) return;
    table_first[table_features[i]] = first[i];
    table_first[table_features[i] + 1] = first[i + 1];  // (a table feature's own, if it is one)
}

// Groups of four places that the values of a task take in every row block.
__global__ __launch_bounds__(256) void k_rare_count(SparsePass sp, CsrBins bins, unsigned *__restrict__ count) {
    __shared__ unsigned values[kSpreadBlocks];
    const RareTask task = sp.rare_tasks[blockIdx.x];
    for (int b = threadIdx.x; b < sp.n_spread; b += 256) values[b] = 0u;
    __syncthreads();
    for (int fi = 0; fi < task.n_feat; ++fi) {
        const int f = sp.rare_fid[task.meta_begin + fi];
        const int v0 = sp.feat_val_begin[f], v1 = sp.feat_val_begin[f + 1];
        for (int v = v0 + (int)threadIdx.x; v < v1; v += 256) atomicAdd(&values[bins.csc_row[v] >> kSpreadLogRows], 1u);
    }
    __syncthreads();
    for (int b = threadIdx.x; b < sp.n_spread; b += 256)
        count[(size_t)b * sp.n_lists + blockIdx.x] = (values[b] + kSpreadGroup - 1) / kSpreadGroup;
}

// Places of the values of a task: spread ones by row block (in a block in any order), else its features one after the other, each
// in the order of the bin-major copy.
__global__ __launch_bounds__(256) void k_rare_setup(SparsePass sp, CsrBins bins, const int *__restrict__ cut_row_ptr,
                                                   int *__restrict__ row, unsigned *__restrict__ key, int *__restrict__ places,
                                                   uint8_t *__restrict__ group, unsigned short *__restrict__ spread_row,
                                                   unsigned *__restrict__ spread_place) {
    __shared__ unsigned first[kSpreadBlocks + 1], taken[kSpreadBlocks], from[kSpreadBlocks];
    const RareTask task = sp.rare_tasks[blockIdx.x];
    const int blocks = sp.n_spread;
    for (int b = threadIdx.x; b < blocks; b += 256) {
        const unsigned *at = sp.spread_begin + (size_t)b * sp.n_lists + blockIdx.x;
        from[b] = at[0] * kSpreadGroup;
        first[b + 1] = (at[1] - at[0]) * kSpreadGroup;
        taken[b] = 0u;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        first[0] = 0u;
        for (int b = 0; b < blocks; ++b) first[b + 1] += first[b];
        places[blockIdx.x] = blocks > 0 ? (int)first[blocks] : task.count;
    }
    __syncthreads();
    int done = 0;
    for (int fi = 0; fi < task.n_feat; ++fi) {
        const int f = sp.rare_fid[task.meta_begin + fi];
        const int v0 = sp.feat_val_begin[f], m = sp.feat_val_begin[f + 1] - v0;
        const int fbegin = cut_row_ptr[f];
        for (int a = threadIdx.x; a < m; a += 256) {
            const int r = bins.csc_row[v0 + a];
            const unsigned sixty_fourth = (unsigned)(a * kRareMaxGroups / m);
            int at = task.v_begin + done + a;
            if (blocks > 0) {
                const int b = r >> kSpreadLogRows;
                const unsigned mine = atomicAdd(&taken[b], 1u);
                at = task.v_begin + (int)(first[b] + mine);
                group[at] = (uint8_t)sixty_fourth;
                spread_row[from[b] + mine] = (unsigned short)(r & (kSpreadRows - 1));
            }
            row[at] = r;
            key[at] = ((unsigned)fi << kRareFeatShift) | sixty_fourth << 8 | (unsigned)(bins.csc_bin[v0 + a] - fbegin);
        }
        done += m;
    }
    __syncthreads();
    for (int b = threadIdx.x; b < blocks; b += 256) {
        const unsigned wide = first[b + 1] - first[b];
        for (unsigned i = taken[b]; i < wide; ++i) {
            const int at = task.v_begin + (int)(first[b] + i);
            row[at] = 0;
            key[at] = kRareEmpty;
            group[at] = 0;
            spread_row[from[b] + i] = 0;
        }
        for (unsigned i = 0; i < wide; i += kSpreadGroup)
            spread_place[(from[b] + i) / kSpreadGroup] = (unsigned)(task.v_begin + (int)(first[b] + i)) / kSpreadGroup;
    }
}

}  // namespace

void launch_sparse_cols(hipStream_t s, long nnz, const int *csc_bin, const int *csc_row, const int *cut_fid,
                        const int *cut_row_ptr, const int *col_of_feature, uint8_t *colbin, size_t col_stride) {
    if (nnz == 0) return;
    const int grid = (int)std::min<long>(16384, (nnz + 255) / 256);
    k_sparse_cols<<<grid, 256, 0, s>>>(nnz, csc_bin, csc_row, cut_fid, cut_row_ptr, col_of_feature, colbin, col_stride);
}

void launch_spread_count(hipStream_t s, const CsrBins &bins, const SparsePass &sp, unsigned *count) {
    if (sp.n_rare_tasks > 0) k_rare_count<<<sp.n_rare_tasks, 256, 0, s>>>(sp, bins, count);
    if (sp.n_table_features > 0)
        k_table_count<<<dim3((sp.n_table_features + 255) / 256, sp.n_spread), 256, 0, s>>>(sp, bins, count);
}

void launch_table_first(hipStream_t s, int n_table, const int *table_features, const int *first, int *table_first) {
    if (n_table > 0) k_table_first<<<(n_table + 255) / 256, 256, 0, s>>>(n_table, table_features, first, table_first);
}

void launch_table_setup(hipStream_t s, const CsrBins &bins, const SparsePass &sp, int n_parts, const TablePart *parts, const int *task_bin0,
                        int *row, unsigned short *table_bin, unsigned short *spread_row, unsigned *spread_place) {
    if (n_parts > 0) k_table_setup<<<n_parts, 256, 0, s>>>(sp, bins, parts, task_bin0, row, table_bin, spread_row, spread_place);
}

void launch_rare_setup(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const SparsePass &sp, int *row, unsigned *key,
                       int *places, uint8_t *group, unsigned short *spread_row, unsigned *spread_place) {
    if (sp.n_rare_tasks == 0) return;
    k_rare_setup<<<sp.n_rare_tasks, 256, 0, s>>>(sp, bins, tb.cut_row_ptr, row, key, places, group, spread_row, spread_place);
}

void launch_sparse_row_words(hipStream_t s, const TreeBuffers &tb, const GHPair *gh, int n_class) {
    if (tb.row_word == nullptr) return;
    k_sparse_row_words<<<dim3(std::max(1, std::min(1024, (tb.n + 255) / 256)), 1, n_class), 256, 0, s>>>(tb, gh);
}

void launch_sparse_level(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const SparsePass &sp,
                         const GHPair *gh, int level, float mcw, float lambda, bool dump_hist, int n_class) {
    // LDS table of a table task: room for one feature of 255 bins with every node of the level, at least 2048 and at
    // most kSparseCells cells (shallow levels: small tables, two workgroups per CU; deep levels: node ranges)
    int n_cells = 2048;
    while (n_cells < kSparseCells && n_cells < 256 * (1 << level)) n_cells *= 2;
    const size_t lds = sizeof(longlong2) * (size_t)n_cells;
    if (dump_hist) {
        // the table kernels store the cells of their features, the rare features' values are added: start from zero
        for (int k = 0; k < n_class; ++k)
            launch_fill_f32(s, reinterpret_cast<float *>(tb.for_class(k).hist(level)), 0.f,
                            (size_t)(1 << level) * tb.n_bins * 4);
    }
#define TGBM_SPARSE_LEVEL(NODES, WORDS, BPL, DEEP)                                                                            \
    {                                                                                                                       \
        static LdsOptIn opt_in;                                                                                             \
        opt_in({reinterpret_cast<const void *>(&k_sparse_level<NODES, WORDS, BPL, DEEP>)});                                  \
        k_sparse_level<NODES, WORDS, BPL, DEEP><<<tasks, kSpBlock, lds, s>>>(tb, sp, gh, level, mcw, lambda, dump_hist ? 1 : 0, n_cells); \
    }
#define TGBM_SPARSE_LEVEL_OF(WORDS, BPL, ROOT_DEEP)                                                                          \
    {                                                                                                                       \
        if (level == 0 && spread && WORDS && sp.table_gh != nullptr) TGBM_SPARSE_LEVEL(kRootWords, true, BPL, ROOT_DEEP)      \
        else if (level == 0) TGBM_SPARSE_LEVEL(kRootNode, WORDS, BPL, ROOT_DEEP)                                             \
        else if (spread && (ROOT_DEEP || level > 3)) TGBM_SPARSE_LEVEL(kSpreadNodes, WORDS, BPL, true)                        \
        else if (spread) TGBM_SPARSE_LEVEL(kSpreadNodes, WORDS, BPL, ROOT_DEEP)                                              \
        else if (ROOT_DEEP || level > 3) TGBM_SPARSE_LEVEL(kRowNodes, WORDS, BPL, true)                                      \
        else TGBM_SPARSE_LEVEL(kRowNodes, WORDS, BPL, ROOT_DEEP)                                                             \
    }
    static LdsOptIn opt_in;
    opt_in({reinterpret_cast<const void *>(&k_sparse_big<1>), reinterpret_cast<const void *>(&k_sparse_big<4>),
            reinterpret_cast<const void *>(&k_sparse_spread<kBringCodes>), reinterpret_cast<const void *>(&k_sparse_spread<kBringPairs>)});
    const bool spread = sp.n_spread > 0 && level <= kSpreadLevel;
    if (spread) {
        // (a workgroup begins with the block's rows: no more of them than the chip holds at once)
        const auto grid = [&](int workgroups) { return dim3(std::max(1, workgroups / (sp.n_spread * n_class)), sp.n_spread, n_class); };
        if (level > 0) k_sparse_spread<kBringNodes><<<grid(512), 1024, kSpreadRows, s>>>(tb, sp, level);
        if (level == 0 && sp.n_rare_tasks > 0) k_sparse_spread<kBringCodes><<<grid(256), 1024, kSpreadRows * sizeof(unsigned), s>>>(tb, sp, level);
        if (level == 0 && sp.gh_words != nullptr && sp.table_gh != nullptr)
            k_sparse_spread<kBringPairs><<<grid(256), 1024, kSpreadRows * sizeof(unsigned), s>>>(tb, sp, level);
    }
    if (sp.n_tasks > 0) {
        const dim3 tasks(sp.n_tasks, 1, n_class);
        if (sp.gh_words != nullptr && sp.max_table_bins <= 64) TGBM_SPARSE_LEVEL_OF(true, 1, false)
        else if (sp.gh_words != nullptr) TGBM_SPARSE_LEVEL_OF(true, 4, true)
        else if (sp.max_table_bins <= 64) TGBM_SPARSE_LEVEL_OF(false, 1, false)
        else TGBM_SPARSE_LEVEL_OF(false, 4, true)
    }
#undef TGBM_SPARSE_LEVEL_OF
#undef TGBM_SPARSE_LEVEL
    if (sp.n_big > 0) {
        // (as many workgroups as the chip holds at once: each is a chain of some ten dependent steps, whatever its nodes are)
        const dim3 grid(sp.n_big, std::min(1 << level, std::max(1, std::min(16, 512 / (sp.n_big * n_class)))), n_class);
        n_cells = std::min(n_cells, sp.max_table_bins * (((1 << level) + (int)grid.y - 1) / (int)grid.y));
        const size_t lds = sizeof(longlong2) * (size_t)n_cells;
        if (sp.max_table_bins <= 64) k_sparse_big<1><<<grid, kSpBlock, lds, s>>>(tb, sp, level, mcw, lambda, dump_hist ? 1 : 0, n_cells);
        else k_sparse_big<4><<<grid, kSpBlock, lds, s>>>(tb, sp, level, mcw, lambda, dump_hist ? 1 : 0, n_cells);
    }
    if (sp.n_rare_tasks > 0) {
        const size_t nodes_lds = (size_t)(1 << level) * 20;
        const dim3 tiles(sp.n_rare_tasks, 1, n_class);
        if (dump_hist && spread) k_sparse_rare_filter<true, true><<<tiles, kRareBlock, nodes_lds, s>>>(tb, sp, gh, level, mcw, lambda);
        else if (dump_hist) k_sparse_rare_filter<true, false><<<tiles, kRareBlock, nodes_lds, s>>>(tb, sp, gh, level, mcw, lambda);
        else if (spread) k_sparse_rare_filter<false, true><<<tiles, kRareBlock, nodes_lds, s>>>(tb, sp, gh, level, mcw, lambda);
        else k_sparse_rare_filter<false, false><<<tiles, kRareBlock, nodes_lds, s>>>(tb, sp, gh, level, mcw, lambda);
        k_sparse_rare_search<<<dim3(sp.n_rare_groups, 1, n_class), kRareBlock, nodes_lds, s>>>(tb, sp, gh, level, mcw, lambda);
    }
}

void launch_sparse_partition(hipStream_t s, const TreeBuffers &all, const CsrBins &bins, const SparsePass &sp, int level, int n_class) {
    // (spread values: nobody asks a row's word for its node but the levels past kSpreadLevel)
    TreeBuffers tb = all;
    if (sp.n_spread > 0 && (level < kSpreadLevel || level + 1 >= tb.depth)) tb.row_word = nullptr;
    const int grid = std::max(1, std::min(1024, (tb.n + kSpBlock * kMoveRows - 1) / (kSpBlock * kMoveRows)));
    k_sparse_partition<<<dim3(grid, 1, n_class), kSpBlock, 0, s>>>(tb, bins, level);
}

}  // namespace tgbm
