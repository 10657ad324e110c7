// Tree-traversal prediction (the reference's Predictor::predict_raw, src/thundergbm/predictor.cu:32-189)
// and the objectives' predict_transform.
#include <type_traits>

#include "device_api.h"

namespace tgbm {
namespace {

constexpr int kBlock = 256;

// Value of feature `f` in a CSR row with ascending column indices; `missing` when not stored.
__device__ __forceinline__ float row_value(const int *__restrict__ ci, const float *__restrict__ cv, int len, int f,
                                           bool *missing) {
    int lo = 0, hi = len;
    while (lo < hi) {
        int mid = lo + (hi - lo) / 2;
        int c = ci[mid];
        if (c == f) {
            *missing = false;
            return cv[mid];
        }
        if (c > f)
            hi = mid;
        else
            lo = mid + 1;
    }
    *missing = true;
    return 0.f;
}

// One thread per row; the model (all trees, 48-byte nodes) is read through the caches. ACC is
// double where the reference takes its shared-memory path (n_features * 128 * 4 <= 48 KB, :85) and
// float otherwise (:166); in the double path a stored +inf counts as missing (:96-118).
template <typename ACC, bool INF_IS_MISSING>
__global__ __launch_bounds__(kBlock) void k_predict(int n, const int *__restrict__ row_ptr, const int *__restrict__ col,
                                                   const float *__restrict__ val, const TreeNode *__restrict__ model,
                                                   int n_iter, int n_class_trees, int n_nodes, float lr,
                                                   float base_score, float *__restrict__ out, size_t out_stride) {
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int rb = row_ptr[i];
    const int len = row_ptr[i + 1] - rb;
    const int *ci = col + rb;
    const float *cv = val + rb;
    for (int t = 0; t < n_class_trees; ++t) {
        ACC sum = base_score;
        for (int it = 0; it < n_iter; ++it) {
            const TreeNode *nd = model + ((size_t)it * n_class_trees + t) * n_nodes;
            int cur = 0;
            while (!nd[cur].is_leaf) {
                const TreeNode &c = nd[cur];
                bool missing;
                float v = row_value(ci, cv, len, c.split_feature_id, &missing);
                if (INF_IS_MISSING && !(v < INFINITY)) missing = true;
                if (!missing)
                    cur = v < c.split_value ? c.lch_index : c.rch_index;
                else
                    cur = c.default_right ? c.rch_index : c.lch_index;
            }
            sum += lr * nd[cur].base_weight;
        }
        out[(size_t)t * out_stride + i] += (float)sum;
    }
}

// The reference's shared-memory path (predictor.cu:85-160): every thread first spreads its row into a dense
// vector of F floats (+inf = not stored, which is why a stored +inf counts as missing there), then walks
// all trees with one LDS read per node instead of a binary search of the CSR row. Feature-major LDS layout
// (f * kStageBlock + thread) keeps the reads of a wavefront on distinct banks. Sums are double as in the
// reference's path.
constexpr int kStageBlock = 128;

__global__ __launch_bounds__(kStageBlock) void k_predict_staged(int n, int F, const int *__restrict__ row_ptr,
                                                               const int *__restrict__ col,
                                                               const float *__restrict__ val,
                                                               const TreeNode *__restrict__ model, int n_iter,
                                                               int n_class_trees, int n_nodes, float lr,
                                                               float base_score, float *__restrict__ out,
                                                               size_t out_stride) {
    extern __shared__ float dense[];  // [F][kStageBlock]
    const int i = blockIdx.x * kStageBlock + threadIdx.x;
    for (int f = 0; f < F; ++f) dense[f * kStageBlock + threadIdx.x] = INFINITY;
    if (i >= n) return;  // no barrier below: a thread only reads what it wrote
    const int rb = row_ptr[i], re = row_ptr[i + 1];
    for (int e = rb; e < re; ++e) {
        const int c = col[e];
        if (c < F) dense[c * kStageBlock + threadIdx.x] = val[e];
    }
    for (int t = 0; t < n_class_trees; ++t) {
        double sum = base_score;
        for (int it = 0; it < n_iter; ++it) {
            const TreeNode *nd = model + ((size_t)it * n_class_trees + t) * n_nodes;
            int cur = 0;
            while (!nd[cur].is_leaf) {
                const TreeNode &c = nd[cur];
                const int f = c.split_feature_id;
                const float v = f < F ? dense[f * kStageBlock + threadIdx.x] : INFINITY;
                if (v < INFINITY)
                    cur = v < c.split_value ? c.lch_index : c.rch_index;
                else
                    cur = c.default_right ? c.rch_index : c.lch_index;
            }
            sum += lr * nd[cur].base_weight;
        }
        out[(size_t)t * out_stride + i] += (float)sum;
    }
}

// The same walk with the trees in LDS: the workgroup's rows are spread into the dense vector as above, then the trees
// of a class are staged a few at a time as 16-byte records (one LDS read per node visit instead of several cached
// global reads of the 48-byte node) and every thread walks the staged trees. Same operations in the same order as
// k_predict_staged, hence the same bits. A walk is cut off after n_nodes steps (a malformed model file).
__global__ void k_pack_model(const TreeNode *__restrict__ model, long n_total, int n_nodes, PackedNode *__restrict__ packed) {
    for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < n_total; i += (long)gridDim.x * blockDim.x) {
        const TreeNode nd = model[i];
        PackedNode p;
        p.split_value = nd.split_value;
        p.base_weight = nd.base_weight;
        const bool children_ok = nd.lch_index >= 0 && nd.lch_index < n_nodes && nd.rch_index >= 0 && nd.rch_index < n_nodes;
        const bool leaf = nd.is_leaf || !children_ok;  // (an index outside the tree ends the walk instead of leaving it)
        p.children = leaf ? 0u : ((unsigned)nd.lch_index | (unsigned)nd.rch_index << 16);
        const unsigned f = (nd.split_feature_id >= 0 && nd.split_feature_id < 0xffffff) ? (unsigned)nd.split_feature_id : 0xffffffu;
        p.meta = f | (nd.default_right ? 1u << 30 : 0u) | (leaf ? 1u << 31 : 0u);
        packed[i] = p;
    }
}

template <int B>
__global__ __launch_bounds__(B) void k_predict_lds(int n, int F, const int *__restrict__ row_ptr,
                                                   const int *__restrict__ col, const float *__restrict__ val,
                                                   const PackedNode *__restrict__ packed, int n_iter, int n_class_trees,
                                                   int n_nodes, float lr, float base_score, float *__restrict__ out,
                                                   size_t out_stride, int trees_per_stage) {
    extern __shared__ float smem[];
    float *dense = smem;                                       // [F][B]
    uint4 *nodes = reinterpret_cast<uint4 *>(smem + F * B);    // [trees_per_stage][n_nodes]
    const int i = blockIdx.x * B + threadIdx.x;
    const bool live = i < n;
    for (int f = 0; f < F; ++f) dense[f * B + threadIdx.x] = INFINITY;
    if (live) {
        const int rb = row_ptr[i], re = row_ptr[i + 1];
        for (int e = rb; e < re; ++e) {
            const int c = col[e];
            if (c < F) dense[c * B + threadIdx.x] = val[e];
        }
    }
    const uint4 *__restrict__ src = reinterpret_cast<const uint4 *>(packed);
    for (int t = 0; t < n_class_trees; ++t) {
        double sum = base_score;
        for (int it0 = 0; it0 < n_iter; it0 += trees_per_stage) {
            const int staged = min(trees_per_stage, n_iter - it0);
            __syncthreads();  // the walks of the previous stage are done
            for (int idx = threadIdx.x; idx < staged * n_nodes; idx += B) {
                const int k = idx / n_nodes, j = idx - k * n_nodes;
                nodes[idx] = src[((size_t)(it0 + k) * n_class_trees + t) * n_nodes + j];
            }
            __syncthreads();
            if (!live) continue;
            for (int k = 0; k < staged; ++k) {
                const uint4 *tree = nodes + k * n_nodes;
                int cur = 0;
                uint4 nd = tree[0];
                for (int step = 0; step < n_nodes && !(nd.w >> 31); ++step) {
                    const unsigned f = nd.w & 0xffffffu;
                    const float v = f < (unsigned)F ? dense[f * B + threadIdx.x] : INFINITY;
                    const unsigned l = nd.z & 0xffffu, r = nd.z >> 16;
                    if (v < INFINITY)
                        cur = v < __uint_as_float(nd.x) ? l : r;
                    else
                        cur = ((nd.w >> 30) & 1u) ? r : l;
                    nd = tree[cur];
                }
                sum += lr * __uint_as_float(nd.y);
            }
        }
        if (live) out[(size_t)t * out_stride + i] += (float)sum;
    }
}

// ---- the walk on order-preserving integer keys
// A float that is not a NaN maps to an unsigned key with the floats' order (-0 counts as +0): `v < t` is
// `key(v) < key(t)`. In a row's dense vector a value that is missing - not stored, or stored as +inf or NaN, which the
// reference's shared-memory path takes for missing (predictor.cu:96-118) - is the largest key, 0xffffffff; nothing else
// maps there. A split node whose default direction is left adds one to the value's key before it compares (the missing
// key wraps to 0 and goes left; every other key keeps its order, as does the node's threshold key, which has the one
// added when the record is packed), so the default direction costs no comparison of its own.
__device__ __forceinline__ unsigned order_key(float v) {
    if (v == 0.f) v = 0.f;  // -0 -> +0
    const unsigned b = __float_as_uint(v);
    return b ^ ((unsigned)((int)b >> 31) | 0x80000000u);
}
constexpr unsigned kMissingKey = 0xffffffffu;
__device__ __forceinline__ unsigned value_key(float v) { return v < INFINITY ? order_key(v) : kMissingKey; }

// The rows of a call as the scoring kernels read them: CSR entries (row_ptr addresses the slice's first row), or a dense
// row-major matrix in which a zero is a value that is not stored (minus_zero_is_stored: -0 is a stored zero,
// upload_doubles_as_floats).
//
// Key of a stored value. NARROW: the reference's shared-memory path, where a stored +inf or NaN counts as missing; else
// its global-memory path (predictor.cu:160-189), where +inf is a value and a NaN, which is not below any threshold, goes
// right like the largest value.
template <bool NARROW>
__device__ __forceinline__ unsigned stored_key(float v) {
    if (NARROW) return value_key(v);
    return v != v ? kMissingKey - 1u : order_key(v);
}
template <bool NARROW>
__device__ __forceinline__ unsigned dense_key(float v, bool minus_zero_is_stored) {
    const bool stored = is_stored(v, minus_zero_is_stored);
    return stored ? stored_key<NARROW>(v) : kMissingKey;
}
// Sums: double where the reference's shared-memory path is (predictor.cu:85-160), else float with the product and the
// sum in one rounding, as the compiler contracts k_predict's.
__device__ __forceinline__ double add_leaf(double sum, float lr, float w) { return sum + lr * w; }
__device__ __forceinline__ float add_leaf(float sum, float lr, float w) { return fmaf(lr, w, sum); }

// Many rows: a thread per row, the row's keys of the features that the model uses in LDS (feature-major, so the reads of
// a wavefront never conflict), the trees of a class staged in LDS tps at a time, ILP trees walked at a time by every
// thread and `depth` steps for every tree: the walks of different trees do not depend on each other, so their LDS round
// trips (node, feature key, node, ...) overlap; a walk that has reached its leaf stays there until the deepest possible
// walk is done (straight-line code: nine vector instructions and two LDS reads per step). The leaf weights are added in
// the order of the trees, as in the other kernels: same bits. 10 M rows x 40 trees of depth 8: 2.0 ms (two trees per
// stage; 2.1 with four, 2.7 with one), bound by the LDS (busy 62 %) and the vector ALUs (57 %).
// CSR rows of equal length with ascending columns (dense data handed over as CSR) are spread into the LDS vectors by
// consecutive lanes reading consecutive entries - whole cache lines per load instruction instead of one 4-byte word from
// each of 64 lines; anything else takes the row-per-thread loop (whose result for a repeated column, the later entry,
// does not depend on the order in which lanes write). A dense matrix is read by the row's thread, used columns only.
template <int B, int ILP, int kFetch, bool NARROW>
__global__ __launch_bounds__(B) void k_score_rows(ScoreRows rows_in, ScoreModel m, float lr, float base_score,
                                                  float *__restrict__ out, size_t out_stride, int trees_per_stage,
                                                  int coalesced_fill, int classes) {
    using Sum = typename std::conditional<NARROW, double, float>::type;
    extern __shared__ unsigned smem_u[];
    const int n = rows_in.n, slots = m.n_slots, n_nodes = m.n_nodes, n_iter = m.n_iter;
    const int class0 = blockIdx.y * classes, class1 = min(m.n_class, class0 + classes);  // (one at least)
    unsigned *dense = smem_u;                                        // [slots][B] keys
    uint2 *nodes = reinterpret_cast<uint2 *>(smem_u + slots * B);    // [trees_per_stage][n_nodes]
    const int row0 = blockIdx.x * B;
    const int i = row0 + threadIdx.x;
    const bool live = i < n;
    for (int f = 0; f < slots; ++f) dense[f * B + threadIdx.x] = f == m.leaf_slot ? 0u : kMissingKey;
    if (rows_in.x != nullptr) {
        const float *__restrict__ x = rows_in.x + (size_t)min(i, n - 1) * rows_in.columns;
        for (int f0 = 0; f0 < m.n_used; f0 += 8) {  // (eight loads in flight; the feature list is read by scalar loads)
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const int f = m.used[min(f0 + u, m.n_used - 1)];
                v[u] = x[min(f, rows_in.columns - 1)];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (f0 + u < m.n_used && m.used[f0 + u] < rows_in.columns)
                    dense[(f0 + u) * B + threadIdx.x] = dense_key<NARROW>(v[u], rows_in.minus_zero_is_stored);
        }
    } else {
        const int *__restrict__ row_ptr = rows_in.row_ptr;
        const int *__restrict__ col = rows_in.col;
        const float *__restrict__ val = rows_in.val;
        const int *__restrict__ slot_of = m.slot_of;
        const int rb = live ? row_ptr[i] : 0, re = live ? row_ptr[i + 1] : 0;
        const int len0 = row_ptr[row0 + 1] - row_ptr[row0];  // (row0 < n: the grid covers no workgroup without rows)
        bool per_row = true;
        if (coalesced_fill && __syncthreads_and(!live || re - rb == len0) && len0 > 0) {
            // (the barrier above also orders the clearing before the writes of other lanes below)
            const int rows = min(B, n - row0);
            const int e0 = row_ptr[row0];
            const int total = rows * len0;
            int r = threadIdx.x / len0, slot = threadIdx.x - r * len0;
            const int dr = B / len0, ds = B - dr * len0;
            bool bad = false;
            // (four entries per lane in flight: the loop is a chain of memory round trips otherwise)
            for (int idx0 = threadIdx.x; idx0 < total; idx0 += 4 * B) {
                int c[4], before[4], at[4];
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int idx = min(idx0 + u * B, total - 1);
                    c[u] = col[e0 + idx];
                    v[u] = val[e0 + idx];
                    // ascending inside the row: the entry before this one sits in the lane below (or, for lane 0, in memory)
                    before[u] = (threadIdx.x & 63) == 0 && idx > 0 ? col[e0 + idx - 1] : 0;
                }
#pragma unroll
                for (int u = 0; u < 4; ++u) at[u] = slot_of[min((unsigned)c[u], (unsigned)m.n_features)];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    const int below = __shfl_up(c[u], 1);
                    if ((threadIdx.x & 63) != 0) before[u] = below;
                    if (idx0 + u * B < total) {
                        if (slot > 0 && before[u] >= c[u]) bad = true;
                        if (at[u] >= 0) dense[at[u] * B + r] = stored_key<NARROW>(v[u]);
                    }
                    r += dr;
                    slot += ds;
                    if (slot >= len0) {
                        slot -= len0;
                        ++r;
                    }
                }
            }
            per_row = __syncthreads_or(bad);
            if (per_row)
                for (int f = 0; f < m.n_used; ++f) dense[f * B + threadIdx.x] = kMissingKey;
        }
        if (per_row) {
            for (int e = rb; e < re; e += 4) {  // (four entries in flight, written in their order)
                int at[4];
                float v[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    at[u] = slot_of[min((unsigned)col[min(e + u, re - 1)], (unsigned)m.n_features)];
                    v[u] = val[min(e + u, re - 1)];
                }
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    if (e + u < re && at[u] >= 0) dense[at[u] * B + threadIdx.x] = stored_key<NARROW>(v[u]);
            }
        }
    }
    // (byte offsets into the workgroup's LDS, so that a step adds record fields to them without further scaling)
    const char *lds = reinterpret_cast<const char *>(smem_u);
    const unsigned mine = threadIdx.x * 4u;  // this row's key of slot 0
    const unsigned trees0 = (unsigned)slots * B * 4u;
    // The trees of a stage are fetched into registers while the stage before is walked and go to the LDS between two
    // barriers after it, so that no walk waits for global memory (kFetch records per thread, as many as the stage needs:
    // the loads are unconditional - clamped -, or the compiler waits for them at once; stages of more than 8 records
    // per thread are copied after the barrier instead).
    const bool prefetch = trees_per_stage * n_nodes <= kFetch * B;
    uint2 fetched[kFetch];
    auto fetch = [&](int t, int it0) {
        const int count = min(trees_per_stage, n_iter - it0) * n_nodes;
        const uint2 *src = m.records + ((size_t)t * n_iter + it0) * n_nodes;
#pragma unroll
        for (int q = 0; q < kFetch; ++q) fetched[q] = src[min((int)threadIdx.x + q * B, count - 1)];
    };
    if (prefetch) fetch(class0, 0);
    for (int t = class0; t < class1; ++t) {
        Sum sum = base_score;
        for (int it0 = 0; it0 < n_iter; it0 += trees_per_stage) {
            const int staged = min(trees_per_stage, n_iter - it0);
            __syncthreads();  // the walks of the previous stage are done (and, the first time, the vectors are filled)
            if (prefetch) {
#pragma unroll
                for (int q = 0; q < kFetch; ++q) {
                    const int idx = threadIdx.x + q * B;
                    if (idx < staged * n_nodes) nodes[idx] = fetched[q];
                }
                // the next stage: of this class, or the first of the next class
                if (it0 + trees_per_stage < n_iter) fetch(t, it0 + trees_per_stage);
                else if (t + 1 < class1) fetch(t + 1, 0);
            } else {
                const uint2 *src = m.records + ((size_t)t * n_iter + it0) * n_nodes;
                for (int idx = threadIdx.x; idx < staged * n_nodes; idx += B) nodes[idx] = src[idx];
            }
            __syncthreads();
            if (!live) continue;
            for (int k = 0; k < staged; k += ILP) {
                unsigned tree[ILP];
                uint2 nd[ILP];
#pragma unroll
                for (int j = 0; j < ILP; ++j) {
                    // (past the last staged tree: the last one is walked again and not added)
                    tree[j] = trees0 + (unsigned)(min(k + j, staged - 1) * n_nodes) * 8u;
                    nd[j] = *reinterpret_cast<const uint2 *>(lds + tree[j]);
                }
                for (int step = 0; step < m.depth; ++step) {
                    unsigned key[ILP];
#pragma unroll
                    for (int j = 0; j < ILP; ++j)
                        key[j] = *reinterpret_cast<const unsigned *>(lds + (mine + (nd[j].y & 0x7fffu) * (B * 4u)));
#pragma unroll
                    for (int j = 0; j < ILP; ++j) {
                        const bool right = key[j] + (nd[j].y >> 31) > nd[j].x;
                        nd[j] = *reinterpret_cast<const uint2 *>(lds + (tree[j] + ((nd[j].y >> 15) & 0xffffu) + (right ? 8u : 0u)));
                    }
                }
#pragma unroll
                for (int j = 0; j < ILP; ++j)
                    if (k + j < staged) sum = add_leaf(sum, lr, __uint_as_float(nd[j].x));
            }
        }
        if (live) out[(size_t)t * out_stride + i] = 0.f + (float)sum;
    }
}

// Few rows, or rows over more features than k_score_rows' vectors hold: G lanes per row (a wavefront, or the whole
// workgroup), a tree per lane. The row's keys of the used features are spread into LDS once; the node records come
// through the caches - the top of a tree is one line that stays in the L1, the lower levels come from the L2 - and the
// leaf weights meet in LDS, where one lane per class adds them in the order of the trees: same bits as k_score_rows.
// One row of 100 trees is two dependent walks of `depth` L2 round trips instead of a hundred LDS walks by one thread.
constexpr int kScoreGroupTrees = 256;  // leaf weights of a row that meet in LDS at a time

template <int G, bool NARROW>
__global__ __launch_bounds__(256) void k_score_group(ScoreRows rows_in, ScoreModel m, float lr, float base_score,
                                                     float *__restrict__ out, size_t out_stride) {
    using Sum = typename std::conditional<NARROW, double, float>::type;
    constexpr int R = 256 / G;  // rows of a workgroup
    extern __shared__ unsigned smem_u[];
    const int g = threadIdx.x / G, lane = threadIdx.x % G;
    const int n_class = m.n_class, n_iter = m.n_iter, slots = m.n_slots;
    Sum *sums = reinterpret_cast<Sum *>(smem_u) + g * n_class;  // [R][n_class]
    float *weights = reinterpret_cast<float *>(reinterpret_cast<Sum *>(smem_u) + R * n_class) + g * kScoreGroupTrees;
    unsigned *keys = reinterpret_cast<unsigned *>(reinterpret_cast<float *>(reinterpret_cast<Sum *>(smem_u) + R * n_class) +
                                                  R * kScoreGroupTrees) + g * slots;
    const int row = blockIdx.x * R + g;
    const int i = min(row, rows_in.n - 1);  // (every wavefront meets every barrier)
    if (rows_in.x != nullptr) {
        const float *__restrict__ x = rows_in.x + (size_t)i * rows_in.columns;
        for (int f = lane; f < slots; f += G) {
            unsigned key = f == m.leaf_slot ? 0u : kMissingKey;
            if (f < m.n_used && m.used[f] < rows_in.columns) key = dense_key<NARROW>(x[m.used[f]], rows_in.minus_zero_is_stored);
            keys[f] = key;
        }
    } else {
        for (int f = lane; f < slots; f += G) keys[f] = f == m.leaf_slot ? 0u : kMissingKey;
        const int rb = rows_in.row_ptr[i], re = rows_in.row_ptr[i + 1];
        const int *__restrict__ col = rows_in.col;
        bool descends = false;
        __syncthreads();
        for (int e = rb + lane; e < re; e += G) {
            const int c = col[e], next = e + 1 < re ? col[e + 1] : 0x7fffffff;
            descends |= next < c;
            const int at = m.slot_of[min((unsigned)c, (unsigned)m.n_features)];
            if (at >= 0 && next != c) keys[at] = stored_key<NARROW>(rows_in.val[e]);  // (of equal columns the later entry)
        }
        if (__syncthreads_or(descends)) {
            // a row whose columns do not ascend may repeat one with others in between: entry by entry, the later one counts
            if (lane == 0)
                for (int e = rb; e < re; ++e) {
                    const int at = m.slot_of[min((unsigned)col[e], (unsigned)m.n_features)];
                    if (at >= 0) keys[at] = stored_key<NARROW>(rows_in.val[e]);
                }
        }
    }
    for (int c = lane; c < n_class; c += G) sums[c] = base_score;
    const int n_trees = n_iter * n_class;
    const char *records = reinterpret_cast<const char *>(m.records);
    for (int k0 = 0; k0 < n_trees; k0 += kScoreGroupTrees) {
        const int k1 = min(k0 + kScoreGroupTrees, n_trees);
        __syncthreads();  // the keys are filled; the previous weights are added
        constexpr int ILP = G == 64 ? 2 : 1;
        for (int k = k0 + lane; k < k1; k += ILP * G) {
            const char *tree[ILP];
            uint2 nd[ILP];
#pragma unroll
            for (int j = 0; j < ILP; ++j) {
                tree[j] = records + (size_t)min(k + j * G, k1 - 1) * m.n_nodes * 8u;
                nd[j] = *reinterpret_cast<const uint2 *>(tree[j]);
            }
            for (int step = 0; step < m.depth; ++step) {
                unsigned key[ILP];
#pragma unroll
                for (int j = 0; j < ILP; ++j) key[j] = keys[nd[j].y & 0x7fffu];
#pragma unroll
                for (int j = 0; j < ILP; ++j) {
                    const bool right = key[j] + (nd[j].y >> 31) > nd[j].x;
                    nd[j] = *reinterpret_cast<const uint2 *>(tree[j] + ((nd[j].y >> 15) & 0xffffu) + (right ? 8u : 0u));
                }
            }
#pragma unroll
            for (int j = 0; j < ILP; ++j)
                if (k + j * G < k1) weights[k + j * G - k0] = __uint_as_float(nd[j].x);
        }
        __syncthreads();
        const int c0 = k0 / n_iter, c1 = (k1 - 1) / n_iter;
        for (int c = c0 + lane; c <= c1; c += G) {
            Sum sum = sums[c];
            const int e = min(k1, (c + 1) * n_iter) - k0;
            for (int k = max(k0, c * n_iter) - k0; k < e; ++k) sum = add_leaf(sum, lr, weights[k]);
            sums[c] = sum;
        }
    }
    __syncthreads();
    if (row < rows_in.n)
        for (int c = lane; c < n_class; c += G) out[(size_t)c * out_stride + row] = 0.f + (float)sums[c];
}

// kind 1: binary label lookup, 2: arg-max label lookup, 3: softmax probabilities in place,
// 4: sigmoid (reg:logistic). regression_obj.h:27-32,76-92 and multiclass_obj.cu:44-88 of the reference.
__global__ void k_predict_transform(int kind, int n, int K, const float *__restrict__ label, float *__restrict__ y) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        if (kind == 1) {
            y[i] = label[y[i] > 0 ? 1 : 0];
        } else if (kind == 2) {
            int nc = K == 2 ? 1 : K;
            int mk = 0;
            float mp = y[i];
            for (int k = 1; k < nc; ++k) {
                float v = y[(size_t)k * n + i];
                if (mp < v) {
                    mp = v;
                    mk = k;
                }
            }
            y[i] = label[mk];
        } else if (kind == 3) {
            float mx = y[i];
            for (int k = 1; k < K; ++k) mx = fmaxf(mx, y[(size_t)k * n + i]);
            float sum = 0;
            for (int k = 0; k < K; ++k) {
                float e = expf(y[(size_t)k * n + i] - mx);
                y[(size_t)k * n + i] = e;
                sum += e;
            }
            for (int k = 0; k < K; ++k) y[(size_t)k * n + i] /= sum;
        } else if (kind == 4) {
            y[i] = 1.f / (1.f + expf(-y[i]));
        }
    }
}

}  // namespace

void launch_predict(hipStream_t s, int n, int F, const int *row_ptr, const int *col, const float *val,
                    const TreeNode *model, int n_iter, int n_class_trees, int n_nodes, float lr, float base_score,
                    float *out, size_t out_stride, const PackedNode *packed) {
    if (n == 0) return;
    if (out_stride == 0) out_stride = (size_t)n;
    if (n_class_trees > 1) base_score = 0;  // predictor.cu:81-83
    const bool dense_path = (size_t)F * 128 * sizeof(float) <= 48 * 1024;
    int grid = (n + kBlock - 1) / kBlock;
    // (TGBM_PREDICT_TPS: trees staged at a time, 0 = walk the 48-byte nodes in global memory; read at every call, so a test
    // can compare the kernels within one process)
    const int tps_given = std::getenv("TGBM_PREDICT_TPS") ? atoi(std::getenv("TGBM_PREDICT_TPS")) : -1;
    const int tps_env = tps_given < 0 ? 4 : tps_given;
    if (dense_path && packed != nullptr && tps_env > 0 && n_nodes <= 0xffff) {  // (16-bit child indices)
        // trees in LDS: 256 rows per workgroup while their dense vectors take at most 48 KB, else 128; trees are staged
        // one at a time unless several fit next to the vectors in 40 KB (four workgroups per CU: measured on 10 M rows
        // x 40 trees of depth 8, 6.0 ms with one tree per stage, 8.0 ms with four, 14.3 ms from global memory)
        const int B = (size_t)F * 256 * sizeof(float) <= 48 * 1024 ? 256 : 128;
        const size_t dense_bytes = (size_t)F * B * sizeof(float), tree_bytes = (size_t)n_nodes * sizeof(PackedNode);
        if (dense_bytes + tree_bytes <= 64 * 1024) {
            size_t fit = dense_bytes + tree_bytes <= 40 * 1024 ? (40 * 1024 - dense_bytes) / tree_bytes : 1;
            const int tps = (int)std::max<size_t>(1, std::min<size_t>((size_t)tps_env, fit));
            const size_t lds = dense_bytes + (size_t)tps * tree_bytes;
            if (B == 256)
                k_predict_lds<256><<<(n + 255) / 256, 256, lds, s>>>(n, F, row_ptr, col, val, packed, n_iter, n_class_trees,
                                                                  n_nodes, lr, base_score, out, out_stride, tps);
            else
                k_predict_lds<128><<<(n + 127) / 128, 128, lds, s>>>(n, F, row_ptr, col, val, packed, n_iter, n_class_trees,
                                                                  n_nodes, lr, base_score, out, out_stride, tps);
            return;
        }
    }
    if (dense_path)
        k_predict_staged<<<(n + kStageBlock - 1) / kStageBlock, kStageBlock, (size_t)F * kStageBlock * sizeof(float), s>>>(
            n, F, row_ptr, col, val, model, n_iter, n_class_trees, n_nodes, lr, base_score, out, out_stride);
    else
        k_predict<float, false><<<grid, kBlock, 0, s>>>(n, row_ptr, col, val, model, n_iter, n_class_trees, n_nodes, lr,
                                                       base_score, out, out_stride);
}

void launch_pack_model(hipStream_t s, const TreeNode *model, long n_total, int n_nodes, PackedNode *packed) {
    if (n_total <= 0) return;
    k_pack_model<<<(int)std::min<long>((n_total + 255) / 256, 4096), 256, 0, s>>>(model, n_total, n_nodes, packed);
}

// k_score_rows: 256 rows per workgroup while their vectors take at most 50 KB, else 128
static int score_block(const ScoreModel &m) { return (size_t)m.n_slots * 256 * sizeof(float) <= 50 * 1024 ? 256 : 128; }

constexpr int kScoreChip = 1024;  // workgroups of k_score_rows that the chip holds at a time

int score_least_rows(const ScoreModel &m) { return (kScoreGroupRows + m.n_class - 1) / m.n_class; }

int score_slice_rows(const ScoreModel &m) {
    return (kScoreChip * score_block(m) + m.n_class - 1) / m.n_class;
}

bool score_rows_fit(const ScoreModel &m) {
    const size_t dense_bytes = (size_t)m.n_slots * score_block(m) * sizeof(float);
    return dense_bytes <= 50 * 1024 && dense_bytes + (size_t)m.n_nodes * sizeof(uint2) <= 64 * 1024;
}

bool launch_score(hipStream_t s, const ScoreRows &rows, const ScoreModel &m, bool narrow, float lr, float base_score,
                  float *out, size_t out_stride) {
    if (rows.n == 0) return true;
    if (m.n_class > 1) base_score = 0;  // predictor.cu:81-83
    // (TGBM_PREDICT_COMPACT=2: without the coalesced spreading of equal-length rows; TGBM_PREDICT_TPS: that many trees per
    // stage of k_score_rows, which then takes every row count; tests and measurements)
    const char *ce = std::getenv("TGBM_PREDICT_COMPACT"), *te = std::getenv("TGBM_PREDICT_TPS");
    const char *ge = std::getenv("TGBM_PREDICT_GROUP");  // 1 / 0: k_score_group always / never where the other serves
    const int fill = ce != nullptr && atoi(ce) == 2 ? 0 : 1;
    const int B = score_block(m);
    const size_t dense_bytes = (size_t)m.n_slots * B * sizeof(float), tree_bytes = (size_t)m.n_nodes * sizeof(uint2);
    const bool rows_fit = score_rows_fit(m);
    // k_score_group
    const size_t sum_bytes = narrow ? sizeof(double) : sizeof(float);
    auto group_bytes = [&](int G) {
        return (size_t)(256 / G) * ((size_t)m.n_class * sum_bytes + kScoreGroupTrees * sizeof(float) + (size_t)m.n_slots * 4);
    };
    // A wavefront per row while four rows leave the LDS room for four workgroups per CU; the whole workgroup for rows too
    // few to fill the chip otherwise, and for wider ones.
    const int G = rows.n > 1024 && group_bytes(64) <= 40 * 1024 ? 64 : 256;
    const bool group_fits = group_bytes(G) <= 150 * 1024;
    bool group = rows.n < score_least_rows(m);
    if (te != nullptr && atoi(te) > 0) group = false;
    if (ge != nullptr) group = atoi(ge) != 0;
    if (group_fits && (group || !rows_fit)) {
        const int grid = (rows.n + 256 / G - 1) / (256 / G);
        const size_t lds = group_bytes(G);
#define TGBM_SCORE_GROUP(GG, NN) k_score_group<GG, NN><<<grid, 256, lds, s>>>(rows, m, lr, base_score, out, out_stride)
        if (G == 64) {
            if (narrow) TGBM_SCORE_GROUP(64, true);
            else TGBM_SCORE_GROUP(64, false);
        } else {
            static LdsOptIn opt_in;
            if (lds > 64 * 1024)  // (what a kernel may ask for without saying so)
                opt_in({reinterpret_cast<const void *>(&k_score_group<256, true>),
                        reinterpret_cast<const void *>(&k_score_group<256, false>)});
            if (narrow) TGBM_SCORE_GROUP(256, true);
            else TGBM_SCORE_GROUP(256, false);
        }
#undef TGBM_SCORE_GROUP
        return true;
    }
    if (!rows_fit) return false;
    const size_t fit = (64 * 1024 - dense_bytes) / tree_bytes;  // (>= 1)
    const int tps = (int)std::max<size_t>(1, std::min<size_t>(te != nullptr && atoi(te) == 1 ? 1 : 2, fit));
    const size_t lds = dense_bytes + (size_t)tps * tree_bytes;
    // Classes are shared out as well where the rows alone make fewer workgroups than twice the chip's (each spreads
    // its rows' keys again): 200 k x 28, 5 x 40 trees, in four launches side by side with the upload instead of one behind it.
    const int row_groups = (rows.n + B - 1) / B, parts = std::min(m.n_class, (2 * kScoreChip + row_groups - 1) / row_groups);
    const int classes = (m.n_class + parts - 1) / parts;
    const dim3 g((unsigned)row_groups, (unsigned)((m.n_class + classes - 1) / classes));
    const int per_thread = (tps * m.n_nodes + B - 1) / B;  // records of a stage
#define TGBM_SCORE_ROWS(BLK, ILP, FETCH, NN) \
    k_score_rows<BLK, ILP, FETCH, NN><<<g, BLK, lds, s>>>(rows, m, lr, base_score, out, out_stride, tps, fill, classes)
#define TGBM_SCORE_FETCH(BLK, ILP, NN)                          \
    if (per_thread <= 2) TGBM_SCORE_ROWS(BLK, ILP, 2, NN);      \
    else if (per_thread <= 4) TGBM_SCORE_ROWS(BLK, ILP, 4, NN); \
    else TGBM_SCORE_ROWS(BLK, ILP, 8, NN)
#define TGBM_SCORE_ILP(BLK, NN)                  \
    if (tps >= 2) { TGBM_SCORE_FETCH(BLK, 2, NN); } \
    else { TGBM_SCORE_FETCH(BLK, 1, NN); }
    if (B == 256) {
        if (narrow) { TGBM_SCORE_ILP(256, true) }
        else { TGBM_SCORE_ILP(256, false) }
    } else {
        if (narrow) { TGBM_SCORE_ILP(128, true) }
        else { TGBM_SCORE_ILP(128, false) }
    }
#undef TGBM_SCORE_ILP
#undef TGBM_SCORE_FETCH
#undef TGBM_SCORE_ROWS
    return true;
}

void launch_predict_transform(hipStream_t s, int kind, int n, int num_class, const float *label, float *y) {
    if (n == 0 || kind == 0) return;
    int grid = (n + kBlock - 1) / kBlock;
    if (grid > 4096) grid = 4096;
    k_predict_transform<<<grid, kBlock, 0, s>>>(kind, n, num_class, label, y);
}

}  // namespace tgbm
