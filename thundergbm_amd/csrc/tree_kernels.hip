// Tree-building kernels for gfx950 (wave64): gradients, LDS-privatised histograms, merge + sibling
// subtraction, wavefront segmented-scan split finding, ballot/popcount row partition, pruning and the
// in-training prediction update. Every stage of a level is one launch over all nodes of the level;
// work lists are planned on the device so the host never waits inside a tree.
#include <algorithm>
#include <type_traits>

#include "device_api.h"
#include "kernel_common.h"
#include "tree_common.h"

namespace tgbm {
namespace {

// Largest p in [0, n) with begin[p] <= item (begin is non-decreasing, begin[0] <= item < begin[n]).
__device__ int find_owner(const int *begin, int n, int item) {
    int lo = 0, hi = n;
    while (hi - lo > 1) {
        int mid = (lo + hi) >> 1;
        if (begin[mid] <= item)
            lo = mid;
        else
            hi = mid;
    }
    return lo;
}

// ------------------------------------------------------------------------------------ fills
__global__ void k_fill_f32(float *p, float v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}
__global__ void k_fill_u32(unsigned *p, unsigned v, size_t n) {
    for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) p[i] = v;
}

// -------------------------------------------------------------------------------- gradients
// Squared / logistic: include/thundergbm/objective/regression_obj.h:130-154 of the reference.
__device__ __forceinline__ GHPair pointwise_gradient(int objective, float yi, float p) {
    GHPair o;
    if (objective == OBJ_SQUARE) {
        o.g = p - yi;
        o.h = 1.f;
    } else {
        float s = 1.f / (1.f + expf(-p));
        o.g = s - yi;
        o.h = fmaxf(s * (1.f - s), 1e-16f);
    }
    return o;
}

__global__ void k_gradient_pointwise(int objective, int n, const float *__restrict__ y, const float *__restrict__ yp,
                                     GHPair *__restrict__ gh) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        gh[i] = pointwise_gradient(objective, y[i], yp[i]);
}

// The gradient pair of a row as one 32-bit word that rides in the spare bytes of the row's bin-matrix record
// (DenseBins::gh_lane), so that a histogram work item that gathers a row gets its pair with the same memory request
// instead of a second one. Whatever computes a round's gradients also leaves the words in an array of their own
// (launch_gh_words, k_tree_end); the root level's histogram launch, which streams every record anyway, reads them
// there and writes the records back with the word in place - whole records, so that memory sees full-sector writes
// (4 bytes of every 32 written by themselves cost a read-modify-write per sector: 90 us per tree on 10 M rows). Squared loss: the gradient itself (the hessian is 1). Logistic loss with 0/1 labels: the
// sigmoid s (never negative) with the label in the sign bit; pair_from_word (kernel_common.h) repeats pointwise_gradient's operations on
// s, so both give the same bits.
__device__ __forceinline__ unsigned word_from_row(int objective, float yi, float p) {
    if (objective == OBJ_SQUARE) return __float_as_uint(p - yi);
    const float s = 1.f / (1.f + expf(-p));
    return __float_as_uint(s) | (yi != 0.f ? 0x80000000u : 0u);
}

__global__ void k_gh_words(int objective, int n, const float *__restrict__ y, const float *__restrict__ yp,
                           unsigned *__restrict__ words) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
        words[i] = word_from_row(objective, y[i], yp[i]);
}

// Softmax: src/thundergbm/objective/multiclass_obj.cu:6-35 (class-major predictions and gradients,
// hessian 2p(1-p)).
__global__ void k_gradient_softmax(int n, int K, const float *__restrict__ y, const float *__restrict__ yp,
                                   GHPair *__restrict__ gh) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
        float mx = yp[i];
        for (int k = 1; k < K; ++k) mx = fmaxf(mx, yp[(size_t)k * n + i]);
        float sum = 0;
        for (int k = 0; k < K; ++k) sum += expf(yp[(size_t)k * n + i] - mx);
        float yi = y[i];
        for (int k = 0; k < K; ++k) {
            float p = expf(yp[(size_t)k * n + i] - mx) / sum;
            GHPair o;
            o.g = (k == yi) ? (p - 1.f) : p;
            o.h = fmaxf(2.f * p * (1.f - p), 1e-16f);
            gh[(size_t)k * n + i] = o;
        }
    }
}

// A wavefront per word of the flags.
__global__ __launch_bounds__(kBlock) void k_column_flags(ColumnFlags in, int count, uint8_t *__restrict__ flags) {
    const int word = __builtin_amdgcn_readfirstlane((int)blockIdx.x * kWaves + wave_id());
    if (word >= kColumnFlagWords) return;
    const int f = word * 64 + lane_id();
    if (f < count) flags[f] = (uint8_t)(in.bits[word] >> lane_id() & 1ull);
}

// Bagging, RowSampler::do_bagging (src/thundergbm/row_sampler.cu:9-38): entry i of the gradient array draws
// idx_i from thrust::default_random_engine(seed) after discard(i) through
// thrust::uniform_int_distribution<int>(0, N - 1); every gradient pair is multiplied by the number of draws
// that hit its index. thrust's default engine is minstd_rand (x <- 48271 x mod 2^31 - 1, a seed of 0 mod m
// becomes 1), its integer distribution maps the engine's output u in [1, m - 1] to
// int((u - 1) / (m - 1) * N) in double precision. The i + 1 steps of the engine are one modular power.
__global__ void k_bagging_draw(int N, unsigned seed, int *__restrict__ count) {
    constexpr unsigned long long M = 2147483647ull, A = 48271ull;
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        unsigned long long x = seed % M;
        if (x == 0) x = 1;
        unsigned long long base = A, e = (unsigned long long)i + 1ull;  // discard(i), then one draw
        while (e) {
            if (e & 1ull) x = x * base % M;
            base = base * base % M;
            e >>= 1;
        }
        double r = (double)(unsigned)(x - 1ull);
        r /= 1.0 + (double)(unsigned)(M - 2ull);  // 1 + (max - min) with min = 1, max = m - 1
        const double lo = 0.0, hi = (double)(N - 1) + 1.0;
        const int idx = (int)(r * (hi - lo) + lo);
        atomicAdd(count + idx, 1);
    }
}

// perm (may be null): original row of every physical position; the draw counts belong to original rows
__global__ void k_bagging_apply(int N, int *__restrict__ count, GHPair *__restrict__ gh, const int *__restrict__ perm,
                                int n_rows) {
    for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < N; i += gridDim.x * blockDim.x) {
        // entry i = (plane, position): the plane (class) stays, the position maps to its original row
        const int src = perm != nullptr ? (i / n_rows) * n_rows + perm[i % n_rows] : i;
        const int c = count[src];
        count[src] = 0;  // ready for the next round (perm is a bijection: every counter is cleared once)
        GHPair v = gh[i];
        v.g = v.g * c;
        v.h = v.h * c;
        gh[i] = v;
    }
}

// Row-blocked reductions: workgroup b owns rows [b * kRowBlock, (b + 1) * kRowBlock), thread t adds its
// rows t, t + threads, ... in that order, then lanes, then wavefronts. The kernels that produce metric partials follow
// this order with as many threads (end_wide), so fused and separate passes give the same bits.
struct RowStats {
    float g = 0, h = 0, gm = 0, hm = 0, hf = 0;
    __device__ __forceinline__ void add(GHPair v) {
        g += v.g;
        h += v.h;
        gm = fmaxf(gm, fabsf(v.g));
        hm = fmaxf(hm, v.h);
        hf = fmaxf(hf, fabsf(v.h - rintf(v.h)));
    }
};

// lds: 5 NW floats (NW wavefronts per workgroup); every thread of the block must call
template <int NW>
__device__ void store_block_stats(RowStats r, float *lds, GradStats *out) {
    float *sg = lds, *sh = lds + NW, *mg = lds + 2 * NW, *mh = lds + 3 * NW, *fh = lds + 4 * NW;
    float g = wave_sum_f(r.g), h = wave_sum_f(r.h), gm = r.gm, hm = r.hm, hf = r.hf;
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        gm = fmaxf(gm, __shfl_xor(gm, d));
        hm = fmaxf(hm, __shfl_xor(hm, d));
        hf = fmaxf(hf, __shfl_xor(hf, d));
    }
    if (lane_id() == 0) {
        sg[wave_id()] = g;
        sh[wave_id()] = h;
        mg[wave_id()] = gm;
        mh[wave_id()] = hm;
        fh[wave_id()] = hf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        GradStats o{0, 0, 0, 0, 0};
        for (int i = 0; i < NW; ++i) {
            o.g += sg[i];
            o.h += sh[i];
            o.gmax = fmaxf(o.gmax, mg[i]);
            o.hmax = fmaxf(o.hmax, mh[i]);
            o.hfrac = fmaxf(o.hfrac, fh[i]);
        }
        *out = o;
    }
}

// lds: NW doubles
template <int NW>
__device__ void store_block_sum_d(double acc, double *lds, double *out) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d);
    if (lane_id() == 0) lds[wave_id()] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < NW; ++i) t += lds[i];
        *out = t;
    }
}

// Block sums of (g,h) and block maxima of |g|, h for one tree.
// Class trees of a round: blockIdx.z selects the class (gradients and outputs are class-major).
__global__ __launch_bounds__(kBlock) void k_sum_gh(int n, const GHPair *__restrict__ gh, GradStats *__restrict__ out) {
    __shared__ float lds[5 * kWaves];
    gh += (size_t)blockIdx.z * n;
    out += (size_t)blockIdx.z * gridDim.x;
    const int r0 = blockIdx.x * kRowBlock, r1 = min(n, r0 + kRowBlock);
    RowStats st;
    for (int i = r0 + threadIdx.x; i < r1; i += kBlock) st.add(gh[i]);
    store_block_stats<kWaves>(st, lds, out + blockIdx.x);
}

// Largest power of two s with rows * (vmax * s + 0.5) < limit; 1 when vmax is 0 or not finite.
__device__ float pow2_scale(float vmax, int rows, float limit) {
    if (!(vmax > 0.f) || !(vmax < INFINITY)) return 1.f;
    float bound = (limit / (float)rows - 0.5f) / vmax;
    if (!(bound < 1e18f)) bound = 1e18f;  // tiny gradients: keep the scale and its inverse well inside float range
    int e;
    frexpf(bound, &e);             // bound = m * 2^e, m in [0.5, 1)
    return ldexpf(1.f, e - 1);     // 2^(e-1) <= bound
}

// ------------------------------------------------------------------------------- tree init
// The tree's scales, from the largest |g| and h of its rows and whether every h is an integer (GradStats): they keep the 64-bit
// sums over all n rows below 2^62; a dense work item coarsens them by its own power of two so that its packed LDS fields hold
// the rows between two drains (item_shift).
__device__ __forceinline__ QuantCtl plan_quant(const TreeBuffers &tb, float gm, float hm, float hf) {
    QuantCtl q;
    // (the sparse layout's kernels round with round_to_ll, good below 2^51: its scales are those of at least
    // 4096 rows, which keeps every row's integers below 2^50)
    const int scale_rows = tb.sparse ? max(tb.n, 4096) : tb.n;
    q.scale_g = pow2_scale(gm, scale_rows, 4.6e18f);
    q.scale_h = pow2_scale(hm, scale_rows, 4.6e18f);
    q.h_bits = 32;
    q.h_integer = 0;
    // every hessian a non-negative integer (squared loss; bagging multiplies by draw counts): the hessian field
    // takes the bits that kHistFlushRowsInt such rows need, the gradient field the rest
    q.flush_rows = kHistFlushRows;
    const float hrows = hm * (float)kHistFlushRowsInt;
    if (!tb.sparse && hf == 0.f && hm >= 1.f && hrows < 4.0e9f) {
        q.h_integer = 1;
        q.h_bits = ilogbf(hrows) + 1;
        q.scale_h = 1.f;
        q.flush_rows = kHistFlushRowsInt;
    }
    q.inv_g = 1.f / q.scale_g;
    q.inv_h = 1.f / q.scale_h;
    q.gq_max = gm * q.scale_g;
    q.hq_max = hm * q.scale_h;
    return q;
}

// Rows per histogram work item of the root.
__device__ __forceinline__ int root_chunk(const TreeBuffers &tb) {
    const int chunk = (tb.n + tb.target_hitems - 1) / tb.target_hitems;
    return max(kHistMinChunk, (chunk + 255) / 256 * 256);
}

// Node array initialisation of the reference's Tree::init2 (src/thundergbm/tree.cu:8-39), root sum
// from the block partials, root segment and the histogram plan of level 0.
// What the previous tree has left to do rides along: its finished nodes go into the model before they are reset, and one more
// workgroup adds up the round's metric (two launches of 4 to 5 us per tree otherwise).
// The first workgroup (part 0) does all but the metric; trees of more than kInitNodes nodes are shared out over `parts` of them
// (with one, the nodes of depth 14 took 85 us). In the dense layout the root level's histogram launch has these workgroups
// (k_hist_dense): a launch of 4.7 us less, 10 k x 8 0.126 -> 0.122 ms a tree, 500 k x 28 0.256 -> 0.252. (10 M x 28: the launch takes 152 us
// instead of 148, what comes before it 6 instead of 13.)
constexpr int kInitNodes = 1024;
int init_parts(const TreeBuffers &tb) { return (tb.n_nodes + kInitNodes - 1) / kInitNodes; }
__device__ void metric_final(int kind, int n, int n_blocks, const double *__restrict__ in, float *__restrict__ out);
// (the workgroup's first kBlock threads do it; all of its threads call, there are barriers inside)
__device__ void tree_init_part(const TreeBuffers &tb, float lambda, const TreeLeftovers &left, int part, int parts) {
    if (part == parts) {
        if (blockIdx.z == 0) metric_final(left.metric_kind, tb.n, left.metric_blocks, left.metric_partial, left.metric_out);
        return;
    }
    __shared__ float sg[kWaves], sh[kWaves], mg[kWaves], mh[kWaves], fh[kWaves];
    const bool on = threadIdx.x < kBlock;
    if (left.small && part == 0 && on) {  // every row starts in the root
        for (int i = threadIdx.x; i < tb.n; i += kBlock) tb.nid[i] = 0;
    }
    if ((left.small || left.run > 0) && part == 0 && on)
        for (int i = 1 + threadIdx.x; i < tb.depth; i += kBlock) tb.ctl[i] = LevelCtl{left.run, 0, 0, 0};
    const GradStats *__restrict__ block_sums = tb.root_partial;
    const int nn = tb.n_nodes;
    for (int i = part * kBlock + threadIdx.x; on && i < nn; i += parts * kBlock) {
        TreeNode nd;
        nd.final_id = i;
        nd.parent_index = i == 0 ? -1 : (i - 1) / 2;
        nd.gain = 0;
        nd.base_weight = 0;
        nd.split_feature_id = -1;
        nd.split_value = 0;
        nd.split_bid = 0;
        nd.default_right = false;
        nd.is_valid = false;
        nd.is_pruned = false;
        nd.sum_gh_pair = GHPair{0, 0};
        if (i < nn / 2) {
            nd.is_leaf = false;
            nd.lch_index = 2 * i + 1;
            nd.rch_index = 2 * i + 2;
        } else {
            nd.is_leaf = true;
            nd.lch_index = -1;
            nd.rch_index = -1;
        }
        // zero the padding bytes too: nodes are written raw into model files
        unsigned *raw = reinterpret_cast<unsigned *>(&nd);
        raw[9] &= 0x000000ffu;  // bytes 37..39 are padding (byte 36 = is_pruned)
        if (left.model != nullptr) {
            const int4 *from = reinterpret_cast<const int4 *>(tb.nodes + i);
            int4 *to = reinterpret_cast<int4 *>(left.model + (size_t)blockIdx.z * nn + i);
            const int4 v0 = from[0], v1 = from[1], v2 = from[2];
            to[0] = v0;
            to[1] = v1;
            to[2] = v2;
        }
        tb.nodes[i] = nd;
        tb.seg[i] = make_int2(0, 0);
        if (tb.node_rows != nullptr) tb.node_rows[i] = i == 0 ? tb.n : 0;
    }
    if (part != 0) return;
    float g = 0, h = 0, gm = 0, hm = 0, hf = 0;
    for (int i = threadIdx.x; on && i < tb.n_grad_blocks; i += kBlock) {
        g += block_sums[i].g;
        h += block_sums[i].h;
        gm = fmaxf(gm, block_sums[i].gmax);
        hm = fmaxf(hm, block_sums[i].hmax);
        hf = fmaxf(hf, block_sums[i].hfrac);
    }
    g = wave_sum_f(g);
    h = wave_sum_f(h);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
        gm = fmaxf(gm, __shfl_xor(gm, d));
        hm = fmaxf(hm, __shfl_xor(hm, d));
        hf = fmaxf(hf, __shfl_xor(hf, d));
    }
    if (on && lane_id() == 0) {
        sg[wave_id()] = g;
        sh[wave_id()] = h;
        mg[wave_id()] = gm;
        mh[wave_id()] = hm;
        fh[wave_id()] = hf;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        GHPair s{0, 0};
        gm = 0;
        hm = 0;
        hf = 0;
        for (int i = 0; i < kWaves; ++i) {
            s.g += sg[i];
            s.h += sh[i];
            gm = fmaxf(gm, mg[i]);
            hm = fmaxf(hm, mh[i]);
            hf = fmaxf(hf, fh[i]);
        }
        TreeNode &root = tb.nodes[0];
        root.sum_gh_pair = s;
        root.is_valid = true;
        root.base_weight = -s.g / (s.h + lambda);
        tb.seg[0] = make_int2(0, tb.n);
        const int chunk = root_chunk(tb), items = (tb.n + chunk - 1) / chunk;
        tb.hpair_begin[0] = 0;
        tb.hpair_begin[1] = items;
        tb.hpair_built[0] = 0;
        LevelCtl c;
        c.hchunk = chunk;
        c.n_hitems = items;
        c.n_pitems = (tb.n + kPartChunk - 1) / kPartChunk;  // the root's partition items (used if it splits)
        c.rows_built = tb.n;
        tb.ctl[0] = c;
        tb.pbegin(0)[0] = 0;
        tb.pbegin(0)[1] = c.n_pitems;
        tb.ctl[tb.depth] = LevelCtl{0, 0, 0, 0};  // the last level plans no further one
        *tb.quant = plan_quant(tb, gm, hm, hf);
    }
}
__global__ __launch_bounds__(kBlock) void k_tree_init(TreeBuffers tb_all, float lambda, TreeLeftovers left, int parts) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    tree_init_part(tb, lambda, left, blockIdx.x, parts);
}

// The tree's scales by every thread of a BLK-wide workgroup for itself; lds: 3 floats per wavefront. One barrier.
template <int BLK>
__device__ __forceinline__ QuantCtl quant_of_stats(const TreeBuffers &tb, float *lds) {
    constexpr int NW = BLK / 64;
    const GradStats *__restrict__ stats = tb.root_partial;
    float gm = 0, hm = 0, hf = 0;
    for (int i = threadIdx.x; i < tb.n_grad_blocks; i += BLK) {
        gm = fmaxf(gm, stats[i].gmax);
        hm = fmaxf(hm, stats[i].hmax);
        hf = fmaxf(hf, stats[i].hfrac);
    }
    gm = wave_max_f(gm);
    hm = wave_max_f(hm);
    hf = wave_max_f(hf);
    if (lane_id() == 0) {
        lds[wave_id()] = gm;
        lds[NW + wave_id()] = hm;
        lds[2 * NW + wave_id()] = hf;
    }
    __syncthreads();
    const int w = lane_id() % NW;
    return plan_quant(tb, wave_max_f(lds[w]), wave_max_f(lds[NW + w]), wave_max_f(lds[2 * NW + w]));
}

// ------------------------------------------------------------------------------ exact root sums
// k_tree_init sets the root's sums from a float reduction over the rows, whose last bits depend on the physical
// order of the rows; every later quantity of a tree (child sums, weights, gains, predictions, the next gradients)
// derives from it. These kernels replace it by the exact fixed-point total - the same integers in any order - so
// that a tree does not depend on the row order at all.
__device__ __forceinline__ GHPair root_sums(const TreeBuffers &tb, long long G, long long H) {
    return {(float)((double)G * (double)tb.quant->inv_g), (float)((double)H * (double)tb.quant->inv_h)};
}
__device__ __forceinline__ void set_root_sums(const TreeBuffers &tb, GHPair s, float lambda) {
    TreeNode &root = tb.nodes[0];
    root.sum_gh_pair = s;
    root.base_weight = -s.g / (s.h + lambda);
}

// From the root histogram: the bins of a feature that is stored in every row add up to the root. One workgroup.
__global__ __launch_bounds__(kBlock) void k_root_sum_bins(TreeBuffers tb_all, float lambda) {
    __shared__ long long s_g[kWaves], s_h[kWaves];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const longlong2 *__restrict__ h = tb.hist(0);
    const int b0 = tb.cut_row_ptr[tb.complete_feature], b1 = tb.cut_row_ptr[tb.complete_feature + 1];
    long long g = 0, hh = 0;
    for (int b = b0 + threadIdx.x; b < b1; b += kBlock) {
        const longlong2 v = h[b];
        g += v.x;
        hh += v.y;
    }
    g = wave_sum_ll(g);
    hh = wave_sum_ll(hh);
    if (lane_id() == 0) {
        s_g[wave_id()] = g;
        s_h[wave_id()] = hh;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int i = 1; i < kWaves; ++i) {
            g += s_g[i];
            hh += s_h[i];
        }
        set_root_sums(tb, root_sums(tb, g, hh), lambda);
    }
}

// From the gradients (no feature is stored in every row): every row's pair rounded at the tree's scales, a pair of 64-bit sums
// per part of the rows into root_total[2 part], [2 part + 1], which whoever needs the root's sums adds up: in the dense layout
// by the root level's histogram launch and by every workgroup of its split search (two launches of 4 to 9 us a tree less:
// 500 k x 54 with 8 classes 0.515 -> 0.503 ms a round). (A ticket that lets the last workgroup finish the job needs a device-scope
// fence, which writes a whole L2 back on this chip: 288 us per round of 8 class trees.)
template <int BLK>
__device__ __forceinline__ void root_sum_rows(const TreeBuffers &tb, const QuantCtl &quant, const GHPair *__restrict__ gh, int begin, int end,
                                              int part) {
    __shared__ long long s_g[BLK / 64], s_h[BLK / 64];
    const float scale_g = quant.scale_g, scale_h = quant.scale_h;
    long long g = 0, hh = 0;
    for (int i = begin + (int)threadIdx.x; i < end; i += BLK) {
        const GHPair v = gh[i];
        g += __float2ll_rn(v.g * scale_g);
        hh += __float2ll_rn(fmaxf(v.h, 0.f) * scale_h);
    }
    g = wave_sum_ll(g);
    hh = wave_sum_ll(hh);
    if (lane_id() == 0) {
        s_g[wave_id()] = g;
        s_h[wave_id()] = hh;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int i = 1; i < BLK / 64; ++i) {
        g += s_g[i];
        hh += s_h[i];
    }
    tb.root_total[2 * part] = g;
    tb.root_total[2 * part + 1] = hh;
}

// By one wavefront, the same in all of its lanes.
__device__ __forceinline__ GHPair root_sums_of_rows(const TreeBuffers &tb, int parts) {
    const longlong2 *__restrict__ from = reinterpret_cast<const longlong2 *>(tb.root_total);
    longlong2 v[kRootParts / 64];
#pragma unroll
    for (int k = 0; k < kRootParts / 64; ++k) v[k] = from[min(k * 64 + lane_id(), parts - 1)];
    long long g = 0, h = 0;
#pragma unroll
    for (int k = 0; k < kRootParts / 64; ++k) {
        g += k * 64 + lane_id() < parts ? v[k].x : 0;
        h += k * 64 + lane_id() < parts ? v[k].y : 0;
    }
    return root_sums(tb, wave_sum_ll(g), wave_sum_ll(h));
}

__global__ __launch_bounds__(kBlock) void k_root_sum_rows(TreeBuffers tb_all, const GHPair *__restrict__ gh) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int per = (tb.n + (int)gridDim.x - 1) / (int)gridDim.x, begin = min(tb.n, (int)blockIdx.x * per);
    root_sum_rows<kBlock>(tb, *tb.quant, gh + (size_t)blockIdx.z * tb.n, begin, min(tb.n, begin + per), blockIdx.x);
}

__global__ __launch_bounds__(64) void k_root_sum_final(TreeBuffers tb_all, int parts, float lambda) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const GHPair s = root_sums_of_rows(tb, parts);
    if (threadIdx.x == 0) set_root_sums(tb, s, lambda);
}

// ------------------------------------------------------------------------- dense histogram
// One workgroup = one work item (a run of rows of one node) x one feature block. The block's
// histogram lives in LDS as one 64-bit integer per bin holding the fixed-point gradient sum in the
// high and the hessian sum in the low field (QuantCtl::h_bits wide); a row contributes with a single
// ds_add_u64 per feature (float LDS atomics run at ~0.3 lanes/clk/CU on gfx950, 64-bit integer ones at ~5).
// The fields are safe for the rows added between two drains (at most kHistFlushRows; fewer in a node with fewer
// rows, whose items therefore count finer: item_shift), so after at most that many rows every thread drains the
// bins it owns into 64-bit register accumulators and clears them; at the end the registers go to the item's slot
// of `partial`, at the item's scale (k_hist_merge shifts them to the tree's).
// LPR consecutive lanes cover one row (one dword = four bin bytes per lane, or two 16-bit bins with BIN16), so a
// wavefront load instruction reads 256 contiguous bytes and the 64 atomics of one step spread over many features.
// (Packing each row's gradient pair next to its bins so that a gathered row costs one 128-byte line
// instead of two was measured: it halves the fetched bytes below the root, but the per-tree refresh of
// the pairs costs what the gathers save.)
// GHW: the rows' gradient pairs come from 32-bit words (word_from_row). Below the root the word sits in the last
// dword of the row's record, which the row's last lane has loaded with the bins anyway: no second gather per row. The
// root launch (DIRECT) reads the words from their own array and puts them there, storing every record back.
struct HistRoot {  // DIRECT: what the root level's launch does besides
    int init_groups = 0, init_parts = 0;  // the tree's set-up by so many workgroups more (tree_init_part)
    bool sum_rows = false;                // the sums of the items' rows into root_total
    float lambda = 0;
    TreeLeftovers left;
};
template <int LPR, bool DIRECT, int BLK, int SLOTS, bool BIN16, bool GHW = false>
__global__ __launch_bounds__(BLK) __attribute__((amdgpu_waves_per_eu(SLOTS <= 8 ? 8 : 4)))  // two 1024-thread groups per CU
void k_hist_dense(TreeBuffers tb_all, DenseBins bins, const GHPair *__restrict__ gh, int level, int n_pairs,
                  std::conditional_t<DIRECT, HistRoot, int> root) {
    extern __shared__ unsigned long long lds[];
    __shared__ int s_shift[2];  // the item's scale shifts (gradient, hessian)
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    const int *__restrict__ ridx = tb.list(level);
    const int *__restrict__ blk_bin_begin = tb.blk_bin_begin;
    const int *__restrict__ feat_lds_off = tb.feat_lds_off;
    longlong2 *__restrict__ partial = tb.partial;
    const int n_bins = tb.n_bins;
    // (the feature blocks of an item are neighbours in the launch order: the item's row list and gradient pairs, which
    // every block reads again, are then fetched while they still sit in an L2 - with the items of a block as
    // neighbours, every block of 500 k x 2000 data fetched them from HBM again: 2.72 -> 2.29 ms per tree)
    int item = blockIdx.y;
    const int fb = blockIdx.x;
    QuantCtl quant;
    if constexpr (DIRECT) {
        if (item < root.init_groups) {  // the tree's set-up, by the first block's workgroups
            if (fb == 0) tree_init_part(tb, root.lambda, root.left, item, root.init_parts);
            return;
        }
        item -= root.init_groups;
    }
    // The item's node and rows: the same few look-ups in every lane (uniform addresses: scalar loads) or in every
    // wavefront, so that the first row loads can be issued before the barrier that publishes the LDS histogram's clearing.
    int node, hchunk;
    int2 sg;
    int first_item;  // of the node
    int item0 = 0;
    if constexpr (!DIRECT) {
        const HistPlan plan = plan_hist_item(tb, n_pairs, item, fb == 0 && item == 0 && threadIdx.x < 64, level);
        if (plan.pair < 0) return;
        node = plan.built;
        sg = plan.seg;
        hchunk = plan.chunk;
        first_item = plan.first_item;
        item0 = plan.item0;
    } else {
        node = 0;
        sg = make_int2(0, tb.n);
        hchunk = root_chunk(tb);
        first_item = 0;
        if (item * hchunk >= tb.n) return;
        if (root.init_groups > 0) {
            __shared__ float s_stats[3 * BLK / 64];
            quant = quant_of_stats<BLK>(tb, s_stats);
        } else {
            quant = *tb.quant;
        }
    }
    const int bin0 = blk_bin_begin[fb];
    const int nb = blk_bin_begin[fb + 1] - bin0;
    if (nb == 0 && fb != 0) return;  // (the first block, with bins or without, stores what an item has once: its scales, its rows' sums)
    if constexpr (!DIRECT) quant = *tb.quant;
    const int h_bits = quant.h_bits;
    const int flush_rows = quant.flush_rows;
    const int gh_objective = bins.gh_objective;
    const bool word_lane = bins.gh_lane >= 0 && (int)(threadIdx.x % LPR) == bins.gh_lane;
    const int begin = __builtin_amdgcn_readfirstlane(sg.x + (item - first_item) * hchunk);
    const int end = __builtin_amdgcn_readfirstlane(min(sg.y, begin + hchunk));
    const int x_in = node - ((1 << level) - 1);
    if (x_in < tb.lvl_x0 || x_in >= tb.lvl_x1) return;  // not in the batch of nodes this launch serves
    if (threadIdx.x == 0) {
        // (the node's rows, not the item's: what a row adds must not depend on the item it falls into, or the sums
        // would change with the order of the rows)
        const int rows = max(1, min(sg.y - sg.x, quant.flush_rows));
        const int2 shift = make_int2(item_shift(quant.gq_max, rows, 63 - h_bits),
                                     quant.h_integer ? 0 : item_shift(quant.hq_max, rows, h_bits));
        s_shift[0] = shift.x;
        s_shift[1] = shift.y;
        if (fb == 0) tb.hitem_shift[item] = shift;
    }
    // (slots of `partial` count from item0, the first item of the served batch of nodes: 0 unless the arena is capped)
    const unsigned long long h_mask = (1ull << h_bits) - 1ull;  // h_bits <= 32
    constexpr int RPS = BLK / LPR;  // rows per step of the whole block
    // rows per thread and stage: what the registers left over by the drain accumulators hold without spills (64
    // registers per thread with two workgroups per CU)
    constexpr int U = (SLOTS <= 4 || SLOTS == 16) ? 4 : 2;
    static_assert(RPS * U <= kHistFlushRows, "one iteration must not exceed the flush interval");
    const int q = threadIdx.x % LPR;
    const int rsub = threadIdx.x / LPR;
    constexpr int FPL = BIN16 ? 2 : 4;  // features per lane (one dword of the row)
    constexpr int ROWB = LPR * 4;       // bytes per row of the block
    const int *fo = feat_lds_off + fb * (LPR * FPL) + q * FPL;
    const int o0 = fo[0], o1 = fo[1], o2 = BIN16 ? 0 : fo[2], o3 = BIN16 ? 0 : fo[3];
    // (a block is smaller than 4 GiB and has fewer than 2^29 rows - checked when the layout is chosen -, so a lane
    // addresses its dword, its gradient pair and its row id with an unsigned 32-bit offset from a uniform base)
    const uint8_t *blk = bins.data + (size_t)fb * bins.block_stride;
    const char *words = reinterpret_cast<const char *>(bins.gh_words);
    const unsigned qoff = q * 4;
    long long accg[SLOTS], acch[SLOTS];
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) accg[k] = acch[k] = 0;
    int pending = 0;  // rows accumulated in LDS since the last drain (uniform across the block)
    unsigned pk[U], pk_next[U];
    GHPair s[U], s_next[U];
    // Three stages in flight per thread: the row ids of the step after next, the bins and gradient pairs of the next
    // step (gathered through row ids that arrived during the previous iteration), the atomics of this step. All
    // loads are unconditional - positions past the item's end are clamped to its last row and their bins replaced by
    // the sentinel - and each stage's loads are issued back to back, so that no load waits for an unrelated one.
    int r_next[U];
    auto load_ids = [&](int base, int(&r)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int pos = min(base + rsub + u * RPS, end - 1);
            r[u] = DIRECT ? pos : *reinterpret_cast<const int *>(reinterpret_cast<const char *>(ridx) + (unsigned)pos * 4u);
        }
    };
    auto load_rows = [&](const int(&r)[U], unsigned(&opk)[U], GHPair(&os)[U]) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            opk[u] = *reinterpret_cast<const unsigned *>(blk + ((unsigned)r[u] * (unsigned)ROWB + qoff));
            if (!GHW) os[u] = *reinterpret_cast<const GHPair *>(reinterpret_cast<const char *>(gh) + (unsigned)r[u] * 8u);
            if (GHW && DIRECT)  // (the word travels in the pair's first slot)
                os[u].g = __uint_as_float(*reinterpret_cast<const unsigned *>(words + (unsigned)r[u] * 4u));
        }
    };
    constexpr int STEP = RPS * U;
    if (begin < end) {
        load_ids(begin, r_next);
        load_rows(r_next, pk, s);
        if (begin + STEP < end) load_ids(begin + STEP, r_next);
    }
    // the first rows are on their way: clear the histogram meanwhile
    for (int i = threadIdx.x; i < nb; i += BLK) lds[i] = 0ull;
    __syncthreads();
    // the item's scales: powers of two well inside the float range, so the products below are exact
    const float scale_g = ldexpf(quant.scale_g, -__builtin_amdgcn_readfirstlane(s_shift[0]));
    const float scale_h = ldexpf(quant.scale_h, -__builtin_amdgcn_readfirstlane(s_shift[1]));
    for (int base = begin; base < end; base += STEP) {
        // the next step's rows are requested before this step's atomics (and before a drain's
        // barriers), so the memory pipeline stays busy
        if (base + STEP < end) {
            load_rows(r_next, pk_next, s_next);
            if (base + 2 * STEP < end) load_ids(base + 2 * STEP, r_next);
        }
        const int step_rows = min(RPS * U, end - base);
        if (pending + step_rows > flush_rows) {
            __syncthreads();
#pragma unroll
            for (int k = 0; k < SLOTS; ++k) {
                const int i = threadIdx.x + k * BLK;
                if (i < nb) {
                    const unsigned long long t = lds[i];
                    lds[i] = 0ull;
                    const unsigned long long lo = t & h_mask;
                    accg[k] += (long long)(t - lo) >> h_bits;
                    acch[k] += (long long)lo;
                }
            }
            __syncthreads();
            pending = 0;
        }
        pending += step_rows;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            unsigned v = (base + rsub + u * RPS < end) ? pk[u] : 0xffffffffu;  // (a clamped position adds nothing)
            GHPair sv = s[u];
            if constexpr (GHW && DIRECT) {
                const unsigned w = __float_as_uint(s[u].g);
                sv = pair_from_word(gh_objective, w);
                // the record goes back with the word in its last dword (whole records: full-sector writes)
                // (positions past the end write the last row's again, as it is)
                const int pos = min(base + rsub + u * RPS, end - 1);
                *reinterpret_cast<unsigned *>(const_cast<uint8_t *>(blk) + ((unsigned)pos * (unsigned)ROWB + qoff)) = word_lane ? w : pk[u];
            } else if constexpr (GHW) {
                // the row's last lane holds the word: every lane of the row takes it from there
                sv = pair_from_word(gh_objective, last_lane_of_row<LPR>(pk[u]));
            }
            if (word_lane) v = 0xffffffffu;  // (that lane's dword holds no bins, whether the word is used or not)
            add_row<BIN16>(lds, v, sv, scale_g, scale_h, h_bits, o0, o1, o2, o3);
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            pk[u] = pk_next[u];
            if (!GHW || DIRECT) s[u] = s_next[u];
        }
    }
    if constexpr (DIRECT)
        if (root.sum_rows && fb == 0) root_sum_rows<BLK>(tb, quant, gh, begin, end, item);
    __syncthreads();
    if (hchunk <= flush_rows) {
        // an item this short was never drained: its packed LDS words are the complete sums and go out as
        // they are (8 bytes per bin instead of 16; k_hist_merge unpacks them)
        unsigned long long *out = reinterpret_cast<unsigned long long *>(partial) + (size_t)(item - item0) * n_bins + bin0;
        for (int i = threadIdx.x; i < nb; i += BLK) out[i] = lds[i];
        return;
    }
    longlong2 *out = partial + (size_t)(item - item0) * n_bins + bin0;
#pragma unroll
    for (int k = 0; k < SLOTS; ++k) {
        const int i = threadIdx.x + k * BLK;
        if (i < nb) {
            const unsigned long long t = lds[i];
            const unsigned long long lo = t & h_mask;
            out[i] = make_longlong2(accg[k] + ((long long)(t - lo) >> h_bits), acch[k] + (long long)lo);
        }
    }
}

// (Adding the work items' histograms straight into the node's histogram with global 64-bit atomics
// instead of storing and merging them was measured: 0.5 ms per tree slower on the 10M x 28 benchmark.)
// Sum the private histograms of the node that was built from rows (64-bit integers, exact, any
// order gives the same bits) and derive its sibling as parent - built (the reference's subtraction
// trick, hist_tree_builder_single.cu:526-540). A block covers kMergeBins bins of one sibling pair; its
// thread groups stride over the pair's work items and are combined through LDS. Near the root a pair has
// hundreds of items and the level only a few pairs, so narrow blocks (8 bins, 32 groups) are used there:
// four times the workgroups and a quarter of the loads per thread.
template <int kMergeBins>
__global__ __launch_bounds__(kBlock) void k_hist_merge(TreeBuffers tb_all, int level) {
    constexpr int kMergeGroups = kBlock / kMergeBins;
    __shared__ long long s_g[kMergeGroups][kMergeBins], s_h[kMergeGroups][kMergeBins];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const longlong2 *__restrict__ partial = tb.partial;
    longlong2 *__restrict__ cur_q = tb.hist(level);
    const longlong2 *__restrict__ prev_q = tb.hist(level + 1);
    const int *__restrict__ hpair_begin = tb.hpair_begin;
    const int *__restrict__ hpair_built = tb.hpair_built;
    const int n_bins = tb.n_bins;
    const int p = blockIdx.y + tb.hpair_lo(level);
    const int built = hpair_built[p];
    if (built < 0) return;
    const int jl = threadIdx.x % kMergeBins, ig = threadIdx.x / kMergeBins;
    const int j = blockIdx.x * kMergeBins + jl;
    const int ib = hpair_begin[p], ie = hpair_begin[p + 1];
    const int item0 = hpair_begin[tb.hpair_lo(level)];  // `partial` slots count from the served batch's first item
    long long sg = 0, sh = 0;
    if (j < n_bins) {
        // every item counted at its own scale (item_shift): shift its sums to the tree's
        const int2 *__restrict__ shift = tb.hitem_shift;
        if (tb.ctl[level].hchunk <= tb.quant->flush_rows) {  // packed 8-byte partials (see k_hist_dense)
            const unsigned long long *packed = reinterpret_cast<const unsigned long long *>(partial);
            const int h_bits = tb.quant->h_bits;
            const unsigned long long h_mask = (1ull << h_bits) - 1ull;
            for (int it = ib + ig; it < ie; it += kMergeGroups) {
                const unsigned long long t = packed[(size_t)(it - item0) * n_bins + j];
                const int2 s = shift[it];
                const unsigned long long lo = t & h_mask;
                sg += ((long long)(t - lo) >> h_bits) << s.x;
                sh += (long long)lo << s.y;
            }
        } else {
            for (int it = ib + ig; it < ie; it += kMergeGroups) {
                longlong2 v = partial[(size_t)(it - item0) * n_bins + j];
                const int2 s = shift[it];
                sg += v.x << s.x;
                sh += v.y << s.y;
            }
        }
    }
    s_g[ig][jl] = sg;
    s_h[ig][jl] = sh;
    __syncthreads();
    if (ig != 0 || j >= n_bins) return;
#pragma unroll
    for (int k = 1; k < kMergeGroups; ++k) {
        sg += s_g[k][jl];
        sh += s_h[k][jl];
    }
    const int off = (1 << level) - 1;
    cur_q[(size_t)(built - off) * n_bins + j] = make_longlong2(sg, sh);
    if (level > 0 && !tb.singles(level)) {
        const int sib = (built & 1) ? built + 1 : built - 1;
        const longlong2 par = prev_q[(size_t)p * n_bins + j];
        cur_q[(size_t)(sib - off) * n_bins + j] = make_longlong2(par.x - sg, par.y - sh);
    }
}

__global__ __launch_bounds__(kBlock) void k_count_bytes(const uint8_t *__restrict__ v, size_t n, uint8_t value,
                                                       unsigned long long *__restrict__ out) {
    unsigned long long c = 0;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) c += v[i] == value;
    c = (unsigned long long)wave_sum_ll((long long)c);
    if (lane_id() == 0 && c) atomicAdd(out, c);
}

__global__ __launch_bounds__(kBlock) void k_count_u16(const uint16_t *__restrict__ v, size_t n, uint16_t value,
                                                     unsigned long long *__restrict__ out) {
    unsigned long long c = 0;
    for (size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x; i < n; i += (size_t)gridDim.x * kBlock) c += v[i] == value;
    c = (unsigned long long)wave_sum_ll((long long)c);
    if (lane_id() == 0 && c) atomicAdd(out, c);
}

// --------------------------------------------------------------------------- sparse histogram
// CSR rows of global bin ids: the histogram is too large for LDS (one slot per cut point of every
// feature), so every stored value adds its row's fixed-point gradient pair to the node's histogram
// in HBM with two 64-bit integer atomics (exact and order-independent, unlike the float atomics of
// hist_tree_builder_single.cu:203-216 / :485-505). One wavefront walks one row at a time.
__global__ __launch_bounds__(kBlock) void k_hist_zero_built(TreeBuffers tb_all, int level) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    longlong2 *__restrict__ cur_q = tb.hist(level);
    const int n_bins = tb.n_bins;
    const int built = tb.hpair_built[blockIdx.y + tb.hpair_lo(level)];
    if (built < 0) return;
    const int off = (1 << level) - 1;
    longlong2 *h = cur_q + (size_t)(built - off) * n_bins;
    for (int j = blockIdx.x * kBlock + threadIdx.x; j < n_bins; j += gridDim.x * kBlock) h[j] = make_longlong2(0, 0);
}

template <bool DIRECT>
__global__ __launch_bounds__(kBlock) void k_hist_csr(TreeBuffers tb_all, CsrBins bins, const GHPair *__restrict__ gh,
                                                    int n_pairs, int level) {
    __shared__ int s_info[3];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    const int *__restrict__ ridx = tb.list(level);
    longlong2 *__restrict__ cur_q = tb.hist(level);
    const LevelCtl c = tb.ctl[level];
    const int item = blockIdx.x;
    if (item >= c.n_hitems) return;
    if (threadIdx.x == 0) {
        int p = find_owner(tb.hpair_begin, n_pairs, item);
        int node = tb.hpair_built[p];
        int2 sg = tb.seg[node];
        int b = sg.x + (item - tb.hpair_begin[p]) * c.hchunk;
        s_info[0] = b;
        s_info[1] = min(sg.y, b + c.hchunk);
        s_info[2] = node - ((1 << level) - 1);
        if (s_info[2] < tb.lvl_x0 || s_info[2] >= tb.lvl_x1) s_info[1] = b;  // not in the served batch: no rows
    }
    __syncthreads();
    const int begin = s_info[0], end = s_info[1];
    unsigned long long *h = reinterpret_cast<unsigned long long *>(cur_q + (size_t)s_info[2] * tb.n_bins);
    const float scale_g = tb.quant->scale_g, scale_h = tb.quant->scale_h;
    const int lane = lane_id(), w = wave_id();
    for (int pos = begin + w; pos < end; pos += kWaves) {
        const int r = DIRECT ? pos : ridx[pos];
        const GHPair s = gh[r];
        const long long gq = __float2ll_rn(s.g * scale_g);
        const long long hq = __float2ll_rn(s.h * scale_h);
        const int e0 = bins.row_ptr[r], e1 = bins.row_ptr[r + 1];
        for (int e = e0 + lane; e < e1; e += 64) {
            const int b = bins.bin[e];
            atomicAdd(h + 2 * (size_t)b, (unsigned long long)gq);
            atomicAdd(h + 2 * (size_t)b + 1, (unsigned long long)hq);
        }
    }
}

// The same with the bins of the most frequent features ("head") accumulated in LDS: with a skewed feature
// distribution most stored values hit a few thousand bins, and global atomics on those serialise (the
// root level of a 2M x 100k Zipf matrix spent 10 ms there). Every head slot is a pair of 64-bit sums, so
// no drain is needed; at the end the workgroup adds its non-zero slots to the node's histogram in HBM.
// 1024 threads (16 wavefronts, one row each, the next row's header prefetched), two workgroups per CU.
template <bool DIRECT>
__global__ __launch_bounds__(kHistBlock) __attribute__((amdgpu_waves_per_eu(8)))
void k_hist_csr_head(TreeBuffers tb_all, CsrBins bins, const GHPair *__restrict__ gh, int n_pairs, int level) {
    extern __shared__ unsigned long long lds[];  // [2 * head_bins]: gradient, hessian of every slot
    __shared__ int s_info[3];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    const int *__restrict__ ridx = tb.list(level);
    longlong2 *__restrict__ cur_q = tb.hist(level);
    const LevelCtl c = tb.ctl[level];
    const int item = blockIdx.x;
    if (item >= c.n_hitems) return;
    if (threadIdx.x == 0) {
        int p = find_owner(tb.hpair_begin, n_pairs, item);
        int node = tb.hpair_built[p];
        int2 sg = tb.seg[node];
        int b = sg.x + (item - tb.hpair_begin[p]) * c.hchunk;
        s_info[0] = b;
        s_info[1] = min(sg.y, b + c.hchunk);
        s_info[2] = node - ((1 << level) - 1);
        if (s_info[2] < tb.lvl_x0 || s_info[2] >= tb.lvl_x1) s_info[1] = b;  // not in the served batch: no rows
    }
    for (int i = threadIdx.x; i < 2 * bins.head_bins; i += kHistBlock) lds[i] = 0ull;
    __syncthreads();
    const int begin = s_info[0], end = s_info[1];
    unsigned long long *h = reinterpret_cast<unsigned long long *>(cur_q + (size_t)s_info[2] * tb.n_bins);
    const float scale_g = tb.quant->scale_g, scale_h = tb.quant->scale_h;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    constexpr int NW = kHistBlock / 64;
    int pos = begin + w;
    GHPair s{0, 0};
    int e0 = 0, e1 = 0;
    if (pos < end) {
        const int r = DIRECT ? pos : ridx[pos];
        s = gh[r];
        e0 = bins.row_ptr[r];
        e1 = bins.row_ptr[r + 1];
    }
    while (pos < end) {
        const int npos = pos + NW;
        GHPair ns{0, 0};
        int ne0 = 0, ne1 = 0;
        if (npos < end) {  // requested before this row's atomics
            const int r = DIRECT ? npos : ridx[npos];
            ns = gh[r];
            ne0 = bins.row_ptr[r];
            ne1 = bins.row_ptr[r + 1];
        }
        const unsigned long long gq = (unsigned long long)__float2ll_rn(s.g * scale_g);
        const unsigned long long hq = (unsigned long long)__float2ll_rn(s.h * scale_h);
        for (int e = e0 + lane; e < e1; e += 64) {
            const int word = bins.hist_word[e];
            if (word < 0) {
                const int slot = ~word;
                atomicAdd(lds + 2 * slot, gq);
                atomicAdd(lds + 2 * slot + 1, hq);
            } else {
                atomicAdd(h + 2 * (size_t)word, gq);
                atomicAdd(h + 2 * (size_t)word + 1, hq);
            }
        }
        pos = npos;
        s = ns;
        e0 = ne0;
        e1 = ne1;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < bins.head_bins; i += kHistBlock) {
        const unsigned long long g = lds[2 * i], hh = lds[2 * i + 1];
        if ((g | hh) != 0ull) {
            const size_t b = (size_t)bins.head_bin[i];
            atomicAdd(h + 2 * b, g);
            atomicAdd(h + 2 * b + 1, hh);
        }
    }
}

// Root histogram of the sparse layout from the bin-major copy: every row takes part at the root, so the sum of a
// bin is the sum over a contiguous run of the copy. A wavefront reduces 64 consecutive values by bin (segmented
// scan over sorted keys) and the last lane of every run adds it to the histogram: one pair of atomics per run
// and wavefront, to addresses that ascend with the position, instead of one pair per stored value to random
// lines of a histogram far larger than the caches (4.3 ms -> 1.1 ms at 69 M values, 6.3 M bins). Same integers
// as k_hist_csr, in another order: the histogram is bit-identical.
__global__ __launch_bounds__(kBlock) void k_hist_root_csc(TreeBuffers tb_all, CsrBins bins, const GHPair *__restrict__ gh) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    gh += (size_t)blockIdx.z * tb.n;
    unsigned long long *h = reinterpret_cast<unsigned long long *>(tb.hist(0));
    const float scale_g = tb.quant->scale_g, scale_h = tb.quant->scale_h;
    const int lane = lane_id();
    const long n_tiles = (bins.nnz + 63) / 64;
    for (long tile = (long)blockIdx.x * kWaves + wave_id(); tile < n_tiles; tile += (long)gridDim.x * kWaves) {
        const long e = tile * 64 + lane;
        int b = -1;
        long long gq = 0, hq = 0;
        if (e < bins.nnz) {
            b = bins.csc_bin[e];
            const GHPair s = gh[bins.csc_row[e]];
            gq = __float2ll_rn(s.g * scale_g);
            hq = __float2ll_rn(s.h * scale_h);
        }
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int ob = __shfl_up(b, d);
            const long long og = shfl_up_ll(gq, d), oh = shfl_up_ll(hq, d);
            if (lane >= d && ob == b) {  // sorted keys: equal ends mean one run in between
                gq += og;
                hq += oh;
            }
        }
        const int nb = __shfl_down(b, 1);
        if (b >= 0 && (lane == 63 || nb != b)) {
            atomicAdd(h + 2 * (size_t)b, (unsigned long long)gq);
            atomicAdd(h + 2 * (size_t)b + 1, (unsigned long long)hq);
        }
    }
}

template <bool DIRECT>
__global__ __launch_bounds__(kBlock) void k_part_count_csr(TreeBuffers tb_all, CsrBins bins, int level) {
    __shared__ int lds[kWaves];
    __shared__ int s_x;
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int *__restrict__ ridx = tb.list(level);
    const int item = blockIdx.x;
    if (item >= tb.ctl[level].n_pitems) return;
    const int nl = 1 << level, off = nl - 1;
    if (threadIdx.x == 0) s_x = find_owner(tb.pbegin(level), nl, item);
    __syncthreads();
    const int x_in = s_x;
    const TreeNode &nd = tb.nodes[off + x_in];
    if (!node_splits(nd)) {
        if (threadIdx.x == 0) tb.pitem_nleft[item] = 0;
        return;
    }
    const int2 sg = tb.seg[off + x_in];
    const int pb = sg.x + (item - tb.pbegin(level)[x_in]) * kPartChunk;
    const int pe = min(sg.y, pb + kPartChunk);
    const int f = nd.split_feature_id;
    const int cb = tb.cut_row_ptr[f], ce = tb.cut_row_ptr[f + 1];
    const int sbid = cb + (tb.split_bin != nullptr ? tb.split_bin[off + x_in] : (int)nd.split_bid);
    const bool dr = nd.default_right;
    int nleft = 0;
    unsigned rights = 0;
#pragma unroll
    for (int k = 0; k < kPartChunk / kBlock; ++k) {
        int pos = pb + k * kBlock + threadIdx.x;
        if (pos < pe) {
            int row = DIRECT ? pos : ridx[pos];
            bool right = csr_goes_right(bins, row, cb, ce, sbid, dr);
            rights |= (right ? 1u : 0u) << k;
            nleft += right ? 0 : 1;
        }
    }
    tb.goes_right[(size_t)item * kBlock + threadIdx.x] = (uint8_t)rights;  // (bit k: the thread's k-th row)
    int tot = block_sum(nleft, lds);
    if (threadIdx.x == 0) tb.pitem_nleft[item] = tot;
}

// ------------------------------------------------------------------------ split finding
// Split search. One wavefront scans one pack of whole features (at most 256 bins, 4 consecutive bins
// per lane) of one node with a segmented inclusive prefix sum over the exact 64-bit fixed-point
// histogram: integer sums are associative, so the parallel scan returns bit-for-bit what a
// sequential one would, and candidates separated only by empty bins tie exactly. Per candidate:
// left = sum of the feature's bins below it, missing = node sum - feature total, gain with missing
// values sent right and left (hist_tree_builder_single.cu:257-325 / :614-681 of the reference);
// the wavefront keeps its best candidate: largest |gain|, ties to the smaller bin index (:330-335).
// Where the split search of level 0 takes the node's sums from: a feature stored in every row, whose bins add up to them, or
// what the histogram launch has added up of the rows.
enum RootSums { kNoRoot = 0, kRootOfBins, kRootOfRows };

// SUB (sparse layout, whose histograms are not merged from work-item partials): the node of a pair that
// was not built from rows is derived here as parent - built while it is scanned, and stored for the next
// level, instead of by a separate pass over the (very long) histograms.
// ROOT, the node's sums by every wavefront for itself (RootSums).
template <bool SUB, int ROOT = kNoRoot>
__global__ __launch_bounds__(kBlock) void k_eval_split(TreeBuffers tb_all, int level, float mcw, float lambda,
                                                      bool store_sibling) {
#pragma clang fp contract(off)
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    longlong2 *__restrict__ hist_q = tb.hist(level);
    const int lane = lane_id(), w = wave_id();
    const int pack = blockIdx.x * kWaves + w;
    const int x_in = blockIdx.y + tb.lvl_x0;
    const int x = (1 << level) - 1 + x_in;
    const TreeNode nd = tb.nodes[x];
    const bool active = pack < tb.n_packs && nd.is_valid;
    int b_begin = 0, b_end = 0;
    if (active) {
        b_begin = tb.pack_begin[pack];
        b_end = tb.pack_begin[pack + 1];
    }
    PackMeta pm;
    pm.load(tb, b_begin, b_end);
    GHPair S = nd.sum_gh_pair;
    longlong2 *h = hist_q + (size_t)x_in * tb.n_bins;
    const double inv_g = tb.quant->inv_g, inv_h = tb.quant->inv_h;
    if constexpr (ROOT == kRootOfRows) {
        S = root_sums_of_rows(tb, tb.ctl[0].n_hitems);
        if (pack == 0 && lane == 0) set_root_sums(tb, S, lambda);
    }
    if constexpr (ROOT == kRootOfBins) {
        long long g = 0, hh = 0;
        const int b0 = tb.cut_row_ptr[tb.complete_feature], b1 = tb.cut_row_ptr[tb.complete_feature + 1];
        for (int b = b0 + lane; b < b1; b += 64) {
            const longlong2 v = h[b];
            g += v.x;
            hh += v.y;
        }
        g = wave_sum_ll(g);
        hh = wave_sum_ll(hh);
        S = root_sums(tb, g, hh);
        if (pack == 0 && lane == 0) set_root_sums(tb, S, lambda);
    }
    // SUB: is this node the sibling of the pair's built node?
    const longlong2 *h_par = nullptr, *h_built = nullptr;
    if (SUB && level > 0 && active && !tb.singles(level)) {
        const int built = tb.hpair_built[x_in >> 1];
        if (built >= 0 && built != x) {
            h_par = tb.hist(level + 1) + (size_t)(x_in >> 1) * tb.n_bins;
            h_built = hist_q + (size_t)(built - ((1 << level) - 1)) * tb.n_bins;
        }
    }

    // The pack's bins are read with consecutive lanes on consecutive bins (whole lines per load) and handed
    // over through LDS to the scan's layout of four consecutive bins per lane.
    __shared__ longlong2 s_v[kWaves][kEvalPackBins];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int b = b_begin + j * 64 + lane;
        if (b < b_end) {
            longlong2 v;
            if (SUB && h_par != nullptr) {
                const longlong2 pv = h_par[b], bv = h_built[b];
                v = make_longlong2(pv.x - bv.x, pv.y - bv.y);
                if (store_sibling) h[b] = v;
            } else {
                v = h[b];
            }
            s_v[w][j * 64 + lane] = v;
        }
    }
    wave_lds_sync();
    search_pack(tb, pm, s_v[w], x_in, pack, active, b_begin, b_end, S, inv_g, inv_h, mcw, lambda);
}

// The sums of `count` <= kEvalPackBins bins from `first` over the work items it0, it0 + step, .. below ie of a pair, four per lane
// of a wavefront (past the end: the last one again, so that all loads of an item are issued at once). it0, ie and step are scalars,
// and with them the items' shifts: where the amount of a 64-bit shift lies in the last vector register that a kernel has, this
// chip now and then shifts by another one, which the compiler does not know.
struct ItemsOfPair {
    int begin, end;
    int h_bits;
    bool packed;  // 8-byte partials (see k_hist_dense)
};
__device__ __forceinline__ void add_items_of_pair(const TreeBuffers &tb, const ItemsOfPair &items, int it0, int step, int first, int count,
                                                  long long (&g)[4], long long (&h)[4]) {
    // every item counted at its own scale (item_shift): shift its sums to the tree's
    const int2 *__restrict__ shift = tb.hitem_shift;
    const bool packed = items.packed;
    const int n_bins = tb.n_bins, h_bits = items.h_bits, ie = items.end;
    const unsigned long long h_mask = (1ull << h_bits) - 1ull;
    int at[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        at[j] = first + min(j * 64 + lane_id(), count - 1);
        g[j] = h[j] = 0;
    }
    if (packed) {
        const unsigned long long *__restrict__ from = reinterpret_cast<const unsigned long long *>(tb.partial);
#pragma unroll 2
        for (int it = it0; it < ie; it += step) {
            unsigned long long t[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) t[j] = from[(size_t)it * n_bins + at[j]];
            const int2 sh = shift[it];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const unsigned long long lo = t[j] & h_mask;
                g[j] += ((long long)(t[j] - lo) >> h_bits) << sh.x;
                h[j] += (long long)lo << sh.y;
            }
        }
    } else {
        for (int it = it0; it < ie; it += step) {
            longlong2 v[4];
#pragma unroll
            for (int j = 0; j < 4; ++j) v[j] = tb.partial[(size_t)it * n_bins + at[j]];
            const int2 sh = shift[it];
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                g[j] += v[j].x << sh.x;
                h[j] += v[j].y << sh.y;
            }
        }
    }
}

// What a workgroup that merges a pair's items looks up first, at addresses that the launch tells: all of it is asked for before
// any of it is waited for (the compiler leaves a load behind the branch that it is not needed for). One after the other, the
// pair, its bins, the level's and the tree's records were four trips to the L2 in front of the first item.
struct PairAhead {
    int built, b_begin, b_end;
    ItemsOfPair items;
    double inv_g, inv_h;
    __device__ __forceinline__ void load(const TreeBuffers &tb, int level, int p, const int *bins_from, const int *bins_to) {
        const QuantCtl *__restrict__ q = tb.quant;
        int hchunk = tb.ctl[level].hchunk, flush_rows = q->flush_rows;
        built = tb.hpair_built[p];
        b_begin = *bins_from;
        b_end = *bins_to;
        items.begin = tb.hpair_begin[p];
        items.end = tb.hpair_begin[p + 1];
        items.h_bits = q->h_bits;
        inv_g = q->inv_g;
        inv_h = q->inv_h;
        // (not volatile: behind an asm that might write memory the items' shifts would not be scalar loads, see above)
        auto now = [](int &v) { v = __builtin_amdgcn_readfirstlane(v); };
        now(built), now(b_begin), now(b_end), now(items.begin), now(items.end), now(items.h_bits), now(hchunk), now(flush_rows);
        asm("" : "+s"(built), "+s"(b_begin), "+s"(b_end), "+s"(items.begin), "+s"(items.end), "+s"(items.h_bits), "+s"(hchunk), "+s"(flush_rows));
        items.packed = hchunk <= flush_rows;
    }
};

// k_hist_merge and k_eval_split of a level in one launch: a workgroup owns a pack of a sibling pair. Its wavefronts share
// out the pair's work items, the sums meet in LDS, parent - built gives the sibling, one wavefront searches the built node
// and one its sibling. The histograms are stored for the next level only (not at a tree's last one, which holds half of a
// tree's nodes) and not read back. NW follows from the items per pair (launch_merge_eval). ROOT: level 0, where every
// workgroup adds up the node's sums as well (RootSums).
template <int NW, int ROOT>
__global__ __launch_bounds__(NW * 64) void k_merge_eval(TreeBuffers tb_all, int level, float mcw, float lambda, bool store) {
    __shared__ longlong2 s_sum[NW][kEvalPackBins];
    __shared__ longlong2 s_root[NW];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int p = blockIdx.y, pack = blockIdx.x;
    PairAhead pair;
    pair.load(tb, level, p, tb.pack_begin + pack, tb.pack_begin + pack + 1);
    const int built = pair.built;
    if (built < 0) return;  // (nobody reads the candidates of nodes that do not exist)
    const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
    const int off = (1 << level) - 1, n_bins = tb.n_bins;
    const int b_begin = pair.b_begin, b_end = pair.b_end, nb = b_end - b_begin;
    // (the first threads carry one bin of the pack each - with two wavefronts two bins - from here to the search)
    constexpr int C = NW * 64 < kEvalPackBins ? kEvalPackBins / (NW * 64) : 1;
    longlong2 parent[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int b = c * NW * 64 + (int)threadIdx.x;
        parent[c] = make_longlong2(0, 0);
        if (!ROOT && b < nb) parent[c] = tb.hist(level + 1)[(size_t)p * n_bins + b_begin + b];
    }
    PackMeta pm;
    if (w < (ROOT ? 1 : 2)) pm.load(tb, b_begin, b_end);
    const int sibling = (built & 1) ? built + 1 : built - 1;
    GHPair S{0, 0};
    if (!ROOT) S = tb.nodes[w == 0 ? built : sibling].sum_gh_pair;
    const double inv_g = pair.inv_g, inv_h = pair.inv_h;
    auto add_items = [&](int first, int count, long long(&g)[4], long long(&h)[4]) {
        add_items_of_pair(tb, pair.items, pair.items.begin + w, NW, first, count, g, h);
    };
    if constexpr (ROOT == kRootOfBins) {
        const int b0 = tb.cut_row_ptr[tb.complete_feature], kf = tb.cut_row_ptr[tb.complete_feature + 1] - b0;
        long long g[4], h[4], G = 0, H = 0;
        add_items(b0, kf, g, h);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            G += j * 64 + lane < kf ? g[j] : 0;
            H += j * 64 + lane < kf ? h[j] : 0;
        }
        G = wave_sum_ll(G);
        H = wave_sum_ll(H);
        if (lane == 0) s_root[w] = make_longlong2(G, H);
    }
    {
        long long g[4], h[4];
        add_items(b_begin, nb, g, h);
#pragma unroll
        for (int j = 0; j < 4; ++j) s_sum[w][j * 64 + lane] = make_longlong2(g[j], h[j]);
    }
    __syncthreads();
    longlong2 sum[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int b = c * NW * 64 + (int)threadIdx.x;
        sum[c] = make_longlong2(0, 0);
        if (b >= nb) continue;
#pragma unroll
        for (int i = 0; i < NW; ++i) {
            const longlong2 v = s_sum[i][b];
            sum[c].x += v.x;
            sum[c].y += v.y;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int b = c * NW * 64 + (int)threadIdx.x;
        if (b >= nb) continue;
        const longlong2 other = make_longlong2(parent[c].x - sum[c].x, parent[c].y - sum[c].y);
        s_sum[0][b] = sum[c];
        if (!ROOT) s_sum[1][b] = other;
        if (store) {
            tb.hist(level)[(size_t)(built - off) * n_bins + b_begin + b] = sum[c];
            if (!ROOT) tb.hist(level)[(size_t)(sibling - off) * n_bins + b_begin + b] = other;
        }
    }
    __syncthreads();
    if (w >= (ROOT ? 1 : 2)) return;
    if constexpr (ROOT) {
        if constexpr (ROOT == kRootOfBins) {
            long long G = 0, H = 0;
#pragma unroll
            for (int i = 0; i < NW; ++i) {
                G += s_root[i].x;
                H += s_root[i].y;
            }
            S = root_sums(tb, G, H);
        } else {
            S = root_sums_of_rows(tb, tb.ctl[0].n_hitems);
        }
        if (pack == 0 && lane == 0) set_root_sums(tb, S, lambda);
    }
    search_pack(tb, pm, s_sum[w], (w == 0 ? built : sibling) - off, pack, true, b_begin, b_end, S, inv_g, inv_h, mcw, lambda);
}

// Split search for features of any number of bins (max_num_bin above 255): one workgroup per (feature, node) walks the
// feature's bins in chunks of kBlock with a block-wide inclusive scan of the exact 64-bit sums and a carry from
// chunk to chunk. Same candidates, gains and tie rule as k_eval_split (whose wavefront holds a whole feature of at
// most 256 bins); one candidate per feature. In the CSR layout the node of a pair that was not built from rows is
// derived as parent - built while it is read (and stored for the next level); the dense layout's k_hist_merge has
// done that already.
__device__ __forceinline__ longlong2 wide_bin(const longlong2 *h, const longlong2 *h_par, const longlong2 *h_built, int b) {
    if (h_par == nullptr) return h[b];
    const longlong2 pv = h_par[b], bv = h_built[b];
    return make_longlong2(pv.x - bv.x, pv.y - bv.y);
}

__global__ __launch_bounds__(kBlock) void k_eval_split_wide(TreeBuffers tb_all, int level, float mcw, float lambda,
                                                           bool store_sibling, bool derive, bool root_of_rows) {
#pragma clang fp contract(off)
    __shared__ long long s_g[kWaves], s_h[kWaves];
    __shared__ float s_abs[kWaves];
    __shared__ int s_idx[kWaves];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int f = blockIdx.x;
    const int x_in = blockIdx.y + tb.lvl_x0;
    const int x = (1 << level) - 1 + x_in;
    const TreeNode nd = tb.nodes[x];
    if (!nd.is_valid) return;  // (nobody reads the candidates of an invalid node)
    GHPair S = nd.sum_gh_pair;
    if (root_of_rows) {
        S = root_sums_of_rows(tb, tb.ctl[0].n_hitems);
        if (f == 0 && threadIdx.x == 0) set_root_sums(tb, S, lambda);
    }
    const int cb = tb.cut_row_ptr[f], ce = tb.cut_row_ptr[f + 1];
    SplitCand *out = &tb.cand[(size_t)x_in * tb.n_packs + f];
    if (cb == ce) {
        if (threadIdx.x == 0) out->index = 0x7fffffff;  // a feature without bins has no candidate
        return;
    }
    const int lane = lane_id(), w = wave_id();
    longlong2 *h = tb.hist(level) + (size_t)x_in * tb.n_bins;
    const longlong2 *h_par = nullptr, *h_built = nullptr;
    if (derive && level > 0 && !tb.singles(level)) {  // (the dense layout's k_hist_merge has derived the siblings)
        const int built = tb.hpair_built[x_in >> 1];
        if (built >= 0 && built != x) {
            h_par = tb.hist(level + 1) + (size_t)(x_in >> 1) * tb.n_bins;
            h_built = tb.hist(level) + (size_t)(built - ((1 << level) - 1)) * tb.n_bins;
        }
    }
    const double inv_g = tb.quant->inv_g, inv_h = tb.quant->inv_h;
    const bool ign = tb.ignored != nullptr && tb.ignored[f] != 0;
    // ---- the feature's total (missing = node sum - total), the derived sibling stored on the way
    long long tg = 0, th = 0;
    for (int b = cb + threadIdx.x; b < ce; b += kBlock) {
        const longlong2 v = wide_bin(h, h_par, h_built, b);
        if (h_par != nullptr && store_sibling) h[b] = v;
        tg += v.x;
        th += v.y;
    }
    tg = wave_sum_ll(tg);
    th = wave_sum_ll(th);
    if (lane == 0) {
        s_g[w] = tg;
        s_h[w] = th;
    }
    __syncthreads();
    tg = th = 0;
    for (int i = 0; i < kWaves; ++i) {
        tg += s_g[i];
        th += s_h[i];
    }
    __syncthreads();
    const GHPair m{S.g - (float)((double)tg * inv_g), S.h - (float)((double)th * inv_h)};
    // ---- candidates, chunk by chunk
    long long carry_g = 0, carry_h = 0;
    float best = -1.f, best_score = 0.f;
    int best_idx = 0x7fffffff;
    GHPair best_left{0, 0};
    for (int base = cb; base < ce; base += kBlock) {
        const int b = base + threadIdx.x;
        longlong2 v = make_longlong2(0, 0);
        if (b < ce) v = (h_par != nullptr && !store_sibling) ? wide_bin(h, h_par, h_built, b) : h[b];
        const long long ig = wave_scan_ll(v.x), ih = wave_scan_ll(v.y);
        if (lane == 63) {
            s_g[w] = ig;
            s_h[w] = ih;
        }
        __syncthreads();
        long long wg = 0, wh = 0, cg = 0, ch = 0;
        for (int i = 0; i < kWaves; ++i) {
            if (i < w) {
                wg += s_g[i];
                wh += s_h[i];
            }
            cg += s_g[i];
            ch += s_h[i];
        }
        __syncthreads();
        if (b < ce) {
            const long long exg = carry_g + wg + ig - v.x, exh = carry_h + wh + ih - v.y;  // bins below b
            const GHPair l{(float)((double)exg * inv_g), (float)((double)exh * inv_h)};
            const float gr = split_gain(S, l, mcw, lambda);
            const GHPair l2{l.g + m.g, l.h + m.h};
            const float gl = split_gain(S, l2, mcw, lambda);
            float score = (gl > gr) ? gl : -gr;
            if (ign) score = 0.f;  // column sampling: hist_tree_builder_single.cu:304 / :663
            const float a = fabsf(score);
            if (a > best) {  // (a thread's bins ascend: the first maximum is the one with the smallest index)
                best = a;
                best_score = score;
                best_idx = b;
                best_left = l;
            }
        }
        carry_g += cg;
        carry_h += ch;
    }
    // workgroup arg-max: larger |score| wins, ties go to the smaller bin index (hist_tree_builder_single.cu:330-335)
    float win;
    int win_idx;
    wave_best(best, best_idx, &win, &win_idx);
    if (lane == 0) {
        s_abs[w] = win;
        s_idx[w] = win_idx;
    }
    __syncthreads();
    for (int i = 0; i < kWaves; ++i) {
        if (s_abs[i] > win || (s_abs[i] == win && s_idx[i] < win_idx)) {
            win = s_abs[i];
            win_idx = s_idx[i];
        }
    }
    if (best == win && best_idx == win_idx) {  // exactly one thread: bin indices are distinct
        SplitCand c;
        c.score = best_score;
        c.index = best_idx;
        c.miss = m;
        c.left = best_left;
        c.feature = f;
        c.bin = best_idx - cb;
        *out = c;
    }
}

// k_merge_eval for features of more bins than a wavefront holds, up to kMergeWideBins: a workgroup owns a feature and a sibling
// pair. Quarters of the bins and groups of the work items are shared out over its wavefronts, then one half of them searches
// the built node and the other one its sibling, consecutive bins per thread, as k_eval_split_wide does (same candidates, gains
// and tie rule). Bound by its chain of steps where a level has few pairs, by the memory at deep ones (77 777 x 37, level 6: 65 MB
// of items, parents and stored histograms in 14 us). ms a tree of 1024 bins, two launches -> this one: 20 k x 28, depth 8 0.317 -> 0.217,
// 500 k x 28 0.496 -> 0.408, 50 k x 200, depth 6 0.332 -> 0.251, 2 M x 28 0.669 -> 0.571.
template <int NW>
__global__ __launch_bounds__(NW * 64) void k_merge_eval_wide(TreeBuffers tb_all, int level, float mcw, float lambda, bool store) {
#pragma clang fp contract(off)
    constexpr int kHalf = NW / 2, V = kMergeWideBins / (kHalf * 64), C = kMergeWideBins / (NW * 64);
    __shared__ longlong2 s_sum[NW * kEvalPackBins];
    __shared__ longlong2 s_tot[NW];
    __shared__ float s_abs[NW];
    static_assert(2 * kMergeWideBins <= NW * kEvalPackBins && NW * 64 <= kMergeWideBins, "both nodes' bins");
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int p = blockIdx.y, f = blockIdx.x;
    PairAhead pair;
    pair.load(tb, level, p, tb.cut_row_ptr + f, tb.cut_row_ptr + f + 1);
    const int built = pair.built;
    if (built < 0) return;  // (nobody reads the candidates of nodes that do not exist)
    const int lane = lane_id(), w = __builtin_amdgcn_readfirstlane(wave_id());
    const int off = (1 << level) - 1, n_bins = tb.n_bins;
    const int cb = pair.b_begin, kf = pair.b_end - cb;
    const int sibling = (built & 1) ? built + 1 : built - 1;
    const int half = w >= kHalf ? 1 : 0, wn = w - half * kHalf, x_in = (half ? sibling : built) - off;
    if (kf == 0) {
        if (lane == 0 && wn == 0) tb.cand[(size_t)x_in * tb.n_packs + f].index = 0x7fffffff;  // a feature without bins has no candidate
        return;
    }
    longlong2 parent[C];
#pragma unroll
    for (int c = 0; c < C; ++c)
        parent[c] = tb.hist(level + 1)[(size_t)p * n_bins + cb + min(c * NW * 64 + (int)threadIdx.x, kf - 1)];
    const GHPair S = tb.nodes[off + x_in].sum_gh_pair;
    const double inv_g = pair.inv_g, inv_h = pair.inv_h;
    const bool ign = tb.ignored != nullptr && tb.ignored[f] != 0;
    const int parts = (kf + kEvalPackBins - 1) / kEvalPackBins, groups = NW / parts;
    {
        const int group = w / parts, part = w - group * parts;
        if (group < groups) {
            long long g[4], h[4];
            add_items_of_pair(tb, pair.items, pair.items.begin + group, groups, cb + part * kEvalPackBins, min(kEvalPackBins, kf - part * kEvalPackBins), g, h);
#pragma unroll
            for (int j = 0; j < 4; ++j) s_sum[w * kEvalPackBins + j * 64 + lane] = make_longlong2(g[j], h[j]);
        }
    }
    __syncthreads();
    longlong2 sum[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int b = c * NW * 64 + (int)threadIdx.x;
        sum[c] = make_longlong2(0, 0);
        if (b >= kf) continue;
        for (int i = 0; i < groups; ++i) {
            const longlong2 v = s_sum[i * parts * kEvalPackBins + b];
            sum[c].x += v.x;
            sum[c].y += v.y;
        }
    }
    __syncthreads();
#pragma unroll
    for (int c = 0; c < C; ++c) {
        const int b = c * NW * 64 + (int)threadIdx.x;
        const longlong2 other = make_longlong2(parent[c].x - sum[c].x, parent[c].y - sum[c].y);
        const bool on = b < kf;
        s_sum[b] = on ? sum[c] : make_longlong2(0, 0);
        s_sum[kMergeWideBins + b] = on ? other : make_longlong2(0, 0);
        if (store && on) {
            tb.hist(level)[(size_t)(built - off) * n_bins + cb + b] = sum[c];
            tb.hist(level)[(size_t)(sibling - off) * n_bins + cb + b] = other;
        }
    }
    __syncthreads();
    const int at = (wn * 64 + lane) * V;  // the thread's bins of its half's node
    long long exg[V], exh[V], g = 0, h = 0;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const longlong2 v = s_sum[half * kMergeWideBins + at + j];
        exg[j] = g;
        exh[j] = h;
        g += v.x;
        h += v.y;
    }
    long long upg = g, uph = h;
    wave_scan_pair(upg, uph);
    if (lane == 63) s_tot[w] = make_longlong2(upg, uph);
    __syncthreads();
    long long tg = 0, th = 0, below_g = upg - g, below_h = uph - h;
#pragma unroll
    for (int i = 0; i < kHalf; ++i) {
        const longlong2 v = s_tot[half * kHalf + i];
        tg += v.x;
        th += v.y;
        below_g += i < wn ? v.x : 0;
        below_h += i < wn ? v.y : 0;
    }
    const GHPair m{S.g - scaled_float(tg, inv_g), S.h - scaled_float(th, inv_h)};
    const float fterm = (S.g * S.g) / (S.h + lambda);
    float best = -1.f, best_score = 0.f;
    GHPair best_left{0, 0};
    int which = 0;
#pragma unroll
    for (int j = 0; j < V; ++j) {
        const GHPair l{scaled_float(below_g + exg[j], inv_g), scaled_float(below_h + exh[j], inv_h)};
        const float gr = split_gain_select(S, fterm, l, mcw, lambda);
        const float gl = split_gain_select(S, fterm, GHPair{l.g + m.g, l.h + m.h}, mcw, lambda);
        const float score = ign ? 0.f : (gl > gr ? gl : -gr);  // column sampling: hist_tree_builder_single.cu:304 / :663
        const float a = at + j < kf ? fabsf(score) : -1.f;
        const bool better = a > best;
        which = better ? j : which;
        best_score = better ? score : best_score;
        best_left.g = better ? l.g : best_left.g;
        best_left.h = better ? l.h : best_left.h;
        best = better ? a : best;
    }
    // larger |score| wins, ties go to the smaller bin index (hist_tree_builder_single.cu:330-335): the first wavefront's, the first lane's
    const float win = wave_max_f(best);
    if (lane == 0) s_abs[w] = win;
    __syncthreads();
    int winner = 0;
    float top = s_abs[half * kHalf];
#pragma unroll
    for (int i = 1; i < kHalf; ++i) {
        const float a = s_abs[half * kHalf + i];
        winner = a > top ? i : winner;
        top = fmaxf(top, a);
    }
    if (wn != winner || lane != __ffsll((long long)__ballot(best == win)) - 1) return;
    SplitCand c;
    c.score = best_score;
    c.index = best < 0.f ? 0x7fffffff : cb + at + which;
    c.miss = m;
    c.left = best_left;
    c.feature = f;
    c.bin = at + which;
    tb.cand[(size_t)x_in * tb.n_packs + f] = c;
}

// Per node: reduce the wavefront candidates, fill the split record (hist_tree_builder_single.cu
// :365-389) and apply it to the tree (update_tree, :860-899). One workgroup per node of the level.
__global__ __launch_bounds__(kBlock) void k_best_update(TreeBuffers tb_all, int level, float rt_eps, float lambda) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    __shared__ float s_abs[kWaves];
    __shared__ int s_idx[kWaves];
    __shared__ int s_pack[kWaves];
    const int x_in = blockIdx.x + tb.lvl_x0;
    const int x = (1 << level) - 1 + x_in;
    TreeNode &node = tb.nodes[x];
    SplitPoint &sp = tb.sp[x_in];
    if (!node.is_valid) {
        if (threadIdx.x == 0) {
            SplitPoint z{};
            z.nid = -1;
            z.split_fea_id = -1;
            sp = z;
        }
        return;
    }
    float best = -1.f;
    int best_idx = 0x7fffffff, best_pack = -1;
    if (tb.best_key != nullptr) {
        // sparse level pass: the tasks have already reduced their candidates to one key per node (larger |gain|,
        // then smaller bin index); the record sits in the slot of the task that searches the winning bin's feature
        if (threadIdx.x == 0) {
            const unsigned long long key = tb.best_key[x_in];
            tb.best_key[x_in] = 0ull;  // ready for the next level
            if (key != 0ull) {
                best_idx = (int)(0xffffffffu - (unsigned)key);
                best_pack = tb.feat_slot[tb.cut_fid[best_idx]];
                best = __uint_as_float((unsigned)(key >> 32));
            }
        }
    } else
    for (int p = threadIdx.x; p < tb.n_packs; p += kBlock) {
        const SplitCand &c = tb.cand[(size_t)x_in * tb.n_packs + p];
        if (c.index == 0x7fffffff) continue;  // a wavefront whose features have no bins
        float a = fabsf(c.score);
        if (a > best || (a == best && c.index < best_idx)) {
            best = a;
            best_idx = c.index;
            best_pack = p;
        }
    }
    {
        float win;
        int win_idx;
        const int owner = wave_best(best, best_idx, &win, &win_idx);
        best_pack = read_lane(best_pack, owner);
        best = win;
        best_idx = win_idx;
    }
    if (lane_id() == 0) {
        s_abs[wave_id()] = best;
        s_idx[wave_id()] = best_idx;
        s_pack[wave_id()] = best_pack;
    }
    __syncthreads();
    if (threadIdx.x != 0) return;
    for (int i = 0; i < kWaves; ++i) {
        if (s_abs[i] > best || (s_abs[i] == best && s_idx[i] < best_idx)) {
            best = s_abs[i];
            best_idx = s_idx[i];
            best_pack = s_pack[i];
        }
    }
    if (best_pack < 0) {  // no candidate at all (a node none of whose rows stores a value): a leaf
        no_split(tb, x, x_in);
        return;
    }
    const SplitCand c = tb.cand[(size_t)x_in * tb.n_packs + best_pack];
    const int f = tb.cut_fid[c.index];
    const int bin = c.index - tb.cut_row_ptr[f];
    apply_split(tb, x, x_in, node, c, f, bin, tb.cut_val[c.index - (bin != 0 ? 1 : 0)], rt_eps, lambda);
}

// ------------------------------------------------------------------------------ partition

// Row lists of the CSR layout. Partition work items: every node of a level that holds rows owns ceil(rows / kPartChunk)
// items, planned one level ahead (k_tree_init for the root, k_part_scan_plan for the children it creates) so that no
// planning step sits between the split search and the partition; the items of a node that did not split return at once.
// (The dense layout's partition plans its items itself: level_kernels.hip.)
// Scan the per-item left counts, publish the children's row segments and plan the histogram work
// of the next level: per sibling pair the child with fewer rows is built (ties: the left one, as
// hist_tree_builder_single.cu:466-467), the other one comes from subtraction. One workgroup.
constexpr int kScanLdsItems = 12 * 1024;  // item offsets that k_part_scan_plan keeps in LDS (25 M rows)
__global__ __launch_bounds__(kBlock) void k_part_scan_plan(TreeBuffers tb_all, int level) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    __shared__ int lds[kWaves];
    __shared__ int s_loff[kScanLdsItems + 1];
    const int nl = 1 << level, off = nl - 1;
    const int n_p = tb.ctl[level].n_pitems;
    const int *pb_cur = tb.pbegin(level);
    int *pb_next = tb.pbegin(level + 1);
    // the offsets of the items also stay in LDS when they fit, so that the per-node step below does not wait for
    // its own global stores
    const bool in_lds = n_p <= kScanLdsItems;
    // (what the per-node step needs from global memory is requested here, next to the item counts: one round trip)
    TreeNode my_node{};
    int2 my_seg = make_int2(0, 0);
    int my_pb0 = 0, my_pb1 = 0;
    const bool fast = nl <= kBlock && !tb.singles(level + 1) && (int)threadIdx.x < nl;
    if (fast) {
        my_node = tb.nodes[off + threadIdx.x];
        my_seg = tb.seg[off + threadIdx.x];
        my_pb0 = pb_cur[threadIdx.x];
        my_pb1 = pb_cur[threadIdx.x + 1];
    }
    int carry = 0;
    constexpr int IPT = 20;  // items per thread and step (10 M rows are 4 883 items: one step)
    for (int base = 0; base < n_p; base += kBlock * IPT) {
        const int i0 = base + threadIdx.x * IPT;
        int v[IPT];
        int local = 0;
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            v[j] = (i0 + j) < n_p ? tb.pitem_nleft[i0 + j] : 0;
            local += v[j];
        }
        int tot;
        int run = carry + block_excl_scan(local, lds, &tot);
#pragma unroll
        for (int j = 0; j < IPT; ++j) {
            if (i0 + j < n_p) {
                tb.pitem_loff[i0 + j] = run;
                if (in_lds) s_loff[i0 + j] = run;
            }
            run += v[j];
        }
        carry += tot;
    }
    if (threadIdx.x == 0) {
        tb.pitem_loff[n_p] = carry;
        if (in_lds) s_loff[n_p] = carry;
    }
    __syncthreads();
    if (tb.singles(level + 1)) {
        // No parent histograms below this level (the arena is smaller than the level): every child of a split node
        // is built from its own rows; the plan's "pairs" are the 2 nl single nodes of the next level.
        int rows_sum = 0, n_built = 0;
        for (int x_in = threadIdx.x; x_in < nl; x_in += kBlock) {
            const TreeNode &nd = tb.nodes[off + x_in];
            const int2 sg = tb.seg[off + x_in];
            if (node_splits(nd)) {
                const int nleft = tb.pitem_loff[pb_cur[x_in + 1]] - tb.pitem_loff[pb_cur[x_in]];
                tb.node_nleft[x_in] = nleft;
                tb.seg[nd.lch_index] = make_int2(sg.x, sg.x + nleft);
                tb.seg[nd.rch_index] = make_int2(sg.x + nleft, sg.y);
                tb.hpair_built[2 * x_in] = nd.lch_index;
                tb.hpair_built[2 * x_in + 1] = nd.rch_index;
                rows_sum += sg.y - sg.x;
                n_built += 2;
            } else {
                tb.node_nleft[x_in] = 0;
                tb.seg[nd.lch_index] = make_int2(0, 0);
                tb.seg[nd.rch_index] = make_int2(0, 0);
                tb.hpair_built[2 * x_in] = -1;
                tb.hpair_built[2 * x_in + 1] = -1;
            }
        }
        const int total_rows = block_sum(rows_sum, lds);
        n_built = block_sum(n_built, lds);
        const int room = max(tb.target_hitems / 4, tb.target_hitems - n_built);
        int chunk = (total_rows + room - 1) / room;
        chunk = max(kHistMinChunk, (chunk + 255) / 256 * 256);
        int hcarry = 0, pcarry = 0;
        for (int base = 0; base < 2 * nl; base += kBlock) {
            const int c_in = base + threadIdx.x;
            int cnt = 0, pc = 0;
            if (c_in < 2 * nl) {
                const int2 sg = tb.seg[2 * nl - 1 + c_in];  // the child's heap id: (2 nl - 1) + c_in
                if (tb.hpair_built[c_in] >= 0) cnt = (sg.y - sg.x + chunk - 1) / chunk;
                pc = (sg.y - sg.x + kPartChunk - 1) / kPartChunk;
            }
            int tot, ptot;
            const int ex = block_excl_scan(cnt, lds, &tot);
            const int pex = block_excl_scan(pc, lds, &ptot);
            if (c_in < 2 * nl) {
                tb.hpair_begin[c_in] = hcarry + ex;
                pb_next[c_in] = pcarry + pex;
            }
            hcarry += tot;
            pcarry += ptot;
        }
        if (threadIdx.x == 0) {
            tb.hpair_begin[2 * nl] = hcarry;
            pb_next[2 * nl] = pcarry;
            LevelCtl c;
            c.hchunk = chunk;
            c.n_hitems = hcarry;
            c.n_pitems = pcarry;
            c.rows_built = total_rows;
            tb.ctl[level + 1] = c;
        }
        return;
    }
    if (nl <= kBlock) {
        // the usual case (levels up to 8): one node per thread, everything after the scan stays in registers
        const int x_in = threadIdx.x;
        int built = -1, rows = 0;
        int pl = 0, pr = 0;  // partition items of the two children
        if (x_in < nl) {
            const TreeNode &nd = my_node;
            const int2 sg = my_seg;
            if (node_splits(nd)) {
                const int nleft = in_lds ? s_loff[my_pb1] - s_loff[my_pb0] : tb.pitem_loff[my_pb1] - tb.pitem_loff[my_pb0];
                const int nright = (sg.y - sg.x) - nleft;
                tb.node_nleft[x_in] = nleft;
                tb.seg[nd.lch_index] = make_int2(sg.x, sg.x + nleft);
                tb.seg[nd.rch_index] = make_int2(sg.x + nleft, sg.y);
                built = (nleft <= nright) ? nd.lch_index : nd.rch_index;
                rows = min(nleft, nright);
                pl = (nleft + kPartChunk - 1) / kPartChunk;
                pr = (nright + kPartChunk - 1) / kPartChunk;
            } else {
                tb.node_nleft[x_in] = 0;
                tb.seg[nd.lch_index] = make_int2(0, 0);
                tb.seg[nd.rch_index] = make_int2(0, 0);
            }
            tb.hpair_built[x_in] = built;
        }
        const int total_rows = block_sum(rows, lds);
        const int n_built = block_sum(built >= 0 ? 1 : 0, lds);
        const int room = max(tb.target_hitems / 4, tb.target_hitems - n_built);
        int chunk = (total_rows + room - 1) / room;
        chunk = max(kHistMinChunk, (chunk + 255) / 256 * 256);
        const int cnt = built >= 0 ? (rows + chunk - 1) / chunk : 0;
        int tot, ptot;
        const int ex = block_excl_scan(cnt, lds, &tot);
        const int pex = block_excl_scan(pl + pr, lds, &ptot);
        if (x_in < nl) {
            tb.hpair_begin[x_in] = ex;
            pb_next[2 * x_in] = pex;
            pb_next[2 * x_in + 1] = pex + pl;
        }
        if (threadIdx.x == 0) {
            tb.hpair_begin[nl] = tot;
            pb_next[2 * nl] = ptot;
            LevelCtl c;
            c.hchunk = chunk;
            c.n_hitems = tot;
            c.n_pitems = ptot;
            c.rows_built = total_rows;
            tb.ctl[level + 1] = c;
        }
        return;
    }
    // children segments + rows of the built child of every pair
    int rows_sum = 0;
    for (int x_in = threadIdx.x; x_in < nl; x_in += kBlock) {
        const TreeNode &nd = tb.nodes[off + x_in];
        const int2 sg = tb.seg[off + x_in];
        int built = -1;
        if (node_splits(nd)) {
            int nleft = tb.pitem_loff[pb_cur[x_in + 1]] - tb.pitem_loff[pb_cur[x_in]];
            int nright = (sg.y - sg.x) - nleft;
            tb.node_nleft[x_in] = nleft;
            tb.seg[nd.lch_index] = make_int2(sg.x, sg.x + nleft);
            tb.seg[nd.rch_index] = make_int2(sg.x + nleft, sg.y);
            built = (nleft <= nright) ? nd.lch_index : nd.rch_index;
            rows_sum += min(nleft, nright);
        } else {
            tb.node_nleft[x_in] = 0;
            tb.seg[nd.lch_index] = make_int2(0, 0);
            tb.seg[nd.rch_index] = make_int2(0, 0);
        }
        tb.hpair_built[x_in] = built;
    }
    const int total_rows = block_sum(rows_sum, lds);
    int n_built = 0;
    for (int x_in = threadIdx.x; x_in < nl; x_in += kBlock) n_built += tb.hpair_built[x_in] >= 0 ? 1 : 0;
    n_built = block_sum(n_built, lds);
    // every built node adds up to one partly filled item: size the items so that their number stays
    // within target_hitems (= the workgroups the chip holds at once; one more would run as a second round)
    const int room = max(tb.target_hitems / 4, tb.target_hitems - n_built);
    int chunk = (total_rows + room - 1) / room;
    chunk = max(kHistMinChunk, (chunk + 255) / 256 * 256);
    carry = 0;
    for (int base = 0; base < nl; base += kBlock) {
        int x_in = base + threadIdx.x;
        int cnt = 0;
        if (x_in < nl) {
            int built = tb.hpair_built[x_in];
            if (built >= 0) {
                int2 sg = tb.seg[built];
                cnt = (sg.y - sg.x + chunk - 1) / chunk;
            }
        }
        int tot;
        int ex = block_excl_scan(cnt, lds, &tot);
        if (x_in < nl) tb.hpair_begin[x_in] = carry + ex;
        carry += tot;
    }
    // partition items of the next level: every child that received rows
    int pcarry = 0;
    for (int base = 0; base < nl; base += kBlock) {
        const int x_in = base + threadIdx.x;
        int pl = 0, pr = 0;
        if (x_in < nl) {
            const TreeNode &nd = tb.nodes[off + x_in];
            const int2 sl = tb.seg[nd.lch_index], sr = tb.seg[nd.rch_index];
            pl = (sl.y - sl.x + kPartChunk - 1) / kPartChunk;
            pr = (sr.y - sr.x + kPartChunk - 1) / kPartChunk;
        }
        int ptot;
        const int pex = block_excl_scan(pl + pr, lds, &ptot);
        if (x_in < nl) {
            pb_next[2 * x_in] = pcarry + pex;
            pb_next[2 * x_in + 1] = pcarry + pex + pl;
        }
        pcarry += ptot;
    }
    if (threadIdx.x == 0) {
        tb.hpair_begin[nl] = carry;
        pb_next[2 * nl] = pcarry;
        LevelCtl c;
        c.hchunk = chunk;
        c.n_hitems = carry;
        c.n_pitems = pcarry;
        c.rows_built = total_rows;
        tb.ctl[level + 1] = c;
    }
}

// Stable two-way compaction of a work item's rows into the children's segments with wavefront
// ballots and popcounts. (Moving the gradient pairs along with the row ids was measured: it makes
// the histogram's gradient reads sequential but costs more in this kernel than it saves there.)
// The row -> node map is not touched here; k_end_bounds / k_tree_end derive it from the row lists
// when it is needed.
template <bool DIRECT>
__global__ __launch_bounds__(kBlock) void k_part_scatter(TreeBuffers tb_all, int level) {
    __shared__ int s_x;
    __shared__ int s_cnt[kPartChunk / kBlock][2][kWaves];
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int *__restrict__ ridx_cur = tb.list(level);
    int *__restrict__ ridx_next = tb.list(level + 1);
    const int item = blockIdx.x;
    if (item >= tb.ctl[level].n_pitems) return;
    const int nl = 1 << level, off = nl - 1;
    if (threadIdx.x == 0) s_x = find_owner(tb.pbegin(level), nl, item);
    __syncthreads();
    const int x_in = s_x;
    if (!node_splits(tb.nodes[off + x_in])) return;
    const int2 sg = tb.seg[off + x_in];
    const int first_item = tb.pbegin(level)[x_in];
    const int pb = sg.x + (item - first_item) * kPartChunk;
    const int pe = min(sg.y, pb + kPartChunk);
    const int loff = tb.pitem_loff[item] - tb.pitem_loff[first_item];
    int left_base = sg.x + loff;
    int right_base = sg.x + tb.node_nleft[x_in] + ((pb - sg.x) - loff);
    const int lane = lane_id(), w = wave_id();
    // all loads of the item first (unconditional, clamped positions), one barrier for the wavefront counts of all
    // eight steps, then all stores
    constexpr int R = kPartChunk / kBlock;
    int row[R];
    const unsigned rights = tb.goes_right[(size_t)item * kBlock + threadIdx.x];  // bit k: the thread's k-th row goes right
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const int pos = min(pb + k * kBlock + (int)threadIdx.x, pe - 1);
        row[k] = DIRECT ? pos : ridx_cur[pos];
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

// ---------------------------------------------------------------------------------- prune
// Bottom-up, level-parallel form of the reference's Tree::prune_self (src/thundergbm/tree.cu:96-128):
// a node whose two children are valid leaves and whose gain is below gamma becomes a leaf and its
// children are marked pruned; then final ids are renumbered over valid, unpruned nodes.
__device__ void prune_tree(const TreeBuffers &tb, float gamma) {  // every thread of a kBlock-wide workgroup
    __shared__ int lds[kWaves];
    for (int level = tb.depth - 1; level >= 0; --level) {
        const int nl = 1 << level, off = nl - 1;
        for (int x_in = threadIdx.x; x_in < nl; x_in += kBlock) {
            TreeNode &p = tb.nodes[off + x_in];
            if (p.is_valid && !p.is_leaf) {
                TreeNode &l = tb.nodes[p.lch_index];
                TreeNode &r = tb.nodes[p.rch_index];
                if (l.is_valid && l.is_leaf && r.is_valid && r.is_leaf && p.gain < gamma) {
                    l.is_pruned = true;
                    r.is_pruned = true;
                    p.is_leaf = true;
                }
            }
        }
        __syncthreads();
    }
    int carry = 0;
    for (int base = 0; base < tb.n_nodes; base += kBlock) {
        int i = base + threadIdx.x;
        int keep = 0;
        if (i < tb.n_nodes) keep = (tb.nodes[i].is_valid && !tb.nodes[i].is_pruned) ? 1 : 0;
        int tot;
        int ex = block_excl_scan(keep, lds, &tot);
        if (keep) tb.nodes[i].final_id = carry + ex;
        carry += tot;
    }
    // value a row adds to its prediction when it ended in node i: the weight of the first ancestor that
    // was not pruned (what predict_in_training finds by climbing, tree_builder.cu:62-74)
    for (int i = threadIdx.x; i < tb.n_nodes; i += kBlock) {
        int x = i;
        while (x != -1 && tb.nodes[x].is_pruned) x = tb.nodes[x].parent_index;
        tb.leaf_value[i] = x >= 0 ? tb.nodes[x].base_weight : 0.f;
    }
}

__global__ __launch_bounds__(kBlock) void k_prune(TreeBuffers tb_all, float gamma) {
    prune_tree(tb_all.for_class(blockIdx.z), gamma);
}

// -------------------------------------------------------------------------- end of a tree
// The trainer keeps rows as per-node lists; everything that happens per row after the last split
// search wants row order: the row -> node map (the reference's ins2node_id), the prediction update
// (tree_builder.cu:62-74), the training metric (pointwise_metric.cu:13-20, multiclass_metric.cu:39-44)
// and the next round's gradients (regression_obj.h:130-154). Scattering node ids from the lists into
// a row-ordered array costs one partial 128-byte line per row, so this kernel goes the other way:
// a workgroup owns kRowBlock consecutive rows, finds for every node that still holds rows the part of
// its (ascending) row list that falls into the block by binary search, drops the node ids into LDS
// and then walks its rows in order with coalesced accesses only.
//   A node holds rows if it is valid and was not split; a split node of level `lookup_level` still
// holds the rows of its children (the last level of a tree is never partitioned into lists: nobody
// reads those lists), each row's child follows from the split feature's bin as in
// hist_tree_builder_single.cu:986-1011.
// MODE 0: write the row -> node map only. 1: prediction update of one tree. 2: prediction update,
// metric partials, next gradients and their block statistics (objectives with one tree per round;
// same arithmetic and order as k_gradient_pointwise, k_sum_gh and k_metric_partial).
__device__ __forceinline__ void metric_row(int kind, int n, int K, int i, float yi, const float *__restrict__ yp,
                                           float p0, double &acc, float &accf);

struct TreeEndArgs {
    int lookup_level;
    const float *y;
    float *yp;
    float lr;
    int objective, metric_kind;
    GHPair *gh;
    GradStats *stats;
    double *metric_partial;
    int with_prune;  // prune the tree first (prune_self with `gamma`)
    float gamma;
    unsigned *gh_words;  // MODE 2: where the rows' gradient words go (word_from_row; nullptr: nowhere)
};

// Threads per row block. While the workgroups fit the chip at once, four rows per thread make every step of the chain list
// position -> row -> bin -> leaf -> prediction one round of loads (500 k rows: 28 us with 256 threads, 14 with 1024);
// beyond that the registers of the 1024 cost residency (10 M rows: 74 and 128 us).
constexpr int kEndWide = 1024;
bool end_wide(int n, int n_class = 1) { return (long)row_blocks(n) * n_class <= 512; }
constexpr int kEndInline = 8;                        // shorter sub-ranges are handled by the finding thread
constexpr int kEndListCap = kRowBlock / kEndInline;  // so at most this many longer ones exist per block

// First position p of the ascending run list[sx, sy) with list[p] >= r, given first = list[sx] < r and
// last = list[sy - 1] >= r. A node's rows are spread roughly evenly over the matrix, so the search
// starts at the interpolated position, brackets the answer by doubling steps and bisects the bracket:
// a handful of probes that (unlike a bisection of the whole run) all fall into a few neighbouring lines.
__device__ int list_lower_bound(const int *__restrict__ list, int sx, int sy, int first, int last, int r) {
    int g = sx + (int)((long long)(r - first) * (sy - 1 - sx) / (last - first));
    g = min(max(g, sx + 1), sy - 1);
    int lo, hi;  // invariant: list[lo] < r <= list[hi]
    if (list[g] < r) {
        lo = g;
        int step = 16;
        while (lo + step < sy - 1 && list[lo + step] < r) {
            lo += step;
            step *= 2;
        }
        hi = min(lo + step, sy - 1);
    } else {
        hi = g;
        int step = 16;
        while (hi - step > sx && list[hi - step] >= r) {
            hi -= step;
            step *= 2;
        }
        lo = max(hi - step, sx);
    }
    while (hi - lo > 1) {
        int mid = lo + (hi - lo) / 2;
        if (list[mid] < r) lo = mid; else hi = mid;
    }
    return hi;
}

template <bool SPARSE>
__device__ __forceinline__ int end_child_of(const TreeBuffers &tb, const DenseBins &dbins, const CsrBins &cbins,
                                            const TreeNode &nd, int row) {
    bool right;
    if (SPARSE) {
        const int cb = tb.cut_row_ptr[nd.split_feature_id], ce = tb.cut_row_ptr[nd.split_feature_id + 1];
        // (the node's own heap id is its children's parent index; wide features keep their split bin in a side array)
        const int sb = tb.split_bin != nullptr ? tb.split_bin[(nd.lch_index - 1) / 2] : (int)nd.split_bid;
        right = csr_goes_right(cbins, row, cb, ce, cb + sb, nd.default_right);
    } else if (dbins.bin_bytes == 2) {
        const int b = reinterpret_cast<const uint16_t *>(dbins.col)[(size_t)nd.split_feature_id * dbins.col_stride + row];
        const int sb = tb.split_bin != nullptr ? tb.split_bin[(nd.lch_index - 1) / 2] : (int)nd.split_bid;
        right = (b == kMissingBin16) ? nd.default_right : (b >= sb);
    } else if (dbins.feat_col != nullptr) {
        const int f = nd.split_feature_id;
        const int t = (int)dbins.col[(size_t)dbins.feat_col[f] * dbins.col_stride + row] - (int)dbins.feat_lo[f];
        right = ((unsigned)t >= (unsigned)(tb.cut_row_ptr[f + 1] - tb.cut_row_ptr[f])) ? nd.default_right
                                                                                     : (t >= (int)nd.split_bid);
    } else {
        const int b = dbins.col[(size_t)nd.split_feature_id * dbins.col_stride + row];
        right = (b == kMissingBin) ? nd.default_right : (b >= nd.split_bid);
    }
    return right ? nd.rch_index : nd.lch_index;
}

// bound[b * n_holders + x] = first position of node x's row list whose row is >= b * kRowBlock (b = 0 ..
// n_blocks), 0 everywhere for nodes that hold no rows: row block b then owns positions [bound[b][x],
// bound[b + 1][x]) of every list. One thread per entry; neighbouring threads search neighbouring
// boundaries of the same list.
// with_prune: the launch has one workgroup more, which prunes the tree meanwhile (the searches read fields of the
// nodes that pruning does not touch; what both produce is first read by k_tree_end).
__global__ __launch_bounds__(kBlock) void k_end_bounds(TreeBuffers tb_all, int lookup_level, int n_blocks,
                                                      int with_prune, float gamma) {
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    const int search_blocks = gridDim.x - (with_prune ? 1 : 0);
    if (with_prune && blockIdx.x == search_blocks) {
        prune_tree(tb, gamma);
        return;
    }
    const int n_holders = (1 << tb.depth) - 1;
    const size_t total = (size_t)n_holders * (n_blocks + 1);
    for (size_t idx = (size_t)blockIdx.x * kBlock + threadIdx.x; idx < total; idx += (size_t)search_blocks * kBlock) {
        const int x = (int)(idx / (n_blocks + 1)), b = (int)(idx % (n_blocks + 1));
        const TreeNode &nd = tb.nodes[x];
        const int level = 31 - __clz(x + 1);
        int pos = 0;
        if (nd.is_valid && (nd.split_feature_id < 0 || level == lookup_level)) {
            const int2 sg = tb.seg[x];
            if (sg.y > sg.x) {
                const long long r = (long long)b * kRowBlock;
                if (level == 0) {  // the root's list is the identity
                    pos = (int)min(max(r, (long long)sg.x), (long long)sg.y);
                } else {
                    const int *list = tb.list(level);
                    const int first = list[sg.x], last = list[sg.y - 1];
                    pos = r <= first ? sg.x : (r > last ? sg.y : list_lower_bound(list, sg.x, sg.y, first, last, (int)r));
                }
            }
        }
        tb.end_bound[(size_t)b * n_holders + x] = pos;
    }
}

// The row-ordered part of the end of a tree: s_leaf holds the node of every row of the block.
template <int MODE, int BLK>
__device__ __forceinline__ void tree_end_rows(const TreeBuffers &tb, const TreeEndArgs &a, const short *s_leaf, int r0, int r1) {
    __shared__ float s_f[5 * BLK / 64];
    __shared__ double s_d[BLK / 64];
    constexpr int U = 4;
    if (MODE == 0) {
        for (int i = r0 + threadIdx.x; i < r1; i += BLK) {
            const int x = s_leaf[i - r0];
            if (x >= 0) tb.nid[i] = x;
        }
        return;
    }
    // rows in order; thread t takes rows t, t + BLK, ... (the order every row-blocked reduction uses)
    const float *__restrict__ y = a.y;
    float *__restrict__ yp = a.yp;
    GHPair *__restrict__ gh = a.gh;
    const float *__restrict__ leaf_value = tb.leaf_value;
    RowStats st;
    double acc = 0;
    float accf = 0;
    for (int i0 = r0 + threadIdx.x; i0 < r1; i0 += BLK * U) {
        float p[U], w[U], yi[U];
        bool ok[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * BLK;
            ok[u] = i < r1;
            const int x = ok[u] ? s_leaf[i - r0] : -1;
            p[u] = ok[u] ? yp[i] : 0.f;
            yi[u] = (MODE == 2 && ok[u]) ? y[i] : 0.f;
            w[u] = x >= 0 ? leaf_value[x] : 0.f;
            ok[u] = ok[u] && (MODE == 2 || x >= 0);
            if (x >= 0) p[u] += a.lr * w[u];
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!ok[u]) continue;
            const int i = i0 + u * BLK;
            yp[i] = p[u];
            if (MODE == 2) {
                metric_row(a.metric_kind, tb.n, 1, i, yi[u], yp, p[u], acc, accf);
                const GHPair o = pointwise_gradient(a.objective, yi[u], p[u]);
                if (gh != nullptr) gh[i] = o;  // (nullptr: the next tree reads the words only)
                if (a.gh_words != nullptr) a.gh_words[i] = word_from_row(a.objective, yi[u], p[u]);
                st.add(o);
            }
        }
    }
    if (MODE == 2) {
        store_block_stats<BLK / 64>(st, s_f, a.stats + blockIdx.x);
        acc += (double)accf;
        store_block_sum_d<BLK / 64>(acc, s_d, a.metric_partial + blockIdx.x);
    }
}


template <int MODE, bool SPARSE, int BLK>
__global__ __launch_bounds__(BLK) void k_tree_end(TreeBuffers tb_all, DenseBins dbins, CsrBins cbins, TreeEndArgs a) {
    __shared__ short s_leaf[kRowBlock];  // node of every row of the block (depth <= 14: ids below 2^15), -1: none
    const TreeBuffers tb = tb_all.for_class(blockIdx.z);
    if (MODE == 1) a.yp += (size_t)blockIdx.z * tb.n;  // class-major predictions
    __shared__ int s_list[kEndListCap][3];  // node, first and one-past-last list position
    __shared__ int s_split[kEndListCap];    // -1: the rows stay in the node; else feature | bin << 16 | default_right << 24
    __shared__ int s_off[kEndListCap];
    __shared__ int s_scan[BLK / 64];
    __shared__ int s_n;
    const int r0 = blockIdx.x * kRowBlock, r1 = min(tb.n, r0 + kRowBlock);
    constexpr int U = 4;
    if (tb.nid16 != nullptr) {
        // sparse level pass: the row -> node map is kept per row, nothing to look up
        for (int i = threadIdx.x; i < kRowBlock; i += BLK) s_leaf[i] = r0 + i < r1 ? (short)tb.nid16[r0 + i] : (short)-1;
    } else {
    for (int i = threadIdx.x; i < kRowBlock; i += BLK) s_leaf[i] = -1;
    if (threadIdx.x == 0) s_n = 0;
    __syncthreads();
    const int n_holders = (1 << tb.depth) - 1;  // nodes of the levels that own row lists
    const int *b_lo = tb.end_bound + (size_t)blockIdx.x * n_holders, *b_hi = b_lo + n_holders;
    for (int x = threadIdx.x; x < n_holders; x += BLK) {
        const int pa = b_lo[x], pb = b_hi[x];
        if (pb <= pa) continue;
        const TreeNode &nd = tb.nodes[x];
        // (trees of up to kEndListCap row-holding nodes list every sub-range: the inline walk is a chain of
        // dependent loads)
        if (pb - pa > kEndInline || n_holders <= kEndListCap) {
            int e = atomicAdd(&s_n, 1);
            s_list[e][0] = x;
            s_list[e][1] = pa;
            s_list[e][2] = pb;
            s_split[e] = nd.split_feature_id < 0
                             ? -1
                             : (nd.split_feature_id | (int)nd.split_bid << 16 | (nd.default_right ? 1 : 0) << 24);
        } else {
            const int *list = tb.list(31 - __clz(x + 1));
            for (int p = pa; p < pb; ++p) {
                const int row = x == 0 ? p : list[p];
                s_leaf[row - r0] = nd.split_feature_id >= 0 ? end_child_of<SPARSE>(tb, dbins, cbins, nd, row) : x;
            }
        }
    }
    __syncthreads();
    // The listed sub-ranges are walked as one flat index space spread over all threads (independent
    // loads in flight instead of one dependent chain per sub-range): s_off = exclusive scan of the lengths.
    const int n_list = s_n;
    int total = 0;
    for (int base = 0; base < n_list; base += BLK) {
        const int e = base + threadIdx.x;
        const int len = e < n_list ? s_list[e][2] - s_list[e][1] : 0;
        int tot;
        const int ex = block_excl_scan<BLK / 64>(len, s_scan, &tot);
        if (e < n_list) s_off[e] = total + ex;
        total += tot;
    }
    __syncthreads();
    for (int j0 = threadIdx.x; j0 < total; j0 += BLK * U) {
        // (every load is unconditional - entries past the end repeat the last one and are skipped when the results
        // are stored -, so a thread's four list entries, then its four bins, are in flight together)
        int node[U], row[U], split[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int j = min(j0 + u * BLK, total - 1);
            int lo = 0, hi = n_list;  // last entry with s_off <= j
            while (hi - lo > 1) {
                const int mid = (lo + hi) / 2;
                if (s_off[mid] <= j) lo = mid; else hi = mid;
            }
            node[u] = s_list[lo][0];
            split[u] = s_split[lo];
            const int p = s_list[lo][1] + (j - s_off[lo]);
            const int listed = tb.list(31 - __clz(node[u] + 1))[p];  // (the root's list is the identity and not stored)
            row[u] = node[u] == 0 ? p : listed;
        }
        // (16-bit bins and bundled columns: the packed split word has no room for what the decision needs)
        if (SPARSE || dbins.bin_bytes == 2 || dbins.feat_col != nullptr) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (j0 + u * BLK >= total) continue;
                s_leaf[row[u] - r0] =
                    split[u] >= 0 ? end_child_of<SPARSE>(tb, dbins, cbins, tb.nodes[node[u]], row[u]) : node[u];
            }
        } else {
            int bin[U];
#pragma unroll
            for (int u = 0; u < U; ++u)  // (feature 0 for the entries of nodes that did not split)
                bin[u] = dbins.col[(size_t)(split[u] >= 0 ? split[u] & 0xffff : 0) * dbins.col_stride + row[u]];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                if (j0 + u * BLK >= total) continue;
                int leaf = node[u];
                if (split[u] >= 0) {
                    const bool right = bin[u] == kMissingBin ? (split[u] >> 24) != 0 : bin[u] >= ((split[u] >> 16) & 0xff);
                    leaf = 2 * node[u] + (right ? 2 : 1);  // heap order: children of x are 2x + 1 and 2x + 2
                }
                s_leaf[row[u] - r0] = leaf;
            }
        }
    }
    }  // row lists
    __syncthreads();
    tree_end_rows<MODE, BLK>(tb, a, s_leaf, r0, r1);
}

// The end of a tree whose rows' nodes are in tb.nid (k_small_level, and k_split_count where launch_partition_hist serves the
// levels), and which is small enough for every workgroup to prune it in LDS by itself; the last one has no rows and writes the
// finished nodes into the model (in place they would change under the other workgroups' eyes). Pruning is a ballot a level in
// one wavefront and every node's own climb instead of two barriers a level: 11.0 -> 8.0 us at 1605 rows and depth 6, 13.3 -> 11.1 at
// 500 k and depth 8. One launch instead of k_end_bounds, k_tree_end and the copy: 31 -> 8 us at 10 k rows. At 500 k x 28 the last
// level's count launch updates the tree and maps the rows (11 us) and the end takes 11, where k_best_update, k_end_bounds and
// k_tree_end took 4.4, 9.7 and 14.7.
// RW: 0, or the dwords of a row's record, where a row has all of its bins in one: then the rows' nodes are not in the map, but every row
// walks the tree here, its record in registers and a word of every node in LDS, and leaves its node there. What the count launches
// stored row by row, 4 bytes to a line of its own each, is what this saves; the last level's update of the tree is a launch of its own again.
// Bound by the walk's vector instructions. Eight trees of 500 k rows of 12 columns, last count and end: 43 and 15.5 us -> 4.9 (the update)
// and 32.7; one tree of 500 k x 28 10.7 and 11.1 -> 4.2 and 18.6, which is why only class trees built together walk.
// (by value: a choice between two places of an array is a choice of addresses to the compiler, and the array goes to scratch memory)
__device__ __forceinline__ unsigned either(bool second, unsigned a, unsigned b) { return second ? b : a; }
template <int RW>
struct RowRecord {
    uint4 v[RW / 4];
    __device__ __forceinline__ void load(const uint8_t *from) {
#pragma unroll
        for (int i = 0; i < RW / 4; ++i) v[i] = reinterpret_cast<const uint4 *>(from)[i];
    }
    __device__ __forceinline__ unsigned dword(unsigned d) const {
        uint4 q = v[0];
        if constexpr (RW == 8) q = make_uint4(either(d & 4u, v[0].x, v[1].x), either(d & 4u, v[0].y, v[1].y), either(d & 4u, v[0].z, v[1].z), either(d & 4u, v[0].w, v[1].w));
        return either(d & 2u, either(d & 1u, q.x, q.y), either(d & 1u, q.z, q.w));
    }
};
template <>
struct RowRecord<2> {
    uint2 v;
    __device__ __forceinline__ void load(const uint8_t *from) { v = *reinterpret_cast<const uint2 *>(from); }
    __device__ __forceinline__ unsigned dword(unsigned d) const { return either(d & 1u, v.x, v.y); }
};
template <>
struct RowRecord<1> {
    unsigned v;
    __device__ __forceinline__ void load(const uint8_t *from) { v = *reinterpret_cast<const unsigned *>(from); }
    __device__ __forceinline__ unsigned dword(unsigned) const { return v; }
};
template <int MODE, int RW>
__global__ __launch_bounds__(kEndWide) void k_map_end(TreeBuffers tb_all, DenseBins bins, TreeEndArgs a, TreeNode *model) {
    constexpr int kNodes = (2 << kSmallDepth) - 1;
    __shared__ short s_leaf[kRowBlock];
    __shared__ float s_value[kNodes];     // what a row adds that ended in the node
    constexpr int kSmallNodes = 1 << (kSmallDepth - 1);  // of the deepest level with split nodes
    __shared__ unsigned char s_flag[kNodes];
    __shared__ int s_scan[kEndWide / 64];
    __shared__ unsigned long long s_folded[kSmallDepth][(kSmallNodes + 63) / 64];  // split nodes that became leaves, a bit each
    __shared__ unsigned long long s_ends[kSmallDepth + 1][2 * (kSmallNodes + 63) / 64];  // leaves, of the tree or folded
    enum { VALID = 1, LEAF = 2, BELOW = 4 };
    TreeBuffers tb = tb_all.for_class(blockIdx.z);
    if (MODE == 1) a.yp += (size_t)blockIdx.z * tb.n;
    const int r0 = blockIdx.x * kRowBlock, r1 = min(tb.n, r0 + kRowBlock);  // (none for the last workgroup)
    constexpr int V = kRowBlock / kEndWide;
    int at[V];
    __shared__ uint2 s_step[RW > 0 ? kNodes : 1];  // x: first bin, bins, split bin, a bit for the default and for a split; y: shift and dword
    RowRecord<(RW > 0 ? RW : 1)> record[V];
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int row = min(r0 + v * kEndWide + (int)threadIdx.x, tb.n - 1);
        if constexpr (RW == 0) {
            at[v] = tb.nid[row];
        } else {
            record[v].load(bins.data + (size_t)row * (RW * 4));
        }
    }
    for (int i = threadIdx.x; i < tb.n_nodes; i += kEndWide) {
        const TreeNode nd = tb.nodes[i];
        if constexpr (RW > 0) {
            uint2 step = make_uint2(0u, 0u);
            if (node_splits(nd)) {  // (see k_split_count)
                unsigned c = (unsigned)nd.split_feature_id, lo = 0, span = kMissingBin;
                if (bins.feat_col != nullptr) {
                    lo = bins.feat_lo[c];
                    span = (unsigned)(tb.cut_row_ptr[c + 1] - tb.cut_row_ptr[c]);
                    c = (unsigned)bins.feat_col[c];
                }
                step = make_uint2(lo | span << 8 | (unsigned)nd.split_bid << 16 | (nd.default_right ? 1u << 24 : 0u) | 1u << 25, (c & 3u) * 8u | (c >> 2) << 8);
            }
            s_step[i] = step;
        }
        s_flag[i] = (unsigned char)((nd.is_valid ? VALID : 0) | (nd.is_leaf ? LEAF : 0) | (nd.gain < a.gamma ? BELOW : 0));
        s_value[i] = nd.base_weight;
    }
    if constexpr (RW > 0) {
        __syncthreads();
#pragma unroll
        for (int v = 0; v < V; ++v) at[v] = 0;
        for (int level = 0; level < tb.depth; ++level) {
            uint2 step[V];
#pragma unroll
            for (int v = 0; v < V; ++v) step[v] = s_step[at[v]];
#pragma unroll
            for (int v = 0; v < V; ++v) {
                const unsigned bin = record[v].dword(step[v].y >> 8) >> (step[v].y & 31u) & 0xffu;
                const int t = (int)bin - (int)(step[v].x & 0xffu);
                const bool right = (unsigned)t >= (step[v].x >> 8 & 0xffu) ? (step[v].x >> 24 & 1u) != 0 : t >= (int)(step[v].x >> 16 & 0xffu);
                at[v] = step[v].x >> 25 ? 2 * at[v] + (right ? 2 : 1) : at[v];  // (heap order)
            }
        }
#pragma unroll
        for (int v = 0; v < V; ++v)
            if (r0 + v * kEndWide + (int)threadIdx.x < r1) tb.nid[r0 + v * kEndWide + (int)threadIdx.x] = at[v];
    }
#pragma unroll
    for (int v = 0; v < V; ++v) {
        const int i = v * kEndWide + (int)threadIdx.x;
        if (r0 + i >= r1) continue;
        int leaf = at[v];
        if (RW == 0 && a.lookup_level >= 0) {  // (that level's split nodes still hold their rows)
            const TreeNode &nd = tb.nodes[leaf];
            if (nd.split_feature_id >= 0 && leaf >= (1 << a.lookup_level) - 1) leaf = end_child_of<false>(tb, bins, CsrBins{}, nd, r0 + i);
        }
        s_leaf[i] = (short)leaf;
    }
    __syncthreads();
    // prune_tree's rule, bottom-up by one wavefront: a bit per node, so that a level is one ballot (64 of its nodes a word)
    if (threadIdx.x < 64) {
        const int lane = lane_id();
        constexpr int kOneWord = 6;  // levels of up to 64 nodes
        auto flags = [&](int level, int k) {
            const int i = k * 64 + lane;
            return i < 1 << level ? (int)s_flag[(1 << level) - 1 + i] : 0;
        };
        int upper[kOneWord + 1];
#pragma unroll
        for (int level = 0; level <= kOneWord; ++level) upper[level] = level <= tb.depth ? flags(level, 0) : 0;
        unsigned long long ends = 0;  // of the level below, where it is one word
        auto fold = [&](int level, int k, int f, unsigned long long below) {
            const bool folds = level < tb.depth && (f & (VALID | LEAF | BELOW)) == (VALID | BELOW) && (below >> (2 * lane & 63) & 3ull) == 3ull;
            const unsigned long long folded = __ballot(folds);
            ends = __ballot((f & (VALID | LEAF)) == (VALID | LEAF)) | folded;
            if (lane == 0) {
                if (level < tb.depth) s_folded[level][k] = folded;
                s_ends[level][k] = ends;
            }
        };
        for (int level = tb.depth; level > kOneWord; --level) {
            for (int k = 0; k < 1 << (level - kOneWord); ++k) fold(level, k, flags(level, k), level < tb.depth ? s_ends[level + 1][2 * k + (lane >> 5)] : 0ull);
            wave_lds_sync();
        }
        if (tb.depth >= kOneWord) fold(kOneWord, 0, upper[kOneWord], tb.depth > kOneWord ? s_ends[kOneWord + 1][lane >> 5] : 0ull);
#pragma unroll
        for (int level = kOneWord - 1; level >= 0; --level)
            if (level <= tb.depth) fold(level, 0, upper[level], lane < 32 ? ends : 0ull);
    }
    __syncthreads();
    auto folded = [&](int x) {  // (any node)
        const int level = 31 - __clz(x + 1), i = x + 1 - (1 << level);
        return level < tb.depth && (s_folded[level][i >> 6] >> (i & 63) & 1ull) != 0;
    };
    // the weight of the first ancestor that was not pruned (tree_builder.cu:62-74): not below a folded node. (Theirs stay as they are.)
    for (int x = threadIdx.x; x < tb.n_nodes; x += kEndWide) {
        int top = x;
        for (int up = x; up > 0;) {
            up = (up - 1) / 2;
            if (!folded(up)) break;
            top = up;
        }
        if (top != x) s_value[x] = s_value[top];
    }
    if (blockIdx.x == gridDim.x - 1) {  // the finished nodes
        model += (size_t)blockIdx.z * tb.n_nodes;
        int carry = 0;
        for (int base = 0; base < tb.n_nodes; base += kEndWide) {
            const int i = base + threadIdx.x;
            const bool in = i < tb.n_nodes;
            const bool pruned = in && i > 0 && folded((i - 1) / 2), leaf = in && ((s_flag[i] & LEAF) || folded(i));
            const bool keep = in && (s_flag[i] & VALID) && !pruned;
            int tot;
            const int ex = block_excl_scan<kEndWide / 64>(keep ? 1 : 0, s_scan, &tot);
            if (in) {
                static_assert(offsetof(TreeNode, final_id) == 0 && offsetof(TreeNode, is_leaf) == 34 && offsetof(TreeNode, is_pruned) == 36,
                              "TreeNode layout");
                const int4 *from = reinterpret_cast<const int4 *>(tb.nodes + i);
                int4 v0 = from[0], v2 = from[2];
                if (keep) v0.x = carry + ex;
                v2.x = (v2.x & ~0x00ff0000) | (leaf ? 1 << 16 : 0);
                v2.y = (v2.y & ~0x000000ff) | (pruned ? 1 : 0);
                int4 *to = reinterpret_cast<int4 *>(model + i);
                to[0] = v0;
                to[1] = from[1];
                to[2] = v2;
            }
            carry += tot;
        }
        return;
    }
    __syncthreads();
    tb.leaf_value = s_value;
    tree_end_rows<MODE, kEndWide>(tb, a, s_leaf, r0, r1);
}

// ---------------------------------------------------------------------------------- metric
// kind 0: sum of squared errors; 1: correct binary decisions (sigmoid > 0.5 in double, like
// multiclass_metric.cu:40); 2: correct arg-max decisions (first maximum wins, :17-29).
__device__ __forceinline__ void metric_row(int kind, int n, int K, int i, float yi, const float *__restrict__ yp,
                                           float p0, double &acc, float &accf) {
    if (kind == 0) {
        float e = p0 - yi;
        accf += e * e;
    } else if (kind == 1) {
        // sigmoid(p) > 0.5 evaluated in double as in the reference; away from zero that is the sign of p
        int k = fabsf(p0) > 1e-6f ? (p0 > 0.f ? 1 : 0) : ((1.0 / (1.0 + exp(-(double)p0)) > 0.5) ? 1 : 0);
        acc += (k == yi) ? 1 : 0;
    } else {
        int mk = 0;
        float mp = p0;
        for (int k = 1; k < K; ++k) {
            float v = yp[(size_t)k * n + i];
            if (v > mp) {
                mp = v;
                mk = k;
            }
        }
        acc += (mk == yi) ? 1 : 0;
    }
}

template <int BLK>
__global__ __launch_bounds__(BLK) void k_metric_partial(int kind, int n, int K, const float *__restrict__ y,
                                                          const float *__restrict__ yp, double *__restrict__ out) {
    __shared__ double sd[BLK / 64];
    double acc = 0;
    float accf = 0;
    const int r0 = blockIdx.x * kRowBlock, r1 = min(n, r0 + kRowBlock);
    for (int i = r0 + threadIdx.x; i < r1; i += BLK) metric_row(kind, n, K, i, y[i], yp, yp[i], acc, accf);
    acc += (double)accf;
    store_block_sum_d<BLK / 64>(acc, sd, out + blockIdx.x);
}

// The counting metrics (kind 1 and 2) do not depend on the order of their additions, so their partials come from
// four times the threads per row block: the class predictions of a row are a chain of dependent-latency loads that
// 256 threads per 4096 rows do not hide.
constexpr int kCountBlock = 1024;
__global__ __launch_bounds__(kCountBlock) void k_metric_count(int kind, int n, int K, const float *__restrict__ y,
                                                             const float *__restrict__ yp, double *__restrict__ out) {
    __shared__ double sd[kCountBlock / 64];
    double acc = 0;
    float accf = 0;
    const int r0 = blockIdx.x * kRowBlock, r1 = min(n, r0 + kRowBlock);
    for (int i = r0 + threadIdx.x; i < r1; i += kCountBlock) metric_row(kind, n, K, i, y[i], yp, yp[i], acc, accf);
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d);
    if (lane_id() == 0) sd[threadIdx.x / 64] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double t = 0;
        for (int i = 0; i < kCountBlock / 64; ++i) t += sd[i];
        out[blockIdx.x] = t;
    }
}

// (the first kBlock threads' work, as tree_init_part)
__device__ void metric_final(int kind, int n, int n_blocks, const double *__restrict__ in, float *__restrict__ out) {
    __shared__ double sd[kWaves];
    const bool on = threadIdx.x < kBlock;
    double acc = 0;
    for (int i = threadIdx.x; on && i < n_blocks; i += kBlock) acc += in[i];
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) acc += __shfl_xor(acc, d);
    if (on && lane_id() == 0) sd[wave_id()] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
        double s = 0;
        for (int i = 0; i < kWaves; ++i) s += sd[i];
        if (kind == 0) {
            out[0] = sqrtf((float)s / n);
        } else {
            float a = (float)s / (float)n;
            out[0] = kind == 1 ? 1.f - a : a;
        }
    }
}

__global__ __launch_bounds__(kBlock) void k_metric_final(int kind, int n, int n_blocks, const double *__restrict__ in,
                                                        float *__restrict__ out) {
    metric_final(kind, n, n_blocks, in, out);
}

int grid_for(size_t n, int cap = 4096) {
    size_t b = (n + kBlock - 1) / kBlock;
    if (b < 1) b = 1;
    if (b > (size_t)cap) b = cap;
    return (int)b;
}

}  // namespace

// =================================================================================== launchers
void launch_fill_f32(hipStream_t s, float *p, float v, size_t n) {
    if (n == 0) return;
    k_fill_f32<<<grid_for(n), kBlock, 0, s>>>(p, v, n);
}

void launch_fill_u8(hipStream_t s, uint8_t *p, uint8_t v, size_t n) {
    // n must be a multiple of 4 (all users allocate padded buffers)
    if (n == 0) return;
    unsigned w = v * 0x01010101u;
    k_fill_u32<<<grid_for(n / 4), kBlock, 0, s>>>(reinterpret_cast<unsigned *>(p), w, n / 4);
}

void launch_gradient(hipStream_t s, int objective, int n, int num_class, const float *y, const float *yp, GHPair *gh,
                     GHPair *, int) {
    if (objective == OBJ_SOFTMAX)
        k_gradient_softmax<<<grid_for(n), kBlock, 0, s>>>(n, num_class, y, yp, gh);
    else
        k_gradient_pointwise<<<grid_for(n), kBlock, 0, s>>>(objective, n, y, yp, gh);
}

void launch_bagging(hipStream_t s, int N, unsigned seed, int *count, GHPair *gh, const int *perm, int n_rows) {
    k_bagging_draw<<<grid_for(N), kBlock, 0, s>>>(N, seed, count);
    k_bagging_apply<<<grid_for(N), kBlock, 0, s>>>(N, count, gh, perm, n_rows);
}

void launch_column_flags(hipStream_t s, const std::vector<unsigned long long> &bits, int F, uint8_t *flags) {
    constexpr int kOf = kColumnFlagWords * 64;
    for (int f0 = 0; f0 < F; f0 += kOf) {
        const int count = std::min(kOf, F - f0), words = (count + 63) / 64;
        ColumnFlags in;
        for (int w = 0; w < words; ++w) in.bits[w] = bits[(size_t)(f0 / 64 + w)];
        for (int w = words; w < kColumnFlagWords; ++w) in.bits[w] = 0;
        k_column_flags<<<(unsigned)((words + kWaves - 1) / kWaves), kBlock, 0, s>>>(in, count, flags + f0);
    }
}

// Launchers: `tb` is the first buffer set to use, `n_class` consecutive sets (class trees of one round)
// are served by the same launch through blockIdx.z; gradient and prediction pointers address the
// first of those classes.
void launch_root_stats(hipStream_t s, const TreeBuffers &tb, const GHPair *gh_class, int n_class) {
    // n_grad_blocks == row_blocks(n)
    k_sum_gh<<<dim3(tb.n_grad_blocks, 1, n_class), kBlock, 0, s>>>(tb.n, gh_class, tb.root_partial);
}

void launch_tree_init(hipStream_t s, const TreeBuffers &tb, const GHPair *gh_class, float lambda, bool stats_ready,
                      int n_class, const TreeLeftovers &left) {
    if (!stats_ready) launch_root_stats(s, tb, gh_class, n_class);
    const int parts = init_parts(tb);
    k_tree_init<<<dim3(parts + (left.metric_out != nullptr ? 1 : 0), 1, n_class), kBlock, 0, s>>>(tb, lambda, left, parts);
    if (tb.nid16 != nullptr) {
        // sparse level pass: every row starts in the root (the n_class maps lie back to back)
        const size_t words = ((size_t)tb.n + 2) / 2 * (size_t)n_class;
        k_fill_u32<<<grid_for(words), kBlock, 0, s>>>(reinterpret_cast<unsigned *>(tb.nid16), 0u, words);
    }
}

template <int LPR, int SLOTS, bool BIN16>
static void hist_dense_launch(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh,
                              int level, int n_class, const HistRoot &root) {
    const int n_pairs = tb.n_hpairs(level);
    // (an upper bound on the work items: whole chunks of the rows that can be built - half of them below the root, unless
    // single nodes are built - and one partly filled item per built node; see plan_hist_item)
    const long rows = level == 0 || tb.singles(level) ? tb.n : tb.n / 2;
    const long by_rows = rows / kHistMinChunk + n_pairs, by_target = std::max(tb.target_hitems, tb.target_hitems / 4 + n_pairs) + 1;
    dim3 grid(bins.n_blocks, (unsigned)std::max(1l, std::min({by_rows, by_target, (long)tb.max_hitems})) + root.init_groups, n_class);
    size_t lds = (size_t)tb.max_block_bins * sizeof(unsigned long long);
    if (lds > 64 * 1024) {
        static LdsOptIn opt_in;
        opt_in({reinterpret_cast<const void *>(&k_hist_dense<LPR, true, kHistBlock, SLOTS, BIN16>),
                reinterpret_cast<const void *>(&k_hist_dense<LPR, false, kHistBlock, SLOTS, BIN16>)});
    }
    if constexpr (!BIN16 && LPR >= 4) {
        if (bins.gh_lane >= 0 && bins.gh_fresh) {
            if (lds > 64 * 1024) {
                static LdsOptIn opt_in_words;
                opt_in_words({reinterpret_cast<const void *>(&k_hist_dense<LPR, true, kHistBlock, SLOTS, BIN16, true>),
                              reinterpret_cast<const void *>(&k_hist_dense<LPR, false, kHistBlock, SLOTS, BIN16, true>)});
            }
            if (level == 0)
                k_hist_dense<LPR, true, kHistBlock, SLOTS, BIN16, true><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, level, n_pairs, root);
            else
                k_hist_dense<LPR, false, kHistBlock, SLOTS, BIN16, true><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, level, n_pairs, 0);
            return;
        }
    }
    if (level == 0)
        k_hist_dense<LPR, true, kHistBlock, SLOTS, BIN16><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, level, n_pairs, root);
    else
        k_hist_dense<LPR, false, kHistBlock, SLOTS, BIN16><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, level, n_pairs, 0);
}

template <int LPR>
static void hist_dense_dispatch(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh,
                                int level, int n_class, const HistRoot &root) {
    const int slots = (tb.max_block_bins + kHistBlock - 1) / kHistBlock;  // bins drained per thread
    if (bins.bin_bytes == 2) {  // (fewer variants: the blocks of 16-bit bins are sized to fill the LDS)
        if (slots <= 4) hist_dense_launch<LPR, 4, true>(s, tb, bins, gh, level, n_class, root);
        else if (slots <= 8) hist_dense_launch<LPR, 8, true>(s, tb, bins, gh, level, n_class, root);
        else if (slots <= 20) hist_dense_launch<LPR, 20, true>(s, tb, bins, gh, level, n_class, root);
        else fatal("feature block with %d bins does not fit the histogram kernel", tb.max_block_bins);
        return;
    }
    if (slots <= 1) hist_dense_launch<LPR, 1, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 2) hist_dense_launch<LPR, 2, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 3) hist_dense_launch<LPR, 3, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 4) hist_dense_launch<LPR, 4, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 6) hist_dense_launch<LPR, 6, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 7) hist_dense_launch<LPR, 7, false>(s, tb, bins, gh, level, n_class, root);  // fewer accumulator registers
    else if (slots <= 8) hist_dense_launch<LPR, 8, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 16) hist_dense_launch<LPR, 16, false>(s, tb, bins, gh, level, n_class, root);
    else if (slots <= 20) hist_dense_launch<LPR, 20, false>(s, tb, bins, gh, level, n_class, root);
    else fatal("feature block with %d bins does not fit the histogram kernel", tb.max_block_bins);
}

void launch_hist_dense(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level,
                       int n_class, bool sum_rows, const TreeLeftovers *init, float lambda) {
    HistRoot root;
    root.sum_rows = sum_rows;
    if (init != nullptr) {
        root.init_parts = init_parts(tb);
        root.init_groups = root.init_parts + (init->metric_out != nullptr ? 1 : 0);
        root.lambda = lambda;
        root.left = *init;
    }
    switch (bins.W * bins.bin_bytes) {  // bytes per row of a block = 4 x lanes per row
        case 4: hist_dense_dispatch<1>(s, tb, bins, gh, level, n_class, root); break;
        case 8: hist_dense_dispatch<2>(s, tb, bins, gh, level, n_class, root); break;
        case 16: hist_dense_dispatch<4>(s, tb, bins, gh, level, n_class, root); break;
        case 32: hist_dense_dispatch<8>(s, tb, bins, gh, level, n_class, root); break;
        case 64: hist_dense_dispatch<16>(s, tb, bins, gh, level, n_class, root); break;
        default: fatal("unsupported dense block width %d x %d bytes", bins.W, bins.bin_bytes);
    }
}

void launch_hist_merge(hipStream_t s, const TreeBuffers &tb, int level, int n_class) {
    const int n_pairs = tb.hpair_hi(level) - tb.hpair_lo(level);  // of the served nodes
    if (tb.target_hitems <= 16) {
        // wide data: many feature blocks, so a node has only a handful of work items and very long histograms;
        // one thread per bin walks them (a block of 8 bins would leave most of its 32 groups without an item)
        dim3 grid((tb.n_bins + kBlock - 1) / kBlock, n_pairs, n_class);
        k_hist_merge<kBlock><<<grid, kBlock, 0, s>>>(tb, level);
    } else if (n_pairs * n_class <= 4) {
        dim3 grid((tb.n_bins + 7) / 8, n_pairs, n_class);
        k_hist_merge<8><<<grid, kBlock, 0, s>>>(tb, level);
    } else {
        dim3 grid((tb.n_bins + 31) / 32, n_pairs, n_class);
        k_hist_merge<32><<<grid, kBlock, 0, s>>>(tb, level);
    }
}

void launch_root_sum(hipStream_t s, const TreeBuffers &tb, const GHPair *gh_class, float lambda, int n_class) {
    if (tb.complete_feature >= 0) {
        k_root_sum_bins<<<dim3(1, 1, n_class), kBlock, 0, s>>>(tb, lambda);
    } else {
        const int blocks = std::max(1, std::min(256, (tb.n + kBlock - 1) / kBlock));
        k_root_sum_rows<<<dim3(blocks, 1, n_class), kBlock, 0, s>>>(tb, gh_class);
        k_root_sum_final<<<dim3(1, 1, n_class), 64, 0, s>>>(tb, blocks, lambda);
    }
}

long device_count_bytes(hipStream_t s, const uint8_t *d_v, size_t n, uint8_t value) {
    unsigned long long *d_out = nullptr, h = 0;
    device_alloc_to(d_out, sizeof(unsigned long long));
    HIP_CHECK(hipMemsetAsync(d_out, 0, sizeof(unsigned long long), s));
    k_count_bytes<<<grid_for(n, 2048), kBlock, 0, s>>>(d_v, n, value, d_out);
    HIP_CHECK(hipMemcpyAsync(&h, d_out, sizeof(h), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    device_free(d_out);
    return (long)h;
}

long device_count_u16(hipStream_t s, const uint16_t *d_v, size_t n, uint16_t value) {
    unsigned long long *d_out = nullptr, h = 0;
    device_alloc_to(d_out, sizeof(unsigned long long));
    HIP_CHECK(hipMemsetAsync(d_out, 0, sizeof(unsigned long long), s));
    k_count_u16<<<grid_for(n, 2048), kBlock, 0, s>>>(d_v, n, value, d_out);
    HIP_CHECK(hipMemcpyAsync(&h, d_out, sizeof(h), hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    device_free(d_out);
    return (long)h;
}

void launch_hist_csr(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const GHPair *gh, int level,
                     int n_class) {
    const int n_pairs = tb.n_hpairs(level);
    const int zgrid = std::min(1024, (tb.n_bins + kBlock - 1) / kBlock);
    k_hist_zero_built<<<dim3(zgrid, tb.hpair_hi(level) - tb.hpair_lo(level), n_class), kBlock, 0, s>>>(tb, level);
    const size_t lds = (size_t)bins.head_bins * 2 * sizeof(unsigned long long);
    if (bins.hist_word != nullptr && lds > 64 * 1024) {
        static LdsOptIn opt_in;
        opt_in({reinterpret_cast<const void *>(&k_hist_csr_head<true>), reinterpret_cast<const void *>(&k_hist_csr_head<false>)});
    }
    if (level == 0 && bins.csc_row != nullptr) {
        const long tiles = (bins.nnz + 63) / 64;
        const int blocks = (int)std::min<long>(8192, (tiles + kWaves - 1) / kWaves);
        if (blocks > 0) k_hist_root_csc<<<dim3(blocks, 1, n_class), kBlock, 0, s>>>(tb, bins, gh);
        return;
    }
    const dim3 grid(tb.max_hitems, 1, n_class);
    if (bins.hist_word != nullptr) {
        if (level == 0) k_hist_csr_head<true><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, n_pairs, level);
        else k_hist_csr_head<false><<<grid, kHistBlock, lds, s>>>(tb, bins, gh, n_pairs, level);
    } else {
        if (level == 0) k_hist_csr<true><<<grid, kBlock, 0, s>>>(tb, bins, gh, n_pairs, level);
        else k_hist_csr<false><<<grid, kBlock, 0, s>>>(tb, bins, gh, n_pairs, level);
    }
    // the sibling histograms (parent - built) are produced by k_eval_split<true>
}

void launch_eval_split(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class,
                       bool store_sibling, bool derive) {
    dim3 grid((tb.n_packs + kWaves - 1) / kWaves, tb.nodes_served(level), n_class);
    if (tb.sparse || derive) k_eval_split<true><<<grid, kBlock, 0, s>>>(tb, level, mcw, lambda, store_sibling);
    else k_eval_split<false><<<grid, kBlock, 0, s>>>(tb, level, mcw, lambda, true);
}

// (as many work items as the level can have, see hist_dense_launch)
static int items_of_level(const TreeBuffers &tb, int level, int run) {
    const int n_pairs = tb.n_hpairs(level);
    if (run > 0 && level > 0) return tb.n / run + n_pairs;
    return std::min(tb.target_hitems, (level == 0 ? tb.n : tb.n / 2) / kHistMinChunk + n_pairs);
}

void launch_merge_eval(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class, bool store, int run) {
    const int n_pairs = tb.n_hpairs(level);
    const dim3 grid(tb.n_packs, n_pairs, n_class);
    const int items = items_of_level(tb, level, run);
    if (level == 0) {
        // One workgroup per pack: with hundreds of items two launches that spread them over the chip are faster (512 items of
        // 28 packs: 12 + 9 instead of 43 us; 245: 8 + 8 and 24; 23 items of 700 packs: 18 instead of 16 + 15).
        if (items > 64) launch_hist_merge(s, tb, level, n_class);
        const dim3 packs((tb.n_packs + kWaves - 1) / kWaves, 1, n_class);
        const bool bins = tb.complete_feature >= 0;
        if (items > 64) {
            if (bins) k_eval_split<false, kRootOfBins><<<packs, kBlock, 0, s>>>(tb, level, mcw, lambda, true);
            else k_eval_split<false, kRootOfRows><<<packs, kBlock, 0, s>>>(tb, level, mcw, lambda, true);
        } else if (items > 8) {
            if (bins) k_merge_eval<16, kRootOfBins><<<grid, 1024, 0, s>>>(tb, level, mcw, lambda, store);
            else k_merge_eval<16, kRootOfRows><<<grid, 1024, 0, s>>>(tb, level, mcw, lambda, store);
        } else {
            if (bins) k_merge_eval<4, kRootOfBins><<<grid, 256, 0, s>>>(tb, level, mcw, lambda, store);
            else k_merge_eval<4, kRootOfRows><<<grid, 256, 0, s>>>(tb, level, mcw, lambda, store);
        }
        return;
    }
    const int per_pair = items / n_pairs;
    if (per_pair > 32) k_merge_eval<16, kNoRoot><<<grid, 1024, 0, s>>>(tb, level, mcw, lambda, store);
    else if (per_pair > 8) k_merge_eval<8, kNoRoot><<<grid, 512, 0, s>>>(tb, level, mcw, lambda, store);
    else if (per_pair > 2) k_merge_eval<4, kNoRoot><<<grid, 256, 0, s>>>(tb, level, mcw, lambda, store);
    else k_merge_eval<2, kNoRoot><<<grid, 128, 0, s>>>(tb, level, mcw, lambda, store);
}

void launch_eval_split_wide(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class,
                            bool store_sibling, bool derive, bool root_of_rows) {
    dim3 grid(tb.F, tb.nodes_served(level), n_class);
    k_eval_split_wide<<<grid, kBlock, 0, s>>>(tb, level, mcw, lambda, store_sibling, derive || tb.sparse, root_of_rows);
}

void launch_merge_eval_wide(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class, bool store, int run,
                            int max_feature_bins) {
    const int n_pairs = tb.n_hpairs(level), per_pair = items_of_level(tb, level, run) / n_pairs;
    const dim3 grid(tb.F, n_pairs, n_class);
    // (many items of few pairs are for launches that spread them over the chip, see launch_merge_eval's root)
    if (max_feature_bins > kMergeWideBins || per_pair > 64) {
        launch_hist_merge(s, tb, level, n_class);
        launch_eval_split_wide(s, tb, level, mcw, lambda, n_class, store, false, false);
    } else if (per_pair > 8) k_merge_eval_wide<16><<<grid, 1024, 0, s>>>(tb, level, mcw, lambda, store);
    else k_merge_eval_wide<8><<<grid, 512, 0, s>>>(tb, level, mcw, lambda, store);
}

void launch_best_update(hipStream_t s, const TreeBuffers &tb, int level, float rt_eps, float lambda, int n_class) {
    k_best_update<<<dim3(tb.nodes_served(level), 1, n_class), kBlock, 0, s>>>(tb, level, rt_eps, lambda);
}

void launch_partition_csr(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, int level, int n_class) {
    if (level == tb.depth - 1) return;
    const dim3 one(1, 1, n_class), items(tb.max_pitems, 1, n_class);
    if (level == 0) {
        k_part_count_csr<true><<<items, kBlock, 0, s>>>(tb, bins, level);
        k_part_scan_plan<<<one, kBlock, 0, s>>>(tb, level);
        k_part_scatter<true><<<items, kBlock, 0, s>>>(tb, level);
    } else {
        k_part_count_csr<false><<<items, kBlock, 0, s>>>(tb, bins, level);
        k_part_scan_plan<<<one, kBlock, 0, s>>>(tb, level);
        k_part_scatter<false><<<items, kBlock, 0, s>>>(tb, level);
    }
}

template <bool SPARSE>
static void tree_end_launch(hipStream_t s, const TreeBuffers &tb, const DenseBins &d, const CsrBins &c, int mode,
                            const TreeEndArgs &a, int n_class) {
    const dim3 grid(row_blocks(tb.n), 1, n_class);
    // (mode 0 has nothing per row to wait for)
    if (mode == 0) k_tree_end<0, SPARSE, kBlock><<<grid, kBlock, 0, s>>>(tb, d, c, a);
    else if (mode == 1 && end_wide(tb.n, n_class)) k_tree_end<1, SPARSE, kEndWide><<<grid, kEndWide, 0, s>>>(tb, d, c, a);
    else if (mode == 1) k_tree_end<1, SPARSE, kBlock><<<grid, kBlock, 0, s>>>(tb, d, c, a);
    else if (end_wide(tb.n)) k_tree_end<2, SPARSE, kEndWide><<<grid, kEndWide, 0, s>>>(tb, d, c, a);
    else k_tree_end<2, SPARSE, kBlock><<<grid, kBlock, 0, s>>>(tb, d, c, a);
}

static void tree_end(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins, int mode,
                     const TreeEndArgs &a, int n_class = 1) {
    const int n_blocks = row_blocks(tb.n);
    const size_t entries = (size_t)((1 << tb.depth) - 1) * (n_blocks + 1);
    if (tb.nid16 == nullptr)
        k_end_bounds<<<dim3(grid_for(entries, 8192) + (a.with_prune ? 1 : 0), 1, n_class), kBlock, 0, s>>>(
            tb, a.lookup_level, n_blocks, a.with_prune, a.gamma);
    else if (a.with_prune)
        k_prune<<<dim3(1, 1, n_class), kBlock, 0, s>>>(tb, a.gamma);
    if (tb.sparse) tree_end_launch<true>(s, tb, DenseBins{}, *cbins, mode, a, n_class);
    else tree_end_launch<false>(s, tb, *dbins, CsrBins{}, mode, a, n_class);
}

void launch_nid_rebuild(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins,
                        int lookup_level) {
    TreeEndArgs a{};
    a.lookup_level = lookup_level;
    tree_end(s, tb, dbins, cbins, 0, a);
}

void launch_predict_in_training(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins,
                                int lookup_level, float *yp_class, float lr, int n_class, const float *prune_gamma) {
    TreeEndArgs a{};
    a.lookup_level = lookup_level;
    a.yp = yp_class;
    a.lr = lr;
    a.with_prune = prune_gamma != nullptr;
    a.gamma = prune_gamma != nullptr ? *prune_gamma : 0.f;
    tree_end(s, tb, dbins, cbins, 1, a, n_class);
}

void launch_round_end(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins,
                      int lookup_level, int objective, int metric_kind, const float *y, float *yp, float lr,
                      GHPair *gh, double *metric_scratch, const float *prune_gamma, unsigned *gh_words) {
    TreeEndArgs a{};
    a.gh_words = gh_words;
    a.with_prune = prune_gamma != nullptr;
    a.gamma = prune_gamma != nullptr ? *prune_gamma : 0.f;
    a.lookup_level = lookup_level;
    a.y = y;
    a.yp = yp;
    a.lr = lr;
    a.objective = objective;
    a.metric_kind = metric_kind;
    a.gh = gh;
    a.stats = tb.root_partial;
    a.metric_partial = metric_scratch;
    tree_end(s, tb, dbins, cbins, 2, a);
}

void launch_map_end(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, int lookup_level, TreeNode *model, float gamma, float *yp,
                      float lr, int n_class, const float *y, int objective, int metric_kind, GHPair *gh,
                      double *metric_scratch, unsigned *gh_words, bool walk) {
    TreeEndArgs a{};
    a.lookup_level = lookup_level;
    a.gamma = gamma;
    a.yp = yp;
    a.lr = lr;
    a.y = y;
    a.objective = objective;
    a.metric_kind = metric_kind;
    a.gh = gh;
    a.stats = tb.root_partial;
    a.metric_partial = metric_scratch;
    a.gh_words = gh_words;
    const dim3 grid(row_blocks(tb.n) + 1, 1, n_class);  // (the last one writes the model)
    if (y != nullptr) return k_map_end<2, 0><<<grid, kEndWide, 0, s>>>(tb, bins, a, model);
    switch (walk ? bins.W : 0) {  // (bytes of a record: split_hist_plan)
        case 0: return k_map_end<1, 0><<<grid, kEndWide, 0, s>>>(tb, bins, a, model);
        case 4: return k_map_end<1, 1><<<grid, kEndWide, 0, s>>>(tb, bins, a, model);
        case 8: return k_map_end<1, 2><<<grid, kEndWide, 0, s>>>(tb, bins, a, model);
        case 16: return k_map_end<1, 4><<<grid, kEndWide, 0, s>>>(tb, bins, a, model);
        case 32: return k_map_end<1, 8><<<grid, kEndWide, 0, s>>>(tb, bins, a, model);
        default: fatal("a walk over records of %d bytes", bins.W);
    }
}

void launch_metric_final(hipStream_t s, int n, const TreeLeftovers &left) {
    k_metric_final<<<1, kBlock, 0, s>>>(left.metric_kind, n, left.metric_blocks, left.metric_partial, left.metric_out);
}

void launch_gh_words(hipStream_t s, int objective, int n, const float *y, const float *yp, unsigned *words) {
    if (n <= 0) return;
    k_gh_words<<<std::min(4096, (n + kBlock - 1) / kBlock), kBlock, 0, s>>>(objective, n, y, yp, words);
}

void launch_metric(hipStream_t s, int kind, int n, int num_class, const float *y, const float *yp, double *scratch) {
    int blocks = row_blocks(n);  // scratch: one double per block
    if (kind == 0)
        end_wide(n) ? k_metric_partial<kEndWide><<<blocks, kEndWide, 0, s>>>(kind, n, num_class, y, yp, scratch)
                    : k_metric_partial<kBlock><<<blocks, kBlock, 0, s>>>(kind, n, num_class, y, yp, scratch);
    else
        k_metric_count<<<blocks, kCountBlock, 0, s>>>(kind, n, num_class, y, yp, scratch);
}

}  // namespace tgbm
