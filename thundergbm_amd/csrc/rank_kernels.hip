// LambdaRank gradients and the list metrics MAP / NDCG on the device.
//
// The reference computes these on the host, one query group per OpenMP iteration
// (src/thundergbm/objective/ranking_obj.cpp:20-96, src/thundergbm/metric/rank_metric.cpp:9-104). Here a
// round is a handful of data-parallel passes over all rows:
//   * labels never change, so the label-descending order of every group, its runs of equal labels and the
//     part of each run that draws partners are tables built once (k_rank_setup; on the host where groups are long);
//   * per round a workgroup per group (k_rank_gradient_group), or one stable radix sort of (run, descending score) keys
//     where groups are long, orders the rows inside their runs, which reproduces "sort by score, then stably by label";
//   * one thread per position draws its partner, evaluates the pair and adds the lambdas to both rows with
//     64-bit fixed-point atomics (exact integer sums: the result does not depend on the order of the adds).
// Two things differ from the reference by necessity, because there they are not reproducible: ties between
// equal scores keep the row order (std::sort leaves it unspecified), and the partner of a position is a
// pure function of (round seed, position) instead of a std::mt19937 stream seeded with std::rand() from
// whichever thread reaches the group first.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <string>
#include <thread>

#include "rank.h"

namespace tgbm {
namespace {

constexpr int kBlock = 256;

// Order-preserving map float -> uint32 (-0.0 folded into +0.0: they compare equal).
__device__ __forceinline__ unsigned float_key(float v) {
    if (v == 0.f) v = 0.f;
    unsigned u = __float_as_uint(v);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}

// Partner draw of position `pos` in round `seed`: a 64-bit finaliser of the pair, scaled to [0, range).
__device__ __forceinline__ unsigned rank_draw(unsigned seed, unsigned pos, unsigned range) {
    unsigned long long x = ((unsigned long long)seed << 32) | pos;
    x += 0x9E3779B97F4A7C15ull;
    x = (x ^ (x >> 30)) * 0xBF58476D1CE4E5B9ull;
    x = (x ^ (x >> 27)) * 0x94D049BB133111EBull;
    x ^= x >> 31;
    return (unsigned)(((x >> 32) * (unsigned long long)range) >> 32);
}

// NDCG::discounted_gain (include/thundergbm/metric/ranking_metric.h:43-45)
__device__ __forceinline__ float discounted_gain(int label, int rank) {
    return (float)((1 << label) - 1) / log2f((float)(rank + 2));
}

// bits of the fixed-point fraction for a group of `len` rows: a row collects at most len + 1 lambdas of
// magnitude <= 2, so sums stay below 2^62
__device__ __forceinline__ int acc_bits(int len) { return 59 - (32 - __clz(max(len, 1))); }

// The tables of a group whose rows one workgroup orders by counting: its rows by label descending, the runs of equal labels
// (numbered by the position of the group's first row + the run's number in the group: ascending, with gaps), the positions that
// draw partners, IDCG and the number of rows with a label. NaNs are ordered as their bits are, each a run of its own.
// log2_of[i] = log2(i + 2) as the host has it: the terms of IDCG and their sum are its own, bit for bit.
// Bound by the counting (len^2 steps of LDS a group). 200 003 rows in 1667 groups: 22 us, where eight threads of the host, the
// copies of their tables and the look at the labels took 1.7 ms (a call of 40 rounds 20.5 -> 19.4 ms).
constexpr int kSetupBlock = 128;
// Threads of the rounds' kernels: 64 where no group is longer than 64 rows, 128 for groups of up to 256 and where they share workgroups, 512
// for longer ones. Those have a launch of their own, so that the others don't ask for LDS for the longest group, and sort in LDS: counting 2000 rows is
// 2000 steps for each of four rows a thread, 95 us a round for one such group among 19 800 of ten rows (200 k x 20, 20 rounds: 12.5 -> 7.1 ms).
constexpr int kPackBlock = 128, kLongGroupBlock = 512;
constexpr size_t kRankGroupBytes = 2 * sizeof(unsigned long long) + 2 * sizeof(int) + sizeof(float);  // LDS of k_rank_gradient_group per row
__global__ __launch_bounds__(kSetupBlock) void k_rank_setup(const float *__restrict__ y, const int *__restrict__ gptr,
                                                            const float *__restrict__ log2_of, int longest, int *__restrict__ static_row,
                                                            int *__restrict__ run_of, int *__restrict__ group_of, RankRun *__restrict__ runs,
                                                            float *__restrict__ idcg, int *__restrict__ hits, int *__restrict__ counts) {
    extern __shared__ unsigned s_mem[];
    __shared__ int s_hits, s_bad, s_runs;
    unsigned *s_key = s_mem;                                          // keys by row, then IDCG's terms by position
    float *s_sorted = reinterpret_cast<float *>(s_key + longest);    // labels by position
    unsigned short *s_run = reinterpret_cast<unsigned short *>(s_sorted + longest);  // run of a position, within the group
    unsigned short *s_first = s_run + longest;                       // first position of a run; the top bit: it draws no partner
    const int g = blockIdx.x, b = gptr[g], len = gptr[g + 1] - b;
    if (threadIdx.x == 0) s_hits = s_bad = s_runs = 0;
    __syncthreads();
    int nonzero = 0, bad = 0;
    for (int i = threadIdx.x; i < len; i += kSetupBlock) {
        const float v = y[b + i];
        s_key[i] = float_key(v);
        group_of[b + i] = g;
        nonzero += v != 0.f ? 1 : 0;
        bad |= v >= 0.f && v < 31.f ? 0 : 1;
    }
    if (nonzero) atomicAdd(&s_hits, nonzero);
    if (bad) s_bad = 1;
    __syncthreads();
    for (int i = threadIdx.x; i < len; i += kSetupBlock) {
        const unsigned key = s_key[i];
        int before = 0;
        for (int j = 0; j < len; ++j) before += s_key[j] > key || (s_key[j] == key && j < i) ? 1 : 0;
        s_sorted[before] = y[b + i];
        static_row[b + before] = b + i;
    }
    __syncthreads();
    bad = s_bad;
    for (int i = threadIdx.x; i < len; i += kSetupBlock) {
        const float term = bad ? 0.f : (float)((1 << (int)s_sorted[i]) - 1) / log2_of[i];
        s_key[i] = __float_as_uint(term);
    }
    if (threadIdx.x < 64) {  // the runs, by one wavefront
        const int lane = threadIdx.x;
        int n_runs = 0;
        for (int base = 0; base < len; base += 64) {
            const int i = base + lane;
            const bool first = i < len && (i == 0 || s_sorted[i] != s_sorted[i - 1]);
            const unsigned long long firsts = __ballot(first);
            const int k = n_runs + __popcll(firsts & (~0ull >> (63 - lane))) - 1;
            if (i < len) s_run[i] = (unsigned short)k;
            if (first) s_first[k] = (unsigned short)i;
            n_runs += __popcll(firsts);
        }
        if (lane == 0) s_runs = n_runs;
    }
    __syncthreads();
    const int n_runs = s_runs;
    if (threadIdx.x == 0) {  // a processed run makes the loop step over the next run's first position
        bool skip = false;
        int first = 0;
        for (int k = 0; k < n_runs; ++k) {
            const int end = k + 1 < n_runs ? s_first[k + 1] : len;
            if (skip) s_first[k] = (unsigned short)(first | 0x8000);
            skip = first + (skip ? 1 : 0) < end;
            first = end;
        }
    }
    if (threadIdx.x == 64) {
        float z = 0.f;
        for (int i = 0; i < len; ++i) z += __uint_as_float(s_key[i]);
        idcg[g] = z;
        hits[g] = s_hits;
        if (s_bad) atomicOr(&counts[0], 1);
        if (z == 0.f) atomicAdd(&counts[1], 1);
        if (s_hits == 0) atomicAdd(&counts[2], 1);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < n_runs; k += kSetupBlock) {
        RankRun r;
        r.group_begin = b;
        r.group_end = b + len;
        r.begin = b + (s_first[k] & 0x7fff);
        r.end = b + (k + 1 < n_runs ? s_first[k + 1] & 0x7fff : len);
        r.first_l = min(r.end, r.begin + (s_first[k] >> 15));
        r.group = g;
        runs[b + k] = r;
    }
    for (int i = threadIdx.x; i < len; i += kSetupBlock) run_of[b + i] = b + s_run[i];
}

int grid_for(size_t n) {
    size_t b = (n + kBlock - 1) / kBlock;
    return (int)std::max<size_t>(1, b);
}

__global__ __launch_bounds__(kBlock) void k_rank_train_keys(int n, const int *__restrict__ static_row,
                                                           const int *__restrict__ run_of,
                                                           const float *__restrict__ score,
                                                           unsigned long long *__restrict__ keys, int *__restrict__ vals) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    const int row = static_row[p];
    keys[p] = ((unsigned long long)(unsigned)run_of[p] << 32) | (unsigned)~float_key(score[row]);
    vals[p] = row;
}

// Keys for the short re-sort of rows that are already in (group, score) order: the run id alone.
__global__ __launch_bounds__(kBlock) void k_rank_run_keys(int n, const int *__restrict__ run_of_row,
                                                         const int *sorted_row, unsigned long long *__restrict__ keys,
                                                         int *vals) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    const int row = sorted_row[p];  // may alias vals: every thread reads and writes its own element
    keys[p] = (unsigned long long)(unsigned)run_of_row[row];
    vals[p] = row;
}

__global__ __launch_bounds__(kBlock) void k_rank_metric_keys(int n, const int *__restrict__ group_of,
                                                            const float *__restrict__ score,
                                                            unsigned long long *__restrict__ keys, int *__restrict__ vals) {
    const int row = blockIdx.x * kBlock + threadIdx.x;
    if (row >= n) return;
    keys[row] = ((unsigned long long)(unsigned)group_of[row] << 32) | (unsigned)~float_key(score[row]);
    vals[row] = row;
}

// The body of the inner loop of LambdaRank::get_gradient (ranking_obj.cpp:63-90) for position p of the (label descending, score
// descending) order of its group: its partner, and what the pair adds to the row nearer the top of the label order (the other
// one gets the gradient's opposite). idcg: of the group, nullptr: rank:pairwise.
struct RankPair {
    int high, low;  // positions inside the group
    long long ql;
    unsigned long long qh;
};
__device__ __forceinline__ bool draw_partner(const RankRun &r, int p, unsigned seed, RankPair &pair) {
    if (p < r.first_l) return false;
    const int nleft = r.first_l - r.group_begin;
    const int nright = r.group_end - r.end;
    if (nleft + nright == 0) return false;
    const int m = (int)rank_draw(seed, (unsigned)p, (unsigned)(nleft + nright));
    const int l = p - r.group_begin;
    const bool left = m < nleft;
    pair.high = left ? m : l;
    pair.low = left ? l : m - nleft + (r.end - r.group_begin);
    return true;
}
__device__ __forceinline__ void weigh_pair(RankPair &pair, const float *idcg, float label_high, float label_low, float score_high,
                                           float score_low, int group_rows) {
    float dz = 1.f;  // LambdaRank::get_delta_z
    if (idcg != nullptr) {  // LambdaRankNDCG::get_delta_z (ranking_obj.cpp:105-113)
        const float z = *idcg;
        if (z == 0.f) {
            dz = 0.f;
        } else {
            const int li = (int)label_high, lj = (int)label_low;
            dz = (discounted_gain(li, pair.high) + discounted_gain(lj, pair.low) - discounted_gain(li, pair.low) -
                  discounted_gain(lj, pair.high)) / z;
        }
    }
    const float adz = fabsf(dz);
    const float rho = 1.f / (1.f + expf(score_high - score_low));
    const float lambda = -adz * rho;
    const float hess = 2.f * fmaxf(adz * rho * (1.f - rho), 1e-16f);
    const int sb = acc_bits(group_rows);
    pair.ql = __double2ll_rn(ldexp((double)lambda, sb));
    pair.qh = (unsigned long long)__double2ll_rn(ldexp((double)hess, sb));
}
__device__ __forceinline__ GHPair pair_of_sums(long long g, long long h, int group_rows) {
    const int sb = acc_bits(group_rows);
    return GHPair{(float)ldexp((double)g, -sb), (float)ldexp((double)h, -sb)};
}

// Groups of at most kRankCountSortMax rows: a workgroup has a group to itself, or several short ones (rank_packs.h), orders it in LDS, by
// counting up to 256 rows, and adds the lambdas up there. Bound by the counting, len^2 steps of LDS a group. 200 003 rows in 1667 groups of
// about 120: the order by score 15 us (keys and counting through the L1: 4.6 and 16.3), the gradients 13 (keys, counting, pairs with four
// 64-bit atomics a row, sums: 4.9, 11, 28, 5.2).
// Keys read four at a time, or eight ahead: 15, 27 us.
__device__ __forceinline__ int rows_before(const unsigned *s_key, int from, int to, unsigned key, int at) {
    int before = 0;
    for (int j = from; j < to; ++j) {
        const unsigned k = s_key[j];
        before += k < key || (k == key && j < at) ? 1 : 0;
    }
    return before;
}

// Ascending order of count (a power of two) keys of the workgroup, by a bitonic network; the caller has waited for them.
template <int BLK>
__device__ __forceinline__ void sort_keys(unsigned long long *s, int count) {
    for (int k = 2; k <= count; k <<= 1)
        for (int j = k >> 1; j > 0; j >>= 1) {
            for (int p = threadIdx.x; p < count / 2; p += BLK) {
                const int a = 2 * p - (p & (j - 1));
                const unsigned long long x = s[a], z = s[a + j];
                if ((x > z) == ((a & k) == 0)) {
                    s[a] = z;
                    s[a + j] = x;
                }
            }
            __syncthreads();
        }
}
__host__ __device__ inline int keys_to_sort(int len) {  // fewer than 2 len
    int count = 1;
    while (count < len) count <<= 1;
    return count;
}

// sorted: the rows of every group by score descending, ties by row. SHARED: some packs are of several groups.
template <int BLK, bool SHARED>
__global__ __launch_bounds__(BLK) void k_rank_order_group(const RankPack *__restrict__ packs, const int *__restrict__ gptr,
                                                          const int *__restrict__ group_of, const float *__restrict__ score,
                                                          int *__restrict__ sorted) {
    extern __shared__ unsigned long long s_order[];  // [keys_to_sort(rows)], as unsigned [rows] where they are counted
    const RankPack pack = packs[blockIdx.x];
    const int b = pack.begin, len = pack.end - b;
    if (BLK == kLongGroupBlock) {
        const int count = keys_to_sort(len);
        for (int i = threadIdx.x; i < count; i += BLK)
            s_order[i] = i < len ? (unsigned long long)~float_key(score[b + i]) << 32 | (unsigned)i : ~0ull;
        __syncthreads();
        sort_keys<BLK>(s_order, count);
        for (int i = threadIdx.x; i < len; i += BLK) sorted[b + i] = b + (int)(unsigned)s_order[i];
        return;
    }
    unsigned *s_key = reinterpret_cast<unsigned *>(s_order);
    for (int i = threadIdx.x; i < len; i += BLK) s_key[i] = ~float_key(score[b + i]);
    __syncthreads();
    for (int i = threadIdx.x; i < len; i += BLK) {
        int from = 0, to = len;
        if (SHARED) {
            const int g = group_of[b + i];
            from = gptr[g] - b;
            to = gptr[g + 1] - b;
        }
        sorted[b + from + rows_before(s_key, from, to, s_key[i], i)] = b + i;
    }
}

// Rows inside their runs of equal labels by score descending, ties by row (static_row ascends inside a run), then every position's pair.
template <int BLK, bool SHARED>
__global__ __launch_bounds__(BLK) void k_rank_gradient_group(const RankPack *__restrict__ packs, int most, const float *__restrict__ score,
                                                             const float *__restrict__ y,
                                                             const int *__restrict__ static_row, const int *__restrict__ run_of,
                                                             const RankRun *__restrict__ runs, const float *__restrict__ idcg, unsigned seed,
                                                             int *__restrict__ sorted, GHPair *__restrict__ gh) {
    extern __shared__ unsigned long long s_acc[];  // [2 most] by row (most: rows of a workgroup of the launch)
    unsigned *s_key = reinterpret_cast<unsigned *>(s_acc + 2 * most);  // by position of static_row
    int *s_row = reinterpret_cast<int *>(s_key + most);                // by position of the order, within the workgroup
    float *s_score = reinterpret_cast<float *>(s_row + most);
    const RankPack pack = packs[blockIdx.x];
    const int b = pack.begin, len = pack.end - b;
    if (BLK == kLongGroupBlock) {  // (run, key, position) where the sums will be
        static_assert(kRankCountSortMax <= 1 << 12, "positions of a group in 12 bits");
        const int count = keys_to_sort(len);
        for (int i = threadIdx.x; i < count; i += BLK)
            s_acc[i] = i < len ? (unsigned long long)(run_of[b + i] - b) << 44 | (unsigned long long)~float_key(score[static_row[b + i]]) << 12 | (unsigned)i : ~0ull;
        __syncthreads();
        sort_keys<BLK>(s_acc, count);
        for (int at = threadIdx.x; at < len; at += BLK) {
            const int row = static_row[b + (int)(s_acc[at] & 4095u)];
            s_row[at] = row - b;
            s_score[at] = score[row];
            sorted[b + at] = row;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < len; i += BLK) s_acc[2 * i] = s_acc[2 * i + 1] = 0ull;
    } else {
        for (int i = threadIdx.x; i < len; i += BLK) {
            s_key[i] = ~float_key(score[static_row[b + i]]);
            s_acc[2 * i] = s_acc[2 * i + 1] = 0ull;
        }
        __syncthreads();
        for (int i = threadIdx.x; i < len; i += BLK) {
            const RankRun r = runs[run_of[b + i]];
            const int row = static_row[b + i], at = r.begin - b + rows_before(s_key, r.begin - b, r.end - b, s_key[i], i);
            s_row[at] = row - b;
            s_score[at] = score[row];
            sorted[b + at] = row;
        }
    }
    __syncthreads();
    for (int i = threadIdx.x; i < len; i += BLK) {
        const RankRun r = runs[run_of[b + i]];
        RankPair pair;
        if (!draw_partner(r, b + i, seed, pair)) continue;
        const int at = SHARED ? r.group_begin - b : 0, high = s_row[at + pair.high], low = s_row[at + pair.low];
        weigh_pair(pair, idcg != nullptr ? idcg + (SHARED ? r.group : pack.group) : nullptr, y[b + high], y[b + low],
                   s_score[at + pair.high], s_score[at + pair.low], SHARED ? r.group_end - r.group_begin : len);
        atomicAdd(&s_acc[2 * high], (unsigned long long)pair.ql);
        atomicAdd(&s_acc[2 * high + 1], pair.qh);
        atomicAdd(&s_acc[2 * low], (unsigned long long)(-pair.ql));
        atomicAdd(&s_acc[2 * low + 1], pair.qh);
    }
    __syncthreads();
    for (int i = threadIdx.x; i < len; i += BLK) {
        int rows = len;
        if (SHARED) {  // (the run at a row's place: of the row's group)
            const RankRun r = runs[run_of[b + i]];
            rows = r.group_end - r.group_begin;
        }
        gh[b + i] = pair_of_sums((long long)s_acc[2 * i], (long long)s_acc[2 * i + 1], rows);
    }
}

// One thread per position, for groups of any length.
__global__ __launch_bounds__(kBlock) void k_rank_pairs(int n, const RankRun *__restrict__ runs,
                                                      const int *__restrict__ run_of, const int *__restrict__ sorted_row,
                                                      const float *__restrict__ score, const float *__restrict__ y,
                                                      const float *__restrict__ idcg, unsigned seed,
                                                      unsigned long long *__restrict__ acc) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p >= n) return;
    const RankRun r = runs[run_of[p]];
    RankPair pair;
    if (!draw_partner(r, p, seed, pair)) return;
    const int high_row = sorted_row[r.group_begin + pair.high], low_row = sorted_row[r.group_begin + pair.low];
    weigh_pair(pair, idcg != nullptr ? idcg + r.group : nullptr, y[high_row], y[low_row], score[high_row], score[low_row], r.group_end - r.group_begin);
    atomicAdd(acc + 2 * (size_t)high_row, (unsigned long long)pair.ql);
    atomicAdd(acc + 2 * (size_t)high_row + 1, pair.qh);
    atomicAdd(acc + 2 * (size_t)low_row, (unsigned long long)(-pair.ql));
    atomicAdd(acc + 2 * (size_t)low_row + 1, pair.qh);
}

// fixed point -> GHPair, and the accumulators are cleared for the next round
__global__ __launch_bounds__(kBlock) void k_rank_finish(int n, const int *__restrict__ group_of,
                                                       const int *__restrict__ gptr, long long *__restrict__ acc,
                                                       GHPair *__restrict__ gh) {
    const int row = blockIdx.x * kBlock + threadIdx.x;
    if (row >= n) return;
    const int g = group_of[row];
    gh[row] = pair_of_sums(acc[2 * (size_t)row], acc[2 * (size_t)row + 1], gptr[g + 1] - gptr[g]);
    acc[2 * (size_t)row] = 0;
    acc[2 * (size_t)row + 1] = 0;
}

// Sum of a block's per-thread doubles in thread order (the same bits on every run).
__device__ __forceinline__ void store_block_sum(double v, double *__restrict__ out) {
    __shared__ double s[kBlock];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) out[blockIdx.x] = s[0];
}

// NDCG::eval_query_group (rank_metric.cpp:81-104): position p of the score order adds gain / IDCG of its group.
__global__ __launch_bounds__(kBlock) void k_rank_ndcg_partial(int n, const int *__restrict__ sorted_row,
                                                             const int *__restrict__ group_of,
                                                             const int *__restrict__ gptr, const float *__restrict__ y,
                                                             const float *__restrict__ idcg,
                                                             double *__restrict__ partial) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    double c = 0;
    if (p < n) {
        const int g = group_of[p];  // groups are runs of consecutive rows, so position p lies in row p's group
        const float z = idcg[g];
        if (z != 0.f) c = (double)discounted_gain((int)y[sorted_row[p]], p - gptr[g]) / (double)z;
    }
    store_block_sum(c, partial);
}

__global__ __launch_bounds__(kBlock) void k_rank_hit_flags(int n, const int *__restrict__ sorted_row,
                                                          const float *__restrict__ y, unsigned *__restrict__ flags) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    if (p < n) flags[p] = y[sorted_row[p]] != 0.f ? 1u : 0u;
}

// MAP::eval_query_group (rank_metric.cpp:47-72): a hit at rank i adds (hits so far) / (i + 1) / (hits of the group).
__global__ __launch_bounds__(kBlock) void k_rank_map_partial(int n, const unsigned *__restrict__ flags,
                                                            const unsigned *__restrict__ hits_before,
                                                            const int *__restrict__ group_of,
                                                            const int *__restrict__ gptr,
                                                            const int *__restrict__ group_hits,
                                                            double *__restrict__ partial) {
    const int p = blockIdx.x * kBlock + threadIdx.x;
    double c = 0;
    if (p < n && flags[p] != 0u) {
        const int g = group_of[p];
        const int b = gptr[g];
        const unsigned nh = hits_before[p] - hits_before[b] + 1u;
        c = (double)nh / (double)(p - b + 1) / (double)group_hits[g];
    }
    store_block_sum(c, partial);
}

// (sum of the partials + groups that score 1 by definition) / number of groups; one workgroup, fixed order
__global__ __launch_bounds__(kBlock) void k_rank_metric_final(const double *__restrict__ partial, int n_partial,
                                                             double constant, int n_groups, float *__restrict__ out) {
    __shared__ double s[kBlock];
    double v = 0;
    for (int i = threadIdx.x; i < n_partial; i += kBlock) v += partial[i];
    s[threadIdx.x] = v;
    __syncthreads();
    for (int w = kBlock / 2; w > 0; w >>= 1) {
        if ((int)threadIdx.x < w) s[threadIdx.x] += s[threadIdx.x + w];
        __syncthreads();
    }
    if (threadIdx.x == 0) *out = (float)((s[0] + constant) / (double)n_groups);
}

int bits_for(long count) {
    int b = 0;
    while ((1l << b) < count) ++b;
    return b;
}

}  // namespace

template <typename T>
T *RankContext::dalloc(size_t count) {
    void *p = nullptr;
    device_alloc_to(p, sizeof(T) * std::max<size_t>(count, 1));
    allocs_.push_back(p);
    return static_cast<T *>(p);
}

RankContext::RankContext(hipStream_t s, const LabelVector &y, const float *d_y, const std::vector<int> &group, bool ndcg)
    : stream_(s), ndcg_(ndcg), d_y_(d_y) {
    n_ = (int)y.size();
    n_groups_ = (int)group.size();
    TGBM_CHECK(n_groups_ > 0, "ranking needs query groups (a .group file or the group argument)");
    std::vector<int> gptr(n_groups_ + 1, 0);  // RankListMetric::configure_gptr (rank_metric.cpp:39-44)
    for (int g = 0; g < n_groups_; ++g) {
        TGBM_CHECK(group[g] >= 0, "negative size of query group %d", g);
        TGBM_CHECK((long)gptr[g] + group[g] <= (long)n_, "query groups cover more than the %d instances", n_);
        gptr[g + 1] = gptr[g] + group[g];
    }
    TGBM_CHECK(gptr.back() == n_, "query groups cover %d instances, the dataset has %d", gptr.back(), n_);

    int longest = 0;
    double steps = 0;
    for (int g : group) {
        longest = std::max(longest, g);
        steps += (double)g * (double)g;
    }
    const char *sort_env = std::getenv("TGBM_RANK_SORT");  // "radix": the radix sort whatever the group sizes (tests)
    short_groups_ = longest <= kRankCountSortMax && steps <= (double)kRankCountSortMean * (double)std::max(n_, 1) &&
                    !(sort_env != nullptr && std::string(sort_env) == "radix");
    group_bits_ = bits_for(n_groups_);
    if (d_y_ == nullptr) {
        float *own = dalloc<float>(n_);
        upload(own, y.data(), sizeof(float) * (size_t)n_);
        d_y_ = own;
    }
    d_static_row_ = dalloc<int>(n_);
    d_run_of_ = dalloc<int>(n_);
    d_group_of_ = dalloc<int>(n_);
    d_gptr_ = dalloc<int>(gptr.size());
    d_idcg_ = dalloc<float>(n_groups_);
    d_group_hits_ = dalloc<int>(n_groups_);
    d_flags_ = dalloc<unsigned>(n_);
    d_hits_before_ = dalloc<unsigned>((size_t)n_ + 1);
    n_partial_ = grid_for(n_);
    d_partial_ = dalloc<double>(n_partial_);
    upload(d_gptr_, gptr.data(), sizeof(int) * gptr.size());
    sorter_.alloc(n_);
    longest_ = longest;
    RankPacks packs;  // (read by the copies until the set-up has waited)
    if (short_groups_) {
        packs = rank_packs(group);
        n_packs_ = (int)packs.packs.size();
        n_wide_ = (int)packs.wide.size();
        pack_rows_ = packs.most;
        shared_ = packs.shared;
        d_packs_ = dalloc<RankPack>(packs.packs.size());
        d_wide_ = dalloc<RankPack>(packs.wide.size());
        upload(d_packs_, packs.packs.data(), sizeof(RankPack) * packs.packs.size());
        upload(d_wide_, packs.wide.data(), sizeof(RankPack) * packs.wide.size());
        setup_short_groups(longest);
    }
    else setup_groups(y, gptr);
    TGBM_CHECK(!ndcg || idcg_valid_, "rank:ndcg needs labels in 0..30");  // (small non-negative integers: 1 << label)
}

void RankContext::upload(void *dst, const void *src, size_t bytes) {
    if (bytes) HIP_CHECK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream_));
}

void RankContext::setup_short_groups(int longest) {
    d_runs_ = dalloc<RankRun>(n_);
    run_bits_ = bits_for(n_);
    std::vector<float> log2_of((size_t)longest);
    for (int i = 0; i < longest; ++i) log2_of[i] = log2f((float)(i + 2));
    float *d_log2 = dalloc<float>((size_t)longest);
    upload(d_log2, log2_of.data(), sizeof(float) * (size_t)longest);
    int *d_counts = dalloc<int>(3);
    HIP_CHECK(hipMemsetAsync(d_counts, 0, sizeof(int) * 3, stream_));
    static_assert(kRankCountSortMax <= 1 << 15, "positions of a group in 15 bits");
    const size_t lds = (size_t)longest * (2 * sizeof(unsigned) + 2 * sizeof(unsigned short));
    static_assert(kRankCountSortMax * 12 <= 48 << 10, "no opt-in for the LDS");
    k_rank_setup<<<n_groups_, kSetupBlock, lds, stream_>>>(d_y_, d_gptr_, d_log2, longest, d_static_row_, d_run_of_, d_group_of_, d_runs_, d_idcg_, d_group_hits_, d_counts);
    HIP_CHECK(hipGetLastError());
    int counts[3];
    HIP_CHECK(hipMemcpyAsync(counts, d_counts, sizeof(counts), hipMemcpyDeviceToHost, stream_));
    HIP_CHECK(hipStreamSynchronize(stream_));  // (and the host's arrays have been read)
    idcg_valid_ = counts[0] == 0;
    ndcg_one_groups_ = idcg_valid_ ? counts[1] : n_groups_;
    zero_hit_groups_ = counts[2];
}

// Groups that the counting sort does not take are ordered on the host.
void RankContext::setup_groups(const LabelVector &y, const std::vector<int> &gptr) {
    bool labels_ok = true;
    for (float v : y) labels_ok = labels_ok && v >= 0.f && v < 31.f;
    // The groups are independent: the threads take contiguous ranges of about equally many rows (one thread: 6.8 ms for
    // 200 k rows in groups of 120). Runs are numbered inside a range first, then moved behind the earlier ranges' runs.
    std::vector<int> static_row(n_), run_of(n_), run_of_row(n_), group_of(n_), hits(n_groups_, 0);
    std::vector<float> idcg(n_groups_, 0.f);
    struct Range {
        int g0 = 0, g1 = 0;
        int ndcg_one = 0;  // groups whose NDCG is 1 by definition (IDCG == 0)
        int zero_hit = 0;
        std::vector<RankRun> runs;
    };
    const int n_ranges = n_ < kRankSetupRows ? 1 : (int)std::min(8u, std::max(1u, std::thread::hardware_concurrency()));
    std::vector<Range> ranges((size_t)n_ranges);
    for (int t = 0; t < n_ranges; ++t) {
        const long first_row = (long)n_ * (t + 1) / n_ranges;  // of the next range
        ranges[t].g0 = t == 0 ? 0 : ranges[t - 1].g1;
        ranges[t].g1 = t + 1 == n_ranges ? n_groups_
                                         : (int)(std::lower_bound(gptr.begin(), gptr.end() - 1, (int)first_row) - gptr.begin());
    }
    auto order_range = [&](Range &range) {
        for (int g = range.g0; g < range.g1; ++g) {
            const int b = gptr[g], e = gptr[g + 1];
            for (int i = b; i < e; ++i) {
                static_row[i] = i;
                group_of[i] = g;
                if (y[i] != 0.f) ++hits[g];
            }
            std::stable_sort(static_row.begin() + b, static_row.begin() + e, [&](int a, int c) { return y[a] > y[c]; });
            if (labels_ok) {  // NDCG::get_IDCG (rank_metric.cpp:106-123): float sum in descending label order
                float z = 0.f;
                for (int i = b; i < e; ++i) z += (float)((1 << (int)y[static_row[i]]) - 1) / log2f((float)(i - b + 2));
                idcg[g] = z;
            }
            if (idcg[g] == 0.f) ++range.ndcg_one;
            if (hits[g] == 0) ++range.zero_hit;
            bool skip_first = false;
            for (int i = b; i < e;) {
                int j = i + 1;
                while (j < e && y[static_row[j]] == y[static_row[i]]) ++j;
                RankRun r;
                r.group_begin = b;
                r.group_end = e;
                r.end = j;
                r.first_l = std::min(j, i + (skip_first ? 1 : 0));
                r.group = g;
                r.begin = i;
                skip_first = r.first_l < j;  // a processed run makes the loop step over the next run's first position
                for (int k = i; k < j; ++k) run_of[k] = (int)range.runs.size();
                range.runs.push_back(r);
                i = j;
            }
        }
    };
    auto number_range = [&](const Range &range, int before) {
        for (int i = gptr[range.g0]; i < gptr[range.g1]; ++i) run_of_row[static_row[i]] = run_of[i] += before;
    };
    std::vector<std::thread> pool;
    for (int t = 1; t < n_ranges; ++t) pool.emplace_back(order_range, std::ref(ranges[t]));
    order_range(ranges[0]);
    for (auto &th : pool) th.join();
    std::vector<RankRun> runs;
    for (const Range &range : ranges) {
        number_range(range, (int)runs.size());
        runs.insert(runs.end(), range.runs.begin(), range.runs.end());
        ndcg_one_groups_ += range.ndcg_one;
        zero_hit_groups_ += range.zero_hit;
    }
    idcg_valid_ = labels_ok;
    run_bits_ = bits_for((long)runs.size());
    d_runs_ = dalloc<RankRun>(runs.size());
    d_run_of_row_ = dalloc<int>(n_);
    d_acc_ = dalloc<long long>(2 * (size_t)n_);
    HIP_CHECK(hipMemsetAsync(d_acc_, 0, sizeof(long long) * 2 * (size_t)std::max(n_, 1), stream_));
    upload(d_static_row_, static_row.data(), sizeof(int) * (size_t)n_);
    upload(d_run_of_, run_of.data(), sizeof(int) * (size_t)n_);
    upload(d_run_of_row_, run_of_row.data(), sizeof(int) * (size_t)n_);
    upload(d_group_of_, group_of.data(), sizeof(int) * (size_t)n_);
    upload(d_runs_, runs.data(), sizeof(RankRun) * runs.size());
    upload(d_idcg_, idcg.data(), sizeof(float) * (size_t)n_groups_);
    upload(d_group_hits_, hits.data(), sizeof(int) * (size_t)n_groups_);
    HIP_CHECK(hipStreamSynchronize(stream_));  // the host vectors go out of scope
}

RankContext::~RankContext() {
    sorter_.release();
    for (void *p : allocs_) device_free(p);
}

void RankContext::gradient(const float *d_score, GHPair *d_gh, unsigned seed, bool order_is_fresh) {
    if (n_ == 0) return;
    const int grid = grid_for(n_);
    if (short_groups_) {
        last_cur_ = 0;
        have_metric_order_ = false;
        static LdsOptIn opt_in;
        const float *idcg = ndcg_ ? d_idcg_ : nullptr;
        if (longest_ * kRankGroupBytes > 48 * 1024) opt_in({reinterpret_cast<const void *>(&k_rank_gradient_group<kLongGroupBlock, false>)});
#define TGBM_RANK_GRADIENT(BLK, SHARED, GROUPS, WHICH, MOST)                                                                                \
    k_rank_gradient_group<BLK, SHARED><<<GROUPS, BLK, (MOST) * kRankGroupBytes, stream_>>>(WHICH, MOST, d_score, d_y_, d_static_row_, \
                                                                                  d_run_of_, d_runs_, idcg, seed, sorter_.vals[0], d_gh)
        if (n_packs_ > 0 && shared_) TGBM_RANK_GRADIENT(kPackBlock, true, n_packs_, d_packs_, pack_rows_);
        else if (n_packs_ > 0 && pack_rows_ <= 64) TGBM_RANK_GRADIENT(64, false, n_packs_, d_packs_, pack_rows_);
        else if (n_packs_ > 0) TGBM_RANK_GRADIENT(kPackBlock, false, n_packs_, d_packs_, pack_rows_);
        if (n_wide_ > 0) TGBM_RANK_GRADIENT(kLongGroupBlock, false, n_wide_, d_wide_, longest_);
#undef TGBM_RANK_GRADIENT
        return;
    }
    if (order_is_fresh && have_metric_order_) {
        // rows already ordered by (group, score descending, row): a stable sort by run id yields
        // (run, score descending, row), the same order as the full sort below
        k_rank_run_keys<<<grid, kBlock, 0, stream_>>>(n_, d_run_of_row_, sorter_.vals[last_cur_], sorter_.keys[0],
                                                     sorter_.vals[0]);
        last_cur_ = sort_pairs(stream_, sorter_, n_, run_bits_);
    } else {
        k_rank_train_keys<<<grid, kBlock, 0, stream_>>>(n_, d_static_row_, d_run_of_, d_score, sorter_.keys[0],
                                                       sorter_.vals[0]);
        last_cur_ = sort_pairs(stream_, sorter_, n_, 32 + run_bits_);
    }
    have_metric_order_ = false;
    k_rank_pairs<<<grid, kBlock, 0, stream_>>>(n_, d_runs_, d_run_of_, sorter_.vals[last_cur_], d_score, d_y_,
                                              ndcg_ ? d_idcg_ : nullptr, seed,
                                              reinterpret_cast<unsigned long long *>(d_acc_));
    k_rank_finish<<<grid, kBlock, 0, stream_>>>(n_, d_group_of_, d_gptr_, d_acc_, d_gh);
}

void RankContext::metric(int kind, const float *d_score, float *d_out) {
    TGBM_CHECK(kind == RANK_METRIC_MAP || kind == RANK_METRIC_NDCG, "unknown ranking metric %d", kind);
    const int grid = grid_for(n_);
    int cur = 0;
    if (short_groups_) {
#define TGBM_RANK_ORDER(BLK, SHARED, GROUPS, WHICH, LDS) \
    k_rank_order_group<BLK, SHARED><<<GROUPS, BLK, LDS, stream_>>>(WHICH, d_gptr_, d_group_of_, d_score, sorter_.vals[0])
        if (n_packs_ > 0 && shared_) TGBM_RANK_ORDER(kPackBlock, true, n_packs_, d_packs_, pack_rows_ * sizeof(unsigned));
        else if (n_packs_ > 0 && pack_rows_ <= 64) TGBM_RANK_ORDER(64, false, n_packs_, d_packs_, pack_rows_ * sizeof(unsigned));
        else if (n_packs_ > 0) TGBM_RANK_ORDER(kPackBlock, false, n_packs_, d_packs_, pack_rows_ * sizeof(unsigned));
        if (n_wide_ > 0) TGBM_RANK_ORDER(kLongGroupBlock, false, n_wide_, d_wide_, keys_to_sort(longest_) * sizeof(unsigned long long));
#undef TGBM_RANK_ORDER
    } else {
        k_rank_metric_keys<<<grid, kBlock, 0, stream_>>>(n_, d_group_of_, d_score, sorter_.keys[0], sorter_.vals[0]);
        cur = sort_pairs(stream_, sorter_, n_, 32 + group_bits_);
    }
    const int *sorted = sorter_.vals[cur];
    double constant;
    if (kind == RANK_METRIC_NDCG) {
        TGBM_CHECK(idcg_valid_, "NDCG needs labels in 0..30");
        k_rank_ndcg_partial<<<grid, kBlock, 0, stream_>>>(n_, sorted, d_group_of_, d_gptr_, d_y_, d_idcg_, d_partial_);
        constant = ndcg_one_groups_;
    } else {
        k_rank_hit_flags<<<grid, kBlock, 0, stream_>>>(n_, sorted, d_y_, d_flags_);
        device_exclusive_scan(stream_, d_flags_, d_hits_before_, n_, sorter_.d_total, sorter_.scan);
        k_rank_map_partial<<<grid, kBlock, 0, stream_>>>(n_, d_flags_, d_hits_before_, d_group_of_, d_gptr_,
                                                        d_group_hits_, d_partial_);
        constant = zero_hit_groups_;
    }
    k_rank_metric_final<<<1, kBlock, 0, stream_>>>(d_partial_, n_partial_, constant, n_groups_, d_out);
    last_cur_ = cur;
    have_metric_order_ = true;
}

}  // namespace tgbm
