// Ranking objectives and metrics on the device: LambdaRank gradients (rank:pairwise, rank:ndcg) and
// the list metrics MAP and NDCG over query groups of consecutive rows.
#pragma once
#include <hip/hip_runtime.h>

#include <vector>

#include "device_api.h"
#include "host.h"
#include "rank_packs.h"

namespace tgbm {

enum RankMetric { RANK_METRIC_MAP = 3, RANK_METRIC_NDCG = 4 };

// Data whose groups have at most kRankCountSortMax rows, and whose average row is in a group of at most kRankCountSortMean
// (sum(len^2) / rows), is ordered in the LDS of workgroups (k_rank_order_group, k_rank_gradient_group); other data takes the radix sort.
// The mean is from an order by counting throughout, quadratic in a group's rows. Groups of more than 256 rows are sorted by now, for
// which it is too low: 20 rounds of 200 k x 8, depth 4, in groups of 300, 500, 1000, 2000 rows take 3.1, 2.5, 2.7, 3.1 ms in LDS (set-up,
// which counts still, 1.1, 1.1, 1.3, 1.9) and 8.7, 8.9, 8.3, 8.4 by the radix sort (set-up 2.4); of 1 M rows in groups of 1000 3.9 (2.3)
// and 13.0 (8.1).
constexpr int kRankCountSortMax = 2048;
constexpr int kRankCountSortMean = 384;

constexpr int kRankSetupRows = 1 << 14;  // the groups of fewer rows are ordered by one thread (about 0.5 ms)

// One run of equal labels inside a query group, in the group's label-descending order. The run owns the
// positions [begin, end) of that order; [first_l, end) are the positions that draw a partner (the reference's
// loop over a group skips the first position of a run that follows a processed run,
// src/thundergbm/objective/ranking_obj.cpp:55-92), first_l == end for a run that draws nothing.
struct RankRun {
    int group_begin, group_end;  // positions of the whole group
    int first_l, end;
    int group;
    int begin;
};

class RankContext {
   public:
    // y: labels of all rows, d_y: the same on the device, where they outlive this object, or none; group: sizes of the query
    // groups (consecutive rows), their sum must be y.size()
    RankContext(hipStream_t s, const LabelVector &y, const float *d_y, const std::vector<int> &group, bool ndcg);
    ~RankContext();
    RankContext(const RankContext &) = delete;
    RankContext &operator=(const RankContext &) = delete;

    // LambdaRank::get_gradient (ranking_obj.cpp:20-96): gh[row] = sum of the lambdas of the sampled pairs the
    // row takes part in. `seed` selects the round's partner draws.
    // order_is_fresh: d_score has not changed since the last metric() call, whose (group, score) order then
    // only needs a stable re-sort by run id
    void gradient(const float *d_score, GHPair *d_gh, unsigned seed, bool order_is_fresh = false);
    // RankListMetric::get_score with MAP or NDCG (metric/rank_metric.cpp:9-104); writes one float to d_out
    void metric(int kind, const float *d_score, float *d_out);
    // the row order and partner draws of the last gradient() call (tests): sorted rows [n]
    const int *last_sorted_rows() const { return sorter_.vals[last_cur_]; }
    int n() const { return n_; }

   private:
    template <typename T>
    T *dalloc(size_t count);
    void upload(void *dst, const void *src, size_t bytes);
    void setup_short_groups(int longest);
    void setup_groups(const LabelVector &y, const std::vector<int> &gptr);
    hipStream_t stream_;
    int n_ = 0, n_groups_ = 0;
    bool ndcg_ = false;
    int run_bits_ = 0, group_bits_ = 0;
    int zero_hit_groups_ = 0;   // groups without a non-zero label: MAP = 1 by definition
    int ndcg_one_groups_ = 0;   // groups with IDCG == 0: NDCG = 1 by definition
    bool idcg_valid_ = false;   // all labels in 0..30
    std::vector<void *> allocs_;
    const float *d_y_ = nullptr;
    int *d_static_row_ = nullptr;  // rows of every group by label descending (ties: row ascending)
    int *d_run_of_ = nullptr;      // run of a position of that order
    int *d_run_of_row_ = nullptr;  // run of a row (long groups)
    RankRun *d_runs_ = nullptr;
    int *d_group_of_ = nullptr;    // group of a row
    int *d_gptr_ = nullptr;
    float *d_idcg_ = nullptr;
    int *d_group_hits_ = nullptr;  // rows with a non-zero label per group
    long long *d_acc_ = nullptr;   // [2n] fixed-point gradient / hessian sums (long groups)
    unsigned *d_flags_ = nullptr, *d_hits_before_ = nullptr;
    double *d_partial_ = nullptr;
    int n_partial_ = 0;
    PairSorter sorter_;
    int last_cur_ = 0;
    bool have_metric_order_ = false;  // sorter_.vals[last_cur_] is the (group, score) order of a metric() call
    int longest_ = 0;                 // group
    RankPack *d_packs_ = nullptr, *d_wide_ = nullptr;  // RankPacks
    int n_packs_ = 0, n_wide_ = 0, pack_rows_ = 0;
    bool shared_ = false;
    bool short_groups_ = false;       // groups short enough to be ordered in LDS (kRankCountSortMax / Mean)
};

}  // namespace tgbm
