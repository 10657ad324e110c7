// Host side of prediction: the reference's Predictor (src/thundergbm/predictor.cu:11-86).
#include <algorithm>
#include <chrono>
#include <cstring>

#include "device_api.h"
#include "host.h"
#include "model_handle.h"
#include "rank.h"
#include "score_slices.h"

namespace tgbm {

// See ScoreModel (device_api.h). One block: records, used features, slots of the features.
struct DeviceModel {
    int device = 0;
    void *block = nullptr;
    ScoreModel m;
    bool usable = false;  // false: the records do not describe this model
    ~DeviceModel() { device_free(block); }
};

namespace {

int transform_kind(const std::string &objective) {
    if (objective == "binary:logistic") return 1;
    if (objective == "multi:softmax") return 2;
    if (objective == "multi:softprob") return 3;
    if (objective == "reg:logistic") return 4;
    return 0;
}

bool children_ok(const TreeNode &nd, int n_nodes) {
    return nd.lch_index >= 0 && nd.lch_index < n_nodes && nd.rch_index >= 0 && nd.rch_index < n_nodes;
}

unsigned order_key(float v) {  // (k_score_rows' keys: predict_kernels.hip)
    if (v == 0.f) v = 0.f;
    unsigned b;
    std::memcpy(&b, &v, 4);
    return b ^ ((unsigned)((int)b >> 31) | 0x80000000u);
}

// Do the eight-byte records describe this model? Every split node keeps its children side by side (right = left + 1) and
// below itself - then a walk needs one child index and ends after at most `depth` steps, the number returned (0: they do
// not apply). Marks the features that splits reachable from a root use.
int records_apply(const Tree *trees, size_t n_trees, int n_nodes, std::vector<uint8_t> &feature_used) {
    if (n_nodes < 1 || n_nodes > 0x1fff) return 0;
    int deepest = 0;
    std::vector<int> level((size_t)n_nodes);
    for (size_t t = 0; t < n_trees; ++t) {
        const TreeNode *nodes = trees[t].nodes.data();
        std::fill(level.begin(), level.end(), -1);
        level[0] = 0;
        for (int self = 0; self < n_nodes; ++self) {
            const TreeNode &nd = nodes[self];
            if (nd.is_leaf || !children_ok(nd, n_nodes)) continue;  // (a walk ends here)
            if (nd.rch_index != nd.lch_index + 1 || nd.lch_index <= self) return 0;
            if (nd.split_value != nd.split_value) return 0;  // (a NaN threshold: the two comparisons would disagree)
            if (level[self] < 0) continue;  // (not reachable from the root)
            level[nd.lch_index] = level[nd.rch_index] = level[self] + 1;
            deepest = std::max(deepest, level[self] + 1);
            const int f = nd.split_feature_id;
            if (f < 0) continue;
            if (f >= (1 << 28)) return 0;
            if ((size_t)f >= feature_used.size()) feature_used.resize((size_t)f + 1, 0);
            feature_used[(size_t)f] = 1;
        }
    }
    return std::max(deepest, 1);
}

size_t align256(size_t b) { return (b + 255) / 256 * 256; }

std::shared_ptr<const DeviceModel> lay_out(hipStream_t s, const tgbm_model &model, int device, int n_iter, int n_class) {
    auto out = std::make_shared<DeviceModel>();
    out->device = device;
    ScoreModel &m = out->m;
    m.n_iter = n_iter;
    m.n_class = n_class;
    m.n_nodes = (int)model.trees[0].nodes.size();
    const size_t n_trees = (size_t)n_iter * n_class;
    std::vector<uint8_t> feature_used;
    m.depth = records_apply(model.trees.data(), n_trees, m.n_nodes, feature_used);
    if (m.depth == 0) return out;
    m.n_features = (int)feature_used.size();
    std::vector<int> used;
    for (int f = 0; f < m.n_features; ++f)
        if (feature_used[(size_t)f]) used.push_back(f);
    m.n_used = (int)used.size();
    m.leaf_slot = m.n_used;
    m.n_slots = m.n_used + 2;
    if (m.n_slots > 0x7fff) return out;
    const size_t rec_bytes = align256(n_trees * m.n_nodes * sizeof(uint2)), used_bytes = align256(used.size() * sizeof(int) + 4);
    std::vector<char> host(rec_bytes + used_bytes + sizeof(int) * ((size_t)m.n_features + 1));
    uint2 *rec = reinterpret_cast<uint2 *>(host.data());
    int *h_used = reinterpret_cast<int *>(host.data() + rec_bytes);
    int *slot_of = reinterpret_cast<int *>(host.data() + rec_bytes + used_bytes);
    std::copy(used.begin(), used.end(), h_used);
    std::fill(slot_of, slot_of + m.n_features + 1, -1);
    for (int k = 0; k < m.n_used; ++k) slot_of[used[(size_t)k]] = k;
    for (int it = 0; it < n_iter; ++it)
        for (int c = 0; c < n_class; ++c) {
            const TreeNode *nodes = model.trees[(size_t)it * n_class + c].nodes.data();
            uint2 *to = rec + ((size_t)c * n_iter + it) * m.n_nodes;
            for (int self = 0; self < m.n_nodes; ++self) {
                const TreeNode &nd = nodes[self];
                uint2 p;
                if (nd.is_leaf || !children_ok(nd, m.n_nodes)) {
                    std::memcpy(&p.x, &nd.base_weight, 4);
                    p.y = (unsigned)m.leaf_slot | (unsigned)self * 8u << 15;
                } else {
                    const int f = nd.split_feature_id;
                    const int slot = f >= 0 && f < m.n_features && slot_of[f] >= 0 ? slot_of[f] : m.n_used + 1;
                    const unsigned left = nd.default_right ? 0u : 1u;
                    p.x = order_key(nd.split_value) + left - 1u;
                    p.y = (unsigned)slot | (unsigned)nd.lch_index * 8u << 15 | left << 31;
                }
                to[self] = p;
            }
        }
    out->block = device_alloc(host.size());
    upload_large(s, out->block, host.data(), host.size());
    HIP_CHECK(hipStreamSynchronize(s));
    char *base = static_cast<char *>(out->block);
    m.records = reinterpret_cast<const uint2 *>(base);
    m.used = reinterpret_cast<const int *>(base + rec_bytes);
    m.slot_of = reinterpret_cast<const int *>(base + rec_bytes + used_bytes);
    out->usable = true;
    return out;
}

std::shared_ptr<const DeviceModel> device_model(hipStream_t s, tgbm_model &model, int n_iter, int n_class) {
    int device = 0;
    HIP_CHECK(hipGetDevice(&device));
    std::lock_guard<std::mutex> lock(model.mutex);
    const DeviceModel *have = model.on_device.get();
    if (have == nullptr || have->device != device || have->m.n_iter != n_iter || have->m.n_class != n_class)
        model.on_device = lay_out(s, model, device, n_iter, n_class);
    return model.on_device;
}

// Bytes of a slice of rows on their way to the device, see score(). Sparse rows: a walk of k_score_group takes about as long as
// the slice's values take over PCIe, so an eighth of a call's values is left to walk when the last ones are there (500 k rows
// of 35 values, 100 trees: 5.4 ms in slices of 64 MB, 4.7 of 32, 4.4 of 16 with every slice a send of its own, 4.3 in one
// send that has the columns in front). Where k_score_rows serves the call no slice has fewer rows than it is for, or the slice would
// go to k_score_group, which is slower there (500 k rows of 40 values, 90 columns, 100 trees of depth 8: 4.6 ms in eighths, 3.5
// with at least kScoreGroupRows rows each, and the same in slices of 24 or 64 MB). Dense rows: up to
// kDenseSlices slices that fill the chip once each (200 k x 28, 5 x 40
// trees of depth 8: 1.19 -> 1.08 ms; 600 k x 28, 100 trees of depth 6: 1.99 -> 1.95).
constexpr int kDenseSlices = 4;
constexpr size_t kLeastSlice = (size_t)8 << 20, kMostSlice = (size_t)64 << 20;

// The reference takes its shared-memory path - double sums, +inf is missing - when a row's dense vector of as many
// floats as the data has features fits 128 times into 48 KB (predictor.cu:85); the number of features is the largest
// column with a stored value + 1.
constexpr int kNarrowFeatures = 48 * 1024 / (128 * (int)sizeof(float));

template <typename Value>
bool stores_beyond(const Value *x, int n, int columns, int first) {  // a stored value in column `first` or later?
    for (int i = 0; i < n; ++i)
        for (int c = first; c < columns; ++c)
            if (x[(size_t)i * columns + c] != 0) return true;
    return false;
}

// What only a dataset with labels asks for: the training metric of the raw scores (class-major in d_out) in the log.
void log_the_metric(hipStream_t s, const GBMParam &param, const DataSet &ds, int n, int n_class, const float *d_out) {
    if (objective_needs_groups(param.objective)) {
        // MAP / NDCG need the query groups of the rows that are scored (Predictor::predict configures the
        // objective with the dataset's groups, predictor.cu:16-24); without them the metric line is left out
        long covered = 0;
        for (int g : ds.group) covered += g;
        if (!ds.group.empty() && covered == (long)n && (int)ds.y.size() == n) {
            const bool ndcg = param.objective == "rank:ndcg";
            RankContext rc(s, ds.y, nullptr, ds.group, ndcg);
            float *d_m = nullptr;
            device_alloc_to(d_m, sizeof(float));
            rc.metric(ndcg ? RANK_METRIC_NDCG : RANK_METRIC_MAP, d_out, d_m);
            float v = 0;
            HIP_CHECK(hipMemcpyAsync(&v, d_m, sizeof(float), hipMemcpyDeviceToHost, s));
            HIP_CHECK(hipStreamSynchronize(s));
            log_info("%s = %g", ndcg ? "NDCG" : "MAP", v);
            device_free(d_m);
        }
    } else if ((int)ds.y.size() == n && n > 0) {
        int kind = 0;
        if (param.objective == "binary:logistic") kind = 1;
        if (param.objective.find("multi:") == 0) kind = 2;
        static const char *names[] = {"RMSE", "test error", "multi-class accuracy"};
        float *d_y = nullptr, *d_m = nullptr;
        double *d_scratch = nullptr;
        device_alloc_to(d_y, sizeof(float) * (size_t)n);
        device_alloc_to(d_m, sizeof(float));
        device_alloc_to(d_scratch, sizeof(double) * (size_t)row_blocks(n));
        HIP_CHECK(hipMemcpyAsync(d_y, ds.y.data(), sizeof(float) * (size_t)n, hipMemcpyHostToDevice, s));
        launch_metric(s, kind, n, n_class, d_y, d_out, d_scratch);
        TreeLeftovers sum;
        sum.metric_out = d_m;
        sum.metric_partial = d_scratch;
        sum.metric_kind = kind;
        sum.metric_blocks = row_blocks(n);
        launch_metric_final(s, n, sum);
        float v = 0;
        HIP_CHECK(hipMemcpyAsync(&v, d_m, sizeof(float), hipMemcpyDeviceToHost, s));
        HIP_CHECK(hipStreamSynchronize(s));
        log_info("%s = %g", names[kind], v);
        device_free(d_y);
        device_free(d_m);
        device_free(d_scratch);
    }
}

// The objective's transform of the scores in `scores`; `labels` (device-readable) has room for the class labels.
// Returns how many floats of it are the predictions.
size_t transform_scores(hipStream_t s, const GBMParam &param, const DataSet &ds, int n, int n_class, float *scores,
                        const float *labels) {
    const int kind = transform_kind(param.objective);
    launch_predict_transform(s, kind, n, kind == 2 || kind == 3 ? n_class : param.num_class, labels, scores);
    return kind == 1 || kind == 2 ? (size_t)n : (size_t)n * n_class;
}

size_t labels_needed(const GBMParam &param, const DataSet &ds) {
    const int kind = transform_kind(param.objective);
    if (kind != 1 && kind != 2) return 0;
    const size_t need = kind == 1 ? 2 : (size_t)std::max(param.num_class, 1);
    TGBM_CHECK(ds.label.size() >= need, "predict: %zu class labels given, %zu needed", ds.label.size(), need);
    return ds.label.size();
}

// Small calls: the kernel reads rows and labels from a pinned block and writes the scores there, so the call is one or
// two launches and one wait. One row of 28 values, 100 trees: 25 us; through device memory, with the copies and waits of larger
// calls, 51 (1000 rows: 31 and 57).
bool score_small(hipStream_t s, const GBMParam &param, const ScoreModel &m, const DataSet &ds, bool transform, float *out) {
    const int n = (int)ds.n_instances();
    const size_t cells = ds.is_dense() ? (size_t)n * ds.dense_columns : (size_t)ds.nnz;
    const size_t in_bytes = ds.is_dense() ? cells * 4 : cells * 8 + ((size_t)n + 1) * 4;
    const size_t n_out = (size_t)n * m.n_class;
    constexpr size_t kMost = (size_t)128 << 10;
    if (in_bytes > kMost || n_out * 4 > kMost || ds.label.size() * 4 > kMost) return false;
    char *pin = static_cast<char *>(pinned_acquire());
    float *scores = reinterpret_cast<float *>(pin), *labels = reinterpret_cast<float *>(pin + kMost);
    char *at = pin + 2 * kMost;
    ScoreRows rows;
    rows.n = n;
    bool narrow = true;
    if (ds.is_dense()) {
        rows.x = reinterpret_cast<float *>(at);
        rows.columns = ds.dense_columns;
        rows.minus_zero_is_stored = ds.dense_f64 != nullptr;
        if (ds.dense_f64 != nullptr) {
            doubles_to_floats(reinterpret_cast<float *>(at), ds.dense_f64, cells);
            narrow = !stores_beyond(ds.dense_f64, n, ds.dense_columns, kNarrowFeatures);
        } else {
            std::memcpy(at, ds.dense_f32, cells * 4);
            narrow = !stores_beyond(ds.dense_f32, n, ds.dense_columns, kNarrowFeatures);
        }
    } else {
        int most = 0, least = 0;
        for (size_t e = 0; e < cells; ++e) {
            most = std::max(most, ds.col_idx[e]);
            least = std::min(least, ds.col_idx[e]);
        }
        TGBM_CHECK(least >= 0, "CSR input: negative column index %d", least);
        narrow = most < kNarrowFeatures;
        std::memcpy(at, ds.row_ptr, ((size_t)n + 1) * 4);
        rows.row_ptr = reinterpret_cast<int *>(at);
        at += ((size_t)n + 1) * 4;
        std::memcpy(at, ds.col_idx, cells * 4);
        rows.col = reinterpret_cast<int *>(at);
        at += cells * 4;
        std::memcpy(at, ds.val, cells * 4);
        rows.val = reinterpret_cast<float *>(at);
    }
    const bool launched = launch_score(s, rows, m, narrow, param.learning_rate, param.base_score, scores, (size_t)n);
    if (launched) {
        size_t n_ret = n_out;
        if (transform) {
            const size_t n_labels = labels_needed(param, ds);
            if (n_labels > 0) std::memcpy(labels, ds.label.data(), n_labels * 4);
            n_ret = transform_scores(s, param, ds, n, m.n_class, scores, labels);
        }
        HIP_CHECK_LAUNCHES("predict");
        HIP_CHECK(hipStreamSynchronize(s));
        std::memcpy(out, scores, n_ret * 4);
    }
    pinned_release(pin);
    return launched;
}

}  // namespace

void score(const GBMParam &param, tgbm_model &model, int n_iter, int n_class, const DataSet &ds, bool transform,
           bool log_metric, float *out) {
    int n_dev = 0;
    hipError_t e = hipGetDeviceCount(&n_dev);
    TGBM_CHECK(e == hipSuccess && n_dev >= 1, "no HIP device available: this library has no CPU path");
    const int n = (int)ds.n_instances();
    const long nnz = ds.nnz;
    TGBM_CHECK(n_iter >= 1 && n_class >= 1, "empty model");
    const size_t n_trees = (size_t)n_iter * n_class;
    TGBM_CHECK(n_trees <= model.trees.size(), "model holds %zu trees, %d x %d requested", model.trees.size(), n_iter, n_class);
    const int n_nodes = (int)model.trees[0].nodes.size();
    for (size_t t = 0; t < n_trees; ++t)
        TGBM_CHECK((int)model.trees[t].nodes.size() == n_nodes, "trees of different size in one model");
    auto t_begin = std::chrono::steady_clock::now();
    auto lap = [&](const char *what) {
        auto now = std::chrono::steady_clock::now();
        log_debug("predict: %s %.3f s", what, std::chrono::duration<double>(now - t_begin).count());
        t_begin = now;
    };
    // (TGBM_PREDICT_COMPACT=0: the 16-byte records also where the 8-byte ones apply; TGBM_PREDICT_TPS=0: the 48-byte nodes)
    const char *ce = std::getenv("TGBM_PREDICT_COMPACT"), *te = std::getenv("TGBM_PREDICT_TPS");
    const bool want_records = !(ce != nullptr && atoi(ce) == 0) && !(te != nullptr && atoi(te) == 0);
    hipStream_t s = stream_acquire();
    std::shared_ptr<const DeviceModel> dm;
    if (want_records) dm = device_model(s, model, n_iter, n_class);
    const bool usable = dm != nullptr && dm->usable;
    if (usable && n > 0 && !log_metric && score_small(s, param, dm->m, ds, transform, out)) {
        lap("rows in pinned memory");
        stream_release(s);
        return;
    }
    float *d_val = nullptr, *d_out = nullptr, *d_label = nullptr, *d_x = nullptr;
    int *d_col = nullptr, *d_row_ptr = nullptr;
    const size_t n_out = (size_t)n * n_class;
    device_alloc_to(d_out, sizeof(float) * std::max(n_out, (size_t)1));
    hipStream_t s_up = stream_acquire();
    bool done = n == 0;
    ScoreRows rows;
    bool narrow = true;
    int F = 0;
    // Slices of whole rows go up on a second stream: the traversal of a slice runs while the next ones cross PCIe.
    hipEvent_t up;
    HIP_CHECK(hipEventCreateWithFlags(&up, hipEventDisableTiming));
    UploadSet slices;
    std::vector<ScoreRows> rows_of;
    std::vector<int> first_of;
    auto score_slice = [&](size_t k) {
        HIP_CHECK(hipEventRecord(up, s_up));
        HIP_CHECK(hipStreamWaitEvent(s, up, 0));
        if (done)
            done = launch_score(s, rows_of[k], dm->m, narrow, param.learning_rate, param.base_score, d_out + first_of[k], (size_t)n);
        HIP_CHECK_LAUNCHES("predict (rows)");  // (a launch's error is its thread's)
    };
    if (!done && ds.is_dense()) {
        rows.columns = ds.dense_columns;
        rows.minus_zero_is_stored = ds.dense_f64 != nullptr;
        narrow = ds.dense_f64 != nullptr ? !stores_beyond(ds.dense_f64, n, ds.dense_columns, kNarrowFeatures)
                                         : !stores_beyond(ds.dense_f32, n, ds.dense_columns, kNarrowFeatures);
        device_alloc_to(d_x, sizeof(float) * (size_t)n * ds.dense_columns);
        const size_t row_bytes = 4 * (size_t)ds.dense_columns;
        int step = n;
        if (usable) {
            if (score_rows_fit(dm->m)) step = (n - 1) / std::max(1, std::min(kDenseSlices, n / score_slice_rows(dm->m))) + 1;
            step = (int)std::max<size_t>(1, std::min((size_t)step, kMostSlice / row_bytes));
        }
        done = usable;
        for (int r0 = 0; r0 < n; r0 += std::min(step, n - r0)) {
            const size_t off = (size_t)r0 * ds.dense_columns;
            rows.n = std::min(step, n - r0);
            rows.x = d_x + off;
            if (ds.dense_f64 != nullptr) slices.add_doubles(d_x + off, ds.dense_f64 + off, (size_t)rows.n * ds.dense_columns);
            else slices.add(d_x + off, ds.dense_f32 + off, (size_t)rows.n * row_bytes);
            rows_of.push_back(rows);
            first_of.push_back(r0);
        }
        slices.send_in_order(s_up, score_slice);
    } else if (!done) {
        // The column indices go up before the values: the feature count, which selects the traversal, may have to be taken from them.
        F = (int)ds.n_features();
        device_alloc_to(d_val, sizeof(float) * (size_t)std::max(nnz, 1l));
        device_alloc_to(d_col, sizeof(int) * (size_t)std::max(nnz, 1l));
        device_alloc_to(d_row_ptr, sizeof(int) * ((size_t)n + 1));
        slices.add(d_row_ptr, ds.row_ptr, sizeof(int) * ((size_t)n + 1));
        slices.add_columns(d_col, ds.col_idx, (size_t)nnz);
        constexpr size_t kBefore = 2;  // the values' slices come behind them
        done = usable;
        const size_t eighth = sizeof(float) * (size_t)nnz / 8 / kPinnedBytes * kPinnedBytes;  // (whole pieces)
        const long slice_entries = usable ? (long)(std::min(std::max(eighth, kLeastSlice), kMostSlice) / sizeof(float)) : nnz;
        rows.col = d_col;
        rows.val = d_val;
        const bool by_rows = usable && n >= score_least_rows(dm->m) && score_rows_fit(dm->m);
        const std::vector<int> first = score_slices(ds.row_ptr, n, slice_entries, by_rows ? kScoreGroupRows : 1);
        for (size_t k = 0; k + 1 < first.size(); ++k) {
            const int r0 = first[k], r1 = first[k + 1];
            const long e0 = ds.row_ptr[r0];
            rows.n = r1 - r0;
            rows.row_ptr = d_row_ptr + r0;
            slices.add(d_val + e0, ds.val + e0, sizeof(float) * (size_t)(ds.row_ptr[r1] - e0));
            rows_of.push_back(rows);
            first_of.push_back(r0);
        }
        slices.send_in_order(s_up, [&](size_t j) {
            if (j >= kBefore) return score_slice(j - kBefore);
            if (j + 1 < kBefore) return;  // (the columns are on their way as well, the values behind them)
            if (!ds.features_counted) F = device_max_int(s_up, d_col, nnz) + 1;
            narrow = F <= kNarrowFeatures;
        });
    }
    lap("rows");
    TreeNode *d_model = nullptr;
    PackedNode *d_packed = nullptr;
    if (!done) {
        // models that the records do not describe, rows over more used features than the LDS holds
        if (ds.is_dense()) {
            const DeviceCsr csr = dense_to_csr(s, n, ds.dense_columns, d_x, ds.dense_f64 != nullptr);
            d_x = nullptr;
            d_val = csr.val;
            d_col = csr.col;
            d_row_ptr = csr.row_ptr;
            F = csr.n_features;
        }
        std::vector<TreeNode> flat(n_trees * n_nodes);
        for (size_t t = 0; t < n_trees; ++t)
            std::memcpy(flat.data() + t * n_nodes, model.trees[t].nodes.data(), sizeof(TreeNode) * (size_t)n_nodes);
        device_alloc_to(d_model, sizeof(TreeNode) * flat.size());
        device_alloc_to(d_packed, sizeof(PackedNode) * flat.size());
        HIP_CHECK(hipMemcpyAsync(d_model, flat.data(), sizeof(TreeNode) * flat.size(), hipMemcpyHostToDevice, s));
        HIP_CHECK(hipStreamSynchronize(s));
        launch_pack_model(s, d_model, (long)flat.size(), n_nodes, d_packed);
        launch_fill_f32(s, d_out, 0.f, n_out);
        launch_predict(s, n, F, d_row_ptr, d_col, d_val, d_model, n_iter, n_class, n_nodes, param.learning_rate,
                       param.base_score, d_out, (size_t)n, d_packed);
    }
    HIP_CHECK_LAUNCHES("predict");
    if (log_metric) log_the_metric(s, param, ds, n, n_class, d_out);
    size_t n_ret = n_out;
    if (transform) {
        const size_t n_labels = labels_needed(param, ds);
        if (n_labels > 0) {
            device_alloc_to(d_label, sizeof(float) * n_labels);
            HIP_CHECK(hipMemcpyAsync(d_label, ds.label.data(), sizeof(float) * n_labels, hipMemcpyHostToDevice, s));
        }
        n_ret = transform_scores(s, param, ds, n, n_class, d_out, d_label);
    }
    HIP_CHECK_LAUNCHES("predict (metric, transform)");
    download_large(s, s_up, out, d_out, sizeof(float) * n_ret);
    HIP_CHECK(hipStreamSynchronize(s_up));
    HIP_CHECK(hipEventDestroy(up));
    lap("traversal, transform and download");
    for (void *p : {(void *)d_val, (void *)d_col, (void *)d_row_ptr, (void *)d_x, (void *)d_model, (void *)d_packed,
                    (void *)d_out, (void *)d_label})
        device_free(p);
    stream_release(s_up);
    stream_release(s);
    lap("release");
}

// (callers that hold the trees as the parser returns them: the CLI and the R interface)
std::vector<float> predict(const GBMParam &param, const std::vector<std::vector<Tree>> &model, const DataSet &dataset,
                           bool log_metric) {
    TGBM_CHECK(!model.empty() && !model.front().empty(), "empty model");
    tgbm_model flat;
    for (const auto &iter : model) {
        TGBM_CHECK(iter.size() == model.front().size(), "ragged model");
        for (const Tree &t : iter) flat.trees.push_back(t);
    }
    const int kind = transform_kind(param.objective);
    const size_t n = dataset.n_instances();
    std::vector<float> out(kind == 1 || kind == 2 ? n : n * model.front().size());
    score(param, flat, (int)model.size(), (int)model.front().size(), dataset, true, log_metric, out.data());
    return out;
}

}  // namespace tgbm
