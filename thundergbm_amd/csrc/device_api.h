// Host-callable launchers of the HIP kernels (gfx950). All launches are stream-ordered and never
// synchronise; sizes are validated by the callers in trainer.hip / predictor.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <atomic>
#include <functional>
#include <initializer_list>
#include <memory>
#include <mutex>
#include <vector>

#include "common.h"
#include "bin_groups.h"
#include "table_places.h"

#define HIP_CHECK(expr)                                                                              \
    do {                                                                                             \
        hipError_t e_ = (expr);                                                                      \
        if (e_ != hipSuccess) ::tgbm::fatal("%s:%d HIP error %s: %s", __FILE__, __LINE__, #expr,     \
                                            hipGetErrorString(e_));                                  \
    } while (0)

// A kernel launch reports a bad configuration (too much LDS, an empty or oversized grid) only through
// hipGetLastError; the host stages call this after their launches so that such a failure aborts with the
// stage's name instead of leaving stale results behind.
#define HIP_CHECK_LAUNCHES(stage)                                                                    \
    do {                                                                                             \
        hipError_t e_ = hipGetLastError();                                                           \
        if (e_ != hipSuccess) ::tgbm::fatal("kernel launch failed in %s: %s", stage, hipGetErrorString(e_)); \
    } while (0)

namespace tgbm {

// Device blocks and streams that are kept for the next call (device_memory.hip). Whoever frees a block or gives a
// stream back has synchronised the work on it; device_mem_info counts the kept blocks as free memory.
void *device_alloc(size_t bytes);
void device_free(void *p);
template <typename T>
void device_alloc_to(T *&p, size_t bytes) {
    p = static_cast<T *>(device_alloc(bytes));
}
void device_mem_info(size_t *free_b, size_t *total_b);

// More dynamic LDS than the default window, for kernels of one launcher: a static object of the launcher, called before
// each launch. The limit belongs to the kernel, not to a launch, so it is set once per device and to the most that the
// kernel can take: set to a launch's own size, it could fall below that of another thread between its call and its launch.
constexpr int kLdsBytes = 160 * 1024;
class LdsOptIn {
  public:
    void operator()(std::initializer_list<const void *> kernels) {
        int dev = 0;
        HIP_CHECK(hipGetDevice(&dev));
        TGBM_CHECK(dev < kDevices, "device %d: more than %d devices", dev, kDevices);
        std::call_once(once_[dev], [&] {
            for (const void *k : kernels) {
                hipFuncAttributes a;
                HIP_CHECK(hipFuncGetAttributes(&a, k));
                HIP_CHECK(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, kLdsBytes - (int)a.sharedSizeBytes));
            }
        });
    }

  private:
    static constexpr int kDevices = 64;
    std::once_flag once_[kDevices];
};
hipStream_t stream_acquire();
void stream_release(hipStream_t s);

constexpr int kMissingBin = 255;   // dense matrix sentinel: the feature has no stored value in this row
constexpr int kMissingBin16 = 65535;  // the same for 16-bit bins
// 16-bit bins: bins of a feature block that leave the LDS room for two histogram workgroups per CU, and the most a
// block may hold at all (160 KB of 8-byte bins)
constexpr int kDense16BlockBins = 8192;
constexpr int kDense16MaxBlockBins = 20480;
constexpr int kPartChunk = 2048;   // rows per partition work item (256 threads x 8 rounds)
// From so many rows on the partition's launches are shared out as far as they go: what every work item would do for itself
// grows with the rows a second time. Items whose counts then also come as one sum:
constexpr int kPartGroupRows = 1 << 24;
constexpr int kPartGroup = 64;
// Dense layout, below so many rows (from there on the rows are re-ordered by leaves: those of a child follow each other, and
// one workgroup has them all): a level's row lists and the next level's histograms in one launch (launch_partition_hist), by
// workgroups of 1, 2 or 4 partition items. As long as a block's columns can be shared out instead (kSplitHistGroups) fewer items
// give as many workgroups and less to store and read back, so it is 2 items; 1 on few rows that store little, where a part of
// fewer columns would be laid out again by too many workgroups of the deep levels; 4 where 2 store more than kSplitHistBytes. Where
// 4 do, the launches for many rows are as fast. ms a tree (depth 8, 6 of the wide ones) with launch_hist_dense, 1, 2, 4 items:
// 20 k x 28 (MB that 1 stores: 0.6) 0.201, 0.154, 0.157; 20 k x 136 (2.8) 0.254, 0.214, 0.234, 0.248; 50 k x 12, 8 classes (4.9) 0.263, 0.234, 0.248;
// 20 k x 300 (6.1) 0.201, 0.168, 0.167; 60 k x 136 (8.3) 0.281, 0.242, 0.229, 0.253; 34 k x 300 (10.4) 0.209, 0.180, 0.173;
// 100 k x 28 (2.8) 0.237, 0.198, 0.197, 0.202; 900 k x 4 (3.6) 0.268, 0.262, 0.233, 0.238; 150 k x 28 (4.2) 0.241, 0.205, 0.197, 0.208;
// 900 k x 10 (9.0) 0.275, 0.291, 0.251, 0.257; 78 k x 37 of 1024 bins (11.5) 0.231, 0.224, 0.203, 0.212; 500 k x 28 (14) 0.274, 0.267, 0.243, 0.253;
// 200 k x 136 (27) 0.330, 0.310, 0.309, 0.315; 1 M x 28 (28) 0.327, 0.347, 0.304, 0.308; 100 k x 300 (30) 0.245, 0.242, 0.228, 0.218;
// 300 k x 28 of 1024 bins (34) 0.320, 0.366, 0.332, 0.286; 50 k x 700 (36) 0.276, 0.281, 0.274, 0.256; 400 k x 30, 6 classes (72) 0.520, 0.600, 0.528, 0.538.
constexpr int kSplitHistRows = 1 << 20;
constexpr int kSplitHistMost = 4;
constexpr size_t kSplitHistBytes = 13 << 20;
constexpr int kSplitHistOneRows = 1 << 16;
constexpr size_t kSplitHistOneBytes = 6 << 20;
// A workgroup's LDS adds about 8 pairs a nanosecond, so up to a workgroup per CU a block's columns are shared out as well
// (each part lays the lists out again): 20 k x 28 0.128 -> 0.111 ms a tree, 100 k x 28 0.198 -> 0.187, 500 k x 28 0.251 -> 0.246; with two per
// CU 0.111, 0.200 and 0.279.
constexpr int kSplitHistGroups = 256;
// Dense layout: up to so many pairs (nodes, where single nodes are built) in a level every workgroup plans for itself.
constexpr int kUnplannedPairs = 256;
constexpr int kMergeWideBins = 1024; // bins of a feature that k_merge_eval_wide holds at most
constexpr int kEvalPackBins = 256; // bins scanned by one wavefront in split finding (4 per lane)
constexpr int kCsrHeadBins = 4864;  // head slots of the sparse histogram: 2 x 8 bytes each, two workgroups per CU
constexpr int kRootParts = 512;     // parts of the rows whose sums add up to the root's (the root's work items at most)
// Rows a packed LDS bin may absorb before it is drained (QuantCtl::flush_rows). With float hessians (32 + 32-bit
// fields) 8192: a row of a large node is then counted at 2^-17 of the tree's largest |g|, and even rows that all
// round the same way (the first logistic tree has two gradient values) stay within 4e-6 of the sum of |g|; 32768
// measured 1.2 % faster on 10 M rows (root items never drained) and put the root sum of that tree beyond the 1e-5
// bound. With integer hessians the gradient field has 47 bits and 32768 rows cost no precision that matters: the
// 500 k x 2000 regression builds a tree in 1.90 instead of 2.00 ms.
constexpr int kHistFlushRows = 8192;
constexpr int kHistFlushRowsInt = 32768;
// Data of so few rows is trained on by the launches of launch_small_level, trees of so many levels at most. ms a tree with
// them and with launch_partition_hist, 28 columns and depth 8: 4000 rows 0.120 and 0.147, 8000 0.131 and 0.150, 12 000 0.143 and 0.154;
// depth 6: 0.090 and 0.105, 0.099 and 0.107, 0.109 and 0.109 (14 000 with the code of sixteen steps 0.116 and 0.108). Features of more
// than 255 bins have their split search in a launch of its own, and the line where it was without it: 28 columns, depth 8, 8000
// rows 0.156 and 0.155, 16 000 0.183 and 0.158.
// Data too wide or of too many classes for launch_partition_hist goes to launch_hist_dense there, which is faster as well (with
// launch_small_level and with it): 14 000 x 3400, depth 6 0.657 and 0.555, 16 000 x 3400, depth 8 1.94 and 1.32, 13 000 x 500 of 8 classes
// 0.749 and 0.615, 10 000 x 1000 of 1024 bins 0.690 and 0.526.
constexpr int kSmallRows = 12288;
constexpr int kSmallRowsWide = 8192;
constexpr int kSmallBlock = 1024;
constexpr int kSmallDepth = 10;
constexpr int kRowBlock = 4096;    // rows owned by one workgroup of the row-ordered passes and reductions
inline int row_blocks(int n) { return n <= 0 ? 1 : (n + kRowBlock - 1) / kRowBlock; }

// Per-level control block written by the planning kernels and read by the worker kernels.
struct LevelCtl {
    int hchunk;      // rows per histogram work item
    int n_hitems;    // histogram work items of the level
    int n_pitems;    // partition work items of the level
    int rows_built;  // rows visited by the histogram build of the level
};

// Fixed-point plan of one tree. Histograms are exact 64-bit integer sums of round(g * scale_g), round(h * scale_h);
// the scales are the largest powers of two that keep the sum over all n rows below 2^62, so the quantum is about
// max|g| * n / 2^62 (2^-38 of the largest gradient at 10 M rows).
//   Dense layout: a work item (a run of rows of one node) accumulates in LDS with one 64-bit integer atomic per
// (row, feature) - gfx950 executes those about 15x faster than float LDS atomics - into a packed bin: gradient in
// the high 64 - h_bits bits (signed), hessian in the low h_bits bits. The fields must hold the sum of the
// rows added between two drains of the LDS bins into 64-bit registers, at most min(rows of the node,
// flush_rows), so the items of a node coarsen the tree's scales by a power of two (shift) that depends on the
// node's row count only: the fewer rows a node has, the finer it counts, and what a row adds to a node does not
// depend on the order of the rows;
// k_hist_merge shifts every item's sums back to the tree's scale. h_bits: 32 in general; when every hessian of the
// tree is a small non-negative integer (squared loss: 1, or the draw count under bagging) the hessian field gets
// exactly the bits that flush_rows * max h needs and the gradient field the rest (47 bits for h = 1), which
// is what keeps heavy-tailed regression residuals at float-like resolution (2^-32 of the largest |g| per row).
// All sums after the LDS stage are 64-bit integers: exact, order-independent, bit-reproducible.
struct QuantCtl {
    float scale_g, scale_h;  // value -> integer of the tree's histograms (powers of two)
    float inv_g, inv_h;      // integer -> value
    float gq_max, hq_max;    // max|g| * scale_g, max h * scale_h: the most one row can add
    int h_bits;              // width of the hessian field of a packed LDS bin
    int h_integer;           // 1: every hessian is an integer, scale_h = 1 and no item shifts it
    int flush_rows;          // rows a packed LDS bin absorbs between two drains (kHistFlushRows / kHistFlushRowsInt)
};

// Block result of the per-tree gradient reduction.
struct GradStats {
    float g, h;        // sums
    float gmax, hmax;  // max |g|, max h
    float hfrac;       // max |h - round(h)|: 0 when every hessian is an integer
};

// Candidate produced by one wavefront of the split finder.
struct SplitCand {
    float score;  // signed gain: > 0 missing goes left, <= 0 missing goes right
    int index;    // global bin index
    GHPair miss;
    GHPair left;  // sum of the bins strictly below the candidate, within its feature
    int feature, bin;  // dense layout: its feature, its bin within the feature
};

// Dense column-blocked bin matrix: block b holds features [b*W, (b+1)*W) as n rows of W bytes.
struct DenseBins {
    const uint8_t *data = nullptr;
    int W = 0;          // features per row of a block (a row of a block is W * bin_bytes bytes, a multiple of 4)
    int n_blocks = 0;
    size_t block_stride = 0;  // bytes between blocks = n * W * bin_bytes
    // Column-major copy (feature f = n consecutive bins at col + f * col_stride * bin_bytes): the partition reads
    // one feature of many rows, which costs one bin per row here instead of one sector per row.
    const uint8_t *col = nullptr;
    size_t col_stride = 0;  // in bins
    // 1: byte bins (at most 255 bins per feature, 255 = no stored value); 2: 16-bit bins for max_num_bin above 255
    // (65535 = no stored value)
    int bin_bytes = 1;
    // Bundles (byte bins only; nullptr: every feature has a column of its own). Consecutive features of which no row
    // stores more than one (one-hot groups) share one column of the matrix: feature f sits in column feat_col[f] and
    // its local bin b is stored as feat_lo[f] + b, where feat_lo[f] counts the bins of the bundle's features before
    // f - the byte is the bin's distance from the bundle's first global bin, which is all the histogram kernel needs.
    // A byte outside [feat_lo[f], feat_lo[f] + bins of f) means that f has no stored value in the row.
    const int *feat_col = nullptr;
    const uint8_t *feat_lo = nullptr;
    int n_cols = 0;  // columns of the matrix (= features when nothing is bundled)
    // Lane (dword) of a row's record that is kept free of bins for the row's gradient word (the last lane of the
    // row), -1: none. gh_fresh: gh_words[row] (launch_gh_words) matches the gradient array of this launch; the root
    // level's histogram launch then decodes the words (gh_objective says how) instead of reading the pairs and copies
    // them into the records, and the launches below the root take them from the records instead of gathering the
    // pairs. That lane never adds bins either way.
    int gh_lane = -1;
    int gh_fresh = 0;
    int gh_objective = 0;
    const unsigned *gh_words = nullptr;  // [n]
};

// Sparse layout for wide, mostly-missing data: the reference's own representation, CSR rows of global
// bin ids (hist_tree_builder_single.cu:49-130).
struct CsrBins {
    const int *row_ptr = nullptr;  // [n + 1]
    const int *bin = nullptr;      // [nnz] global bin id, ascending within a row
    // Histogram addressing of the same stored values: the bins of the most frequent features (the
    // "head", at most kCsrHeadBins of them) are accumulated in LDS. word >= 0: global bin id,
    // word < 0: ~word is the head slot. nullptr: no head (every value goes to HBM).
    const int *hist_word = nullptr;  // [nnz]
    const int *head_bin = nullptr;   // [head_bins] global bin id of every head slot
    int head_bins = 0;
    // The same stored values sorted by global bin id (rows ascending inside a bin): the root histogram, where
    // every row takes part, is a segmented sum over this copy instead of atomics to random bins. nullptr: none.
    const int *csc_bin = nullptr;  // [nnz] (with the level pass until its values have places of their own)
    const int *csc_row = nullptr;  // [nnz]
    long nnz = 0;
    // Sparse level pass: byte columns of the frequent features (local bin id of the row, kMissingBin = no stored
    // value), column col_of_feature[f] at colbin + col * col_stride; col_of_feature[f] < 0: the feature has none
    const uint8_t *colbin = nullptr;
    const int *col_of_feature = nullptr;  // [F]
    size_t col_stride = 0;
};

// Sparse layout, level pass: one pass per level over the bin-major copy of the stored values (sorted by global bin,
// rows ascending inside a bin). A task is a run of whole features, or a chunk of one feature that has too many
// values for one workgroup ("big" feature); a task accumulates (node, bin) tables of its features in LDS and
// searches them for every node's best candidate right there, so no per-node histogram exists in HBM.
constexpr int kSparseCells = 8192;      // (node, bin) cells of 16 bytes an LDS table holds
constexpr int kSparseMaxLevelNodes = 1024;  // deepest level the pass serves (depth <= 11)
constexpr int kSparseBatchFeatures = 2047;  // features whose tables share one LDS batch at most
constexpr int kSparseTasks = 1024;          // smaller tasks where there would be fewer than that
struct SparseTask {
    int f_begin, f_end;  // features [f_begin, f_end) (a chunk task: one feature)
    int g_begin, g_end;  // groups of kSpreadGroup places of its values (SparsePass::table_bin)
    int cand_slot;       // candidate slot the task fills, -1: a chunk (its feature's slot is filled by k_sparse_big)
    int partial_slot;    // chunk: where its table goes in SparsePass::partial, else -1
};
// Features with few stored values (Trainer::sparse_feature_in_tables) are not searched through tables: k_sparse_rare_filter looks for the (feature, node)
// runs of their values that could win at all and searches only those. A task is a run of whole features whose values
// fit one tile; a workgroup of the search takes every n_rare_groups-th task.
constexpr int kRareBlock = 512;
constexpr int kRareTile = 4096;       // values per task at most
constexpr int kRareTileLeast = 512;   // a value per thread: smaller tasks leave threads without one
constexpr int kRareFeatures = 2047;   // features per task at most (one more would meet the mark of an empty place)
// Features with more than kRareLeast values (at most this many, the most frequent ones) are served through tables too.
constexpr int kRareExempt = 128;
constexpr int kRareLeast = 256;
constexpr int kRareGroupTiles = 16;   // tasks of a search workgroup at most
constexpr int kRareGroups = 512;      // search workgroups that are resident together (two per CU)
struct RareTask {
    int v_begin;     // first place of the task's values in SparsePass::rare_row / rare_key
    int count;       // stored values of its features (SparsePass::rare_places: places that they take)
    int meta_begin;  // first entry of its features in SparsePass::rare_meta / rare_fid
    int n_feat;      // features of the task
};
// key of a stored value: feature (index inside its task) << 20 | sixty-fourth of the feature's values << 8 | local bin
constexpr int kRareFeatShift = 20;
// Spread values: the rows are cut into blocks whose nodes fit the LDS beside other workgroups, and the values of a rare task and of
// a table feature lie in the order of their rows' blocks, four places of one block at a time (kRareEmpty in rare_key, kTableEmpty
// in table_bin: nobody's).
constexpr int kSpreadLogRows = 15;
constexpr int kSpreadRows = 1 << kSpreadLogRows;
constexpr int kSpreadLevel = 7;       // deepest level with its nodes in a byte (all ones: the row has come to rest above)
constexpr int kSpreadBlocks = 341;    // (more leave less than three quarters of a tile to values)
// Stored values from which on they are spread: a launch more a level, and less time per value. ms a tree of depth 8, looked up / spread:
// 0.7 M values 0.395 / 0.440, 2.2 M 0.647 / 0.648, 3.6 M 0.630 / 0.616, 7.2 M 0.769 / 0.649, 18 M 1.31 / 1.02, 36 M 2.50 / 1.76.
constexpr long kSpreadValues = 3000000;
constexpr unsigned kRareEmpty = ~0u;
constexpr unsigned kTableEmpty = 0xffffu;
inline int spread_blocks(int n) { return (int)(((long)n + kSpreadRows - 1) >> kSpreadLogRows); }
struct SparseBig {
    int feature;
    int slot_begin, slot_end;  // partial slots of its chunks
    int cand_slot;
};
struct SparsePass {
    const SparseTask *tasks = nullptr;
    int n_tasks = 0;
    const SparseBig *big = nullptr;
    int n_big = 0;
    int max_table_bins = 0;  // most bins of a feature of theirs
    // rare features
    const RareTask *rare_tasks = nullptr;
    int n_rare_tasks = 0, n_rare_groups = 0;
    int rare_slot = 0;                  // candidate slot of the first group
    const int2 *rare_meta = nullptr;    // per feature of a task: (first global bin, number of bins)
    const int *rare_fid = nullptr;      // its feature id
    const int *rare_row = nullptr;      // [n_rare_places] rows and keys of their values
    const unsigned *rare_key = nullptr;
    const int *rare_places = nullptr;   // per task
    long n_rare = 0;                    // stored values
    size_t n_rare_places = 0;           // (a multiple of 16)
    unsigned long long *rare_item = nullptr;  // [n_sets][n_rare_places] values of a level that may matter, tile by tile
    // Spread values (n_spread > 0: row blocks; else nullptr): a value's group as in its key; groups of places by row block - the
    // groups of block b in list l (the rare tasks, then the table features) from spread_begin[b * n_lists + l] on -, their rows inside
    // the block and where they lie, the table values' places after the rare ones'.
    // Of the current tree and level: a rare value's row word with its feature in the node's place, a value's row's node.
    int n_spread = 0, n_lists = 0;
    const uint8_t *rare_group = nullptr;           // [n_rare_places]
    const unsigned *spread_begin = nullptr;        // [n_spread * n_lists + 1]
    const unsigned short *spread_row = nullptr;    // [groups][kSpreadGroup]
    const unsigned *spread_place = nullptr;        // [groups] first place / kSpreadGroup
    unsigned *rare_code = nullptr;                 // [n_sets][n_rare_places]
    uint8_t *value_node = nullptr;                 // [n_sets][n_rare_places + n_table_places]
    int *rare_passed = nullptr;               // [n_sets][n_rare_tasks] how many of a tile
    const int *feat_val_begin = nullptr;  // [F + 1] first position of every feature in the bin-major copy
    // Values of the table features, a feature's in row order
    const int *table_features = nullptr;  // [n_table_features]
    int n_table_features = 0;
    size_t n_table_places = 0;            // (a multiple of 16)
    const int *table_first = nullptr;     // [F + 1] first group of places of every feature's values (other features: none)
    const unsigned short *table_bin = nullptr;  // [n_table_places] bin, counted from the first one of the feature's task
    const int *table_row = nullptr;             // [n_table_places]
    // [n_sets][n_table_places] the gradient pair of every value's row, left there by the pass of level 0: those below then stream it
    // instead of fetching a cache line per value (nullptr: no room, gather). With gh_words (below) the words instead.
    GHPair *table_gh = nullptr;
    // the rows' pairs as words (launch_gh_words) and what they are made of, where they match the gradients of the level 0
    const unsigned *gh_words = nullptr;
    int gh_objective = 0;
    longlong2 *partial = nullptr;         // [n_sets][n_partial_slots][partial_stride] chunk tables, (bin, node) cells
    size_t partial_stride = 0;            // cells per slot: most bins of a big feature x kSparseMaxLevelNodes at most
    int n_partial_slots = 0;
    int n_cand_slots = 0;
};

struct TreeBuffers {
    int n = 0, n_bins = 0, F = 0, depth = 0, n_nodes = 0;
    int sparse = 0;                // 1: CSR layout, histograms accumulated directly in hist_q
    TreeNode *nodes = nullptr;     // [n_nodes]
    int2 *seg = nullptr;           // [n_nodes] row-list segment [x, y) of every node
    int *nid = nullptr;            // [n]
    int *ridx[2] = {nullptr, nullptr};  // [n] row lists, ping-pong by level parity
    uint8_t *goes_right = nullptr; // [max_pitems * 256] per partition item and thread: bit k = its k-th row goes right
    longlong2 *hist_q[2] = {nullptr, nullptr};  // [max_level_nodes * n_bins] exact fixed-point histograms (g, h)
                                                // of the nodes of a level, ping-pong by level parity
    longlong2 *partial = nullptr;  // [max_hitems * n_bins] per-item fixed-point sums (g, h)
    QuantCtl *quant = nullptr;     // scales of the current tree
    int2 *hitem_shift = nullptr;   // [max_hitems] powers of two by which a dense work item (its node) coarsened (g, h)
    // sparse level pass only (else nullptr): node every row has reached (heap id) and rows per node
    unsigned short *nid16 = nullptr;  // [n + 2]
    int *node_rows = nullptr;         // [n_nodes]
    // sparse level pass: the row's node of the level and what bounds its part in a candidate, see k_sparse_rare_filter
    // (nullptr: no rare features)
    unsigned *row_word = nullptr;     // [n]
    // sparse level pass: best candidate key of every node of the level over all tasks, and the candidate slot of
    // the task that searches a feature (k_best_update reads the winner's record from that slot)
    unsigned long long *best_key = nullptr;  // [max_level_nodes]
    const int *feat_slot = nullptr;          // [F]
    // Root sums as exact integers at the tree's scales (what a row order cannot change), from the gradients when no
    // feature is stored in every row: [2 i], [2 i + 1] the sums of part i of the rows (kRootParts at most)
    long long *root_total = nullptr;
    int complete_feature = -1;     // dense layout: a feature stored in every row (its bins add up to the root), or -1
    int max_hitems = 0, target_hitems = 0, max_pitems = 0;
    float *leaf_value = nullptr;   // [n_nodes] prediction increment of a row that ended in the node (after pruning)
    int *end_bound = nullptr;      // [(row_blocks(n) + 1) x (2^depth - 1)] list positions of the row block boundaries
    int *hpair_begin = nullptr;    // [max_level_nodes + 1] first histogram item of every sibling pair
    int4 *hpair_plan = nullptr;    // [max_pairs] dense layout: (hpair_built, its row-list segment), see plan_hist_item
    int *hpair_built = nullptr;    // [max_pairs] heap id of the node built from rows, -1 = inactive pair
    int *pitem_begin = nullptr;    // [2][max_level_nodes + 1] first partition item of every node of a level, by level parity
    int *pitem_nleft = nullptr;    // [max_pitems]
    // [max_pitems] per-node path of the sparse layout: pitem_nleft added up; dense layout of many rows: its sums over
    // kPartGroup items each (not a pointer of its own: every launch takes these as arguments)
    int *pitem_loff = nullptr;
    int *node_nleft = nullptr;     // [max_level_nodes]
    LevelCtl *ctl = nullptr;       // [depth + 1]
    SplitPoint *sp = nullptr;      // [max_level_nodes]
    SplitCand *cand = nullptr;     // [max_level_nodes * n_packs]
    GradStats *root_partial = nullptr;  // [n_grad_blocks] block results of the per-tree gradient reduction
    int n_grad_blocks = 0;
    // split finder packing: wavefront w scans global bins [pack_begin[w], pack_begin[w+1]) (whole features)
    const int *pack_begin = nullptr;
    // per bin: distance to the last bin of its feature (low byte), distance from the first one (next byte), and in the
    // dense layout, whose feature ids fit 16 bits, the feature (high half)
    const unsigned *bin_meta = nullptr;  // [n_bins]
    int n_packs = 0;
    const uint8_t *ignored = nullptr;  // [F] columns whose candidates score 0 this round (nullptr: none)
    // Features with more than 255 cut points (max_num_bin up to 65 535; CSR layout, per-node path): the node's split
    // bin does not fit TreeNode::split_bid, a byte as in the reference's model format, so the row -> node update
    // reads it from here. nullptr: every feature has at most 255 bins.
    int *split_bin = nullptr;          // [n_nodes] local bin id of the node's split
    const int *cut_row_ptr = nullptr;
    const int *cut_fid = nullptr;
    const float *cut_val = nullptr;
    // dense block tables
    const int *blk_bin_begin = nullptr;  // [n_blocks + 1] first global bin of every block
    const int *feat_lds_off = nullptr;   // [n_blocks * W] bin offset of a feature inside its block
    int max_block_bins = 0;
    // Every per-tree array above is allocated n_sets times back to back (one set per class tree of a
    // boosting round, so that the trees of a round can be built by the same launches, class = blockIdx.z).
    int n_sets = 1;
    int max_level_nodes = 0;
    // Histogram arena smaller than the deepest level (it is sized against the free memory; the reference does the
    // same with its last_hist buffer and builds both siblings from rows beyond the depth that fits,
    // hist_tree_builder_single.cu:811-832, :544-570): hist_nodes node histograms per buffer. A level with more nodes
    // is served in batches of nodes [lvl_x0, lvl_x1) (the buffer pointer is shifted so that node x still sits at
    // x * n_bins); from level singles_from on no parent histogram exists any more, so every child of a split node
    // is built from its own rows and the "pairs" of the work-item plan are single nodes.
    int hist_nodes = 0;
    int lvl_x0 = 0, lvl_x1 = 1 << 30;
    int singles_from = 1 << 30;
    __host__ __device__ bool singles(int level) const { return level >= singles_from; }
    __host__ __device__ int n_hpairs(int level) const {
        return level == 0 ? 1 : (singles(level) ? (1 << level) : (1 << (level - 1)));
    }
    __host__ __device__ bool planned(int level) const { return n_hpairs(level) > kUnplannedPairs; }
    __host__ __device__ int hpair_lo(int level) const { return singles(level) ? lvl_x0 : (lvl_x0 >> 1); }
    __host__ __device__ int hpair_hi(int level) const {  // end of the pairs of the served nodes
        const int n = n_hpairs(level);
        const long hi = singles(level) ? (long)lvl_x1 : (((long)lvl_x1 + 1) >> 1);
        return hi < n ? (int)hi : n;
    }
    __host__ __device__ int nodes_served(int level) const {
        const int nl = 1 << level;
        return (lvl_x1 < nl ? lvl_x1 : nl) - lvl_x0;
    }
    size_t n_end_bound = 0, n_partial = 0;

    // Row list / histogram buffer of a level (selected without indexing an array member dynamically: a
    // kernel's local copy of this struct would otherwise be placed in scratch memory).
    __host__ __device__ int *list(int level) const { return (level & 1) ? ridx[1] : ridx[0]; }
    __host__ __device__ longlong2 *hist(int level) const { return (level & 1) ? hist_q[1] : hist_q[0]; }
    __host__ __device__ int *pbegin(int level) const { return pitem_begin + (level & 1) * (max_level_nodes + 1); }

    // The buffers of set k (k = 0: this object itself).
    __host__ __device__ TreeBuffers for_class(int k) const {
        TreeBuffers t = *this;
        if (k == 0) return t;
        const size_t K = (size_t)k;
        t.nodes += K * n_nodes;
        t.seg += K * n_nodes;
        t.nid += K * n;
        t.ridx[0] += K * n;
        t.ridx[1] += K * n;
        t.goes_right += K * (size_t)max_pitems * 256;
        t.hist_q[0] += K * hist_nodes * n_bins;
        t.hist_q[1] += K * hist_nodes * n_bins;
        t.partial += K * n_partial;
        t.quant += K;
        t.hitem_shift += K * max_hitems;
        t.root_total += K * 2 * kRootParts;
        if (nid16 != nullptr) {
            t.nid16 += K * (((size_t)n + 2) / 2 * 2);
            t.node_rows += K * n_nodes;
            if (row_word != nullptr) t.row_word += K * n;
            t.best_key += K * max_level_nodes;
        }
        t.leaf_value += K * n_nodes;
        t.end_bound += K * n_end_bound;
        t.hpair_begin += K * (max_level_nodes + 1);
        t.hpair_plan += K * max_level_nodes;
        t.hpair_built += K * max_level_nodes;
        t.pitem_begin += K * 2 * (max_level_nodes + 1);
        t.pitem_nleft += K * ((size_t)max_pitems + 1);
        t.pitem_loff += K * ((size_t)max_pitems + 1);
        t.node_nleft += K * max_level_nodes;
        t.ctl += K * (depth + 2);
        t.sp += K * max_level_nodes;
        t.cand += K * max_level_nodes * n_packs;
        t.root_partial += K * n_grad_blocks;
        if (split_bin != nullptr) t.split_bin += K * n_nodes;
        return t;
    }
};

// objective codes
enum Objective { OBJ_SQUARE = 0, OBJ_LOGISTIC = 1, OBJ_SOFTMAX = 2, OBJ_RANK = 3 };

void launch_gradient(hipStream_t s, int objective, int n, int num_class, const float *y, const float *yp, GHPair *gh,
                     GHPair *block_sums, int n_blocks);
// flags[f] = the f-th bit of the caller's, which travel with the launches' arguments: nothing is copied and nobody waits.
constexpr int kColumnFlagWords = 64;  // of a launch
struct ColumnFlags {
    unsigned long long bits[kColumnFlagWords];
};
void launch_column_flags(hipStream_t s, const std::vector<unsigned long long> &bits, int F, uint8_t *flags);
// RowSampler::do_bagging over the N gradient pairs; `count` holds N zeroed ints and is left zeroed. perm (may
// be null): original row of each of the n_rows physical positions; the N entries are planes of n_rows rows
void launch_bagging(hipStream_t s, int N, unsigned seed, int *count, GHPair *gh, const int *perm = nullptr,
                    int n_rows = 0);
// Tree-building launchers: `tb` is the first buffer set, `n_class` consecutive sets (the class trees of one
// round) are served by one launch; gradient / prediction pointers address the first of those classes.
// stats_ready: tb.root_partial already holds the block statistics of gh_class (fused round end)
struct TreeLeftovers {  // of the tree before: see k_tree_init
    TreeNode *model = nullptr;  // where its nodes go (nullptr: they are there)
    float *metric_out = nullptr;  // where its round's metric goes (nullptr: it is there), and what to add up
    const double *metric_partial = nullptr;
    int metric_kind = 0, metric_blocks = 0;
    bool small = false;  // (of the tree that begins) the rows' nodes are kept in tb.nid
    int run = 0;         // (of the tree that begins) the levels' histograms are launch_partition_hist's, see there
};
void launch_tree_init(hipStream_t s, const TreeBuffers &tb, const GHPair *gh_class, float lambda,
                      bool stats_ready = false, int n_class = 1, const TreeLeftovers &left = TreeLeftovers());
void launch_root_stats(hipStream_t s, const TreeBuffers &tb, const GHPair *gh_class, int n_class);
void launch_metric_final(hipStream_t s, int n, const TreeLeftovers &left);
// sum_rows (level 0): also the sums of the items' rows into tb.root_total, for a split search with root_of_rows. init (level 0):
// also what launch_tree_init does; tb.root_partial is ready (launch_root_stats).
void launch_hist_dense(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level,
                       int n_class = 1, bool sum_rows = false, const TreeLeftovers *init = nullptr, float lambda = 0);
void launch_hist_merge(hipStream_t s, const TreeBuffers &tb, int level, int n_class = 1);
// After the root histogram exists: replaces the root's float sums (whose last bits depend on the order of the rows)
// by the exact fixed-point totals, from the bins of tb.complete_feature or, without one, from the gradients.
void launch_root_sum(hipStream_t s, const TreeBuffers &tb, const GHPair *gh_class, float lambda, int n_class = 1);
// Number of bytes equal to `value` among n bytes in device memory (synchronises).
long device_count_bytes(hipStream_t s, const uint8_t *d_v, size_t n, uint8_t value);
long device_count_u16(hipStream_t s, const uint16_t *d_v, size_t n, uint16_t value);
void launch_hist_csr(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const GHPair *gh, int level,
                     int n_class = 1);
void launch_partition_csr(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, int level, int n_class = 1);
// store_sibling (sparse layout only): keep the derived sibling histograms; nobody reads those of a tree's
// last level. derive: the nodes that were not built are parent - built (always so in the sparse layout).
void launch_eval_split(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class = 1,
                       bool store_sibling = true, bool derive = false);
// Dense layout, all nodes of the level at once: launch_hist_merge and launch_eval_split in one launch (level 0: and
// launch_root_sum, from the bins of a complete feature or from what launch_hist_dense has summed up of the rows). store: the
// histograms are kept (nobody reads those of a tree's last level).
// run: the histograms' work items are launch_partition_hist's, of so many rows of the parents (0: launch_hist_dense's).
void launch_merge_eval(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class, bool store, int run = 0);
// Split search with one workgroup per (feature, node): any number of bins per feature (n_packs = F candidates per node)
void launch_eval_split_wide(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class = 1,
                            bool store_sibling = true, bool derive = false, bool root_of_rows = false);
// launch_hist_merge and launch_eval_split_wide below the root: one launch where the features' bins and the pairs' items allow it.
void launch_merge_eval_wide(hipStream_t s, const TreeBuffers &tb, int level, float mcw, float lambda, int n_class, bool store, int run,
                            int max_feature_bins);
void launch_best_update(hipStream_t s, const TreeBuffers &tb, int level, float rt_eps, float lambda, int n_class = 1);
// Dense layout: the rows of a level's split nodes move into the children's lists. update: the nodes' best candidates have
// not been applied to the tree yet (launch_best_update); it happens here.
void launch_partition_dense(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, int level, bool update,
                            float rt_eps, float lambda, int n_class = 1);
// Dense layout, moderately many rows: launch_partition_dense and the histograms of the next level's built nodes in two
// launches instead of three (k_split_hist). split_hist_plan: rows of a level's node that a workgroup of the second one serves,
// run 0: such data goes through launch_partition_dense and launch_hist_dense. Inside boost() only: the level's candidates are fresh,
// and every row leaves the node where it ends in tb.nid (launch_map_end), at level tb.depth - 1 the last of them.
// Feature blocks are shared out over 1 << log_split workgroups where there would be few. part_bins[k]: most bins of a part of
// a block in 1 << k parts.
struct SplitHistPlan {
    int run = 0, log_split = 0;
    int lds_bins = 0;  // part_bins[log_split]
    // Class trees whose rows have all of their bins, of a byte each, in one record: launch_map_end walks the trees with them, and
    // tb.nid is left alone until then. From so many rows of all trees on: calls of 10 rounds, depth 8, without and with, ms: 8 x 60 k one-hot rows
    // 3.53, 3.52; 3 x 250 k 4.28, 4.16; 4 x 200 k x 28 4.51, 4.39; 4 x 500 k 6.69, 6.62; 20 rounds of 8 x 500 k 12.9, 12.55.
    bool walk = false;
};
constexpr int kWalkRows = 5 << 17;
// (split_hist_run: the rows as far as what is stored decides them; the plan's are as many or more)
int split_hist_run(const TreeBuffers &tb, int n_class);
SplitHistPlan split_hist_plan(const TreeBuffers &tb, const DenseBins &bins, const int *part_bins, int n_class);
void launch_partition_hist(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level, const SplitHistPlan &plan,
                           float rt_eps, float lambda, int n_class = 1);
// Dense layout, few rows: the level's splits, the children's lists and the histograms of the next level's built nodes in one
// launch. The split search of the next level then derives the siblings (launch_eval_split with derive).
bool small_levels_fit(const TreeBuffers &tb);
// next_cand (nullptr: never): room for the next level's candidates, a slot per column of every node. True: they are there, that
// split search is done.
bool launch_small_level(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, const GHPair *gh, int level, float rt_eps,
                        float lambda, const int *part_bins, int n_class, SplitCand *next_cand, float mcw);
// The end of a tree whose rows' nodes are in tb.nid (lookup_level >= 0: split nodes of that level still hold the rows of their
// children): prunes the tree into `model` (n_class trees back to back; tb.nodes
// stays as it is) and updates the predictions; y: also the metric partials, the next gradients and their statistics. walk (not with y):
// SplitHistPlan::walk.
void launch_map_end(hipStream_t s, const TreeBuffers &tb, const DenseBins &bins, int lookup_level, TreeNode *model, float gamma, float *yp,
                      float lr, int n_class = 1, const float *y = nullptr, int objective = 0, int metric_kind = 0,
                      GHPair *gh = nullptr, double *metric_scratch = nullptr, unsigned *gh_words = nullptr, bool walk = false);
// Sparse level pass (tb.nid16 set): split search of a level (candidates into tb.cand, one slot per task / big
// feature; launch_best_update follows) and the row -> node update. dump_hist: also store the (node, bin) tables
// into tb.hist(level) (stage-wise driving and tests; needs tb.hist_q).
void launch_sparse_level(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const SparsePass &sp,
                         const GHPair *gh, int level, float mcw, float lambda, bool dump_hist, int n_class = 1);
void launch_sparse_partition(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const SparsePass &sp, int level, int n_class = 1);
// Byte columns of the frequent features (CsrBins::colbin, pre-filled with kMissingBin) from the bin-major copy.
void launch_sparse_cols(hipStream_t s, long nnz, const int *csc_bin, const int *csc_row, const int *cut_fid,
                        const int *cut_row_ptr, const int *col_of_feature, uint8_t *colbin, size_t col_stride);
// Fills what SparsePass points to under the same names from the bin-major copy; the spread_* arrays where sp.n_spread > 0:
// launch_spread_count leaves the groups of every (block, list) in `count` (their exclusive sums are spread_begin). task_bin0: [n_table_features] first
// bin of the task that a table feature belongs to; parts: of their values (add_table_parts).
void launch_spread_count(hipStream_t s, const CsrBins &bins, const SparsePass &sp, unsigned *count);
void launch_rare_setup(hipStream_t s, const TreeBuffers &tb, const CsrBins &bins, const SparsePass &sp, int *row, unsigned *key,
                       int *places, uint8_t *group, unsigned short *spread_row, unsigned *spread_place);
void launch_table_first(hipStream_t s, int n_table, const int *table_features, const int *first /* [n_table + 1] */, int *table_first);
void launch_table_setup(hipStream_t s, const CsrBins &bins, const SparsePass &sp, int n_parts, const TablePart *parts, const int *task_bin0,
                        int *row, unsigned short *table_bin, unsigned short *spread_row, unsigned *spread_place);
// The rows' words of a tree (TreeBuffers::row_word).
void launch_sparse_row_words(hipStream_t s, const TreeBuffers &tb, const GHPair *gh, int n_class);
// Row-ordered passes over the row lists (one of dbins / cbins by tb.sparse). lookup_level: the level
// whose split nodes still hold their children's rows (-1: none).
void launch_nid_rebuild(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins,
                        int lookup_level);
// (prune_gamma, here and below: prune the tree with this gamma first - launch_prune's work inside the same launches)
void launch_predict_in_training(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins,
                                int lookup_level, float *yp_class, float lr, int n_class = 1,
                                const float *prune_gamma = nullptr);
// prediction update + metric partials + next gradients + their block statistics (tb.root_partial); metric_scratch
// holds row_blocks(n) doubles
void launch_round_end(hipStream_t s, const TreeBuffers &tb, const DenseBins *dbins, const CsrBins *cbins,
                      int lookup_level, int objective, int metric_kind, const float *y, float *yp, float lr,
                      GHPair *gh, double *metric_scratch, const float *prune_gamma = nullptr, unsigned *gh_words = nullptr);
// words[i] = the gradient word of row i (the pair of a squared or 0/1-label logistic loss in 32 bits, which the
// histogram kernels decode to the very pair launch_gradient computes; see DenseBins::gh_lane)
void launch_gh_words(hipStream_t s, int objective, int n, const float *y, const float *yp, unsigned *words);
// scratch: row_blocks(n) doubles, which launch_metric_final adds up
void launch_metric(hipStream_t s, int objective_metric, int n, int num_class, const float *y, const float *yp,
                   double *scratch);
void launch_fill_f32(hipStream_t s, float *p, float v, size_t n);
void launch_fill_u8(hipStream_t s, uint8_t *p, uint8_t v, size_t n);

// data preparation
// F: columns of the matrix; feat_col / feat_lo: DenseBins' bundle tables or nullptr; group_first: bin_groups on the device, n_groups runs
void launch_bin_dense(hipStream_t s, int n, const int *row_ptr, const int *col, const float *val, const float *cut_val,
                      const int *cut_row_ptr, uint8_t *binmat, int W, size_t block_stride, uint8_t *colmat,
                      size_t col_stride, int bin_bytes, int F, const int *feat_col,
                      const uint8_t *feat_lo, bool rows_ascend, int n_features, int n_bins, const int *group_first = nullptr,
                      int n_groups = 0);
// false when some row holds a column index below its predecessor's
bool device_rows_ascend(hipStream_t s, int n, const int *row_ptr, const int *col);
// min_next[c] (pre-filled with INT_MAX) = smallest column index that follows column c in a row (equal neighbours, a
// column stored twice, do not count); *descending is set when a row's columns do not ascend
void launch_min_next_col(hipStream_t s, int n, int F, const int *row_ptr, const int *col, int *min_next, int *descending);
// feat_slot (may be nullptr): first head slot of a feature or -1; then hist_word is written as well
void launch_bin_csr(hipStream_t s, long nnz, const int *col, const float *val, const float *cut_val,
                    const int *cut_row_ptr, int *bin_id, const int *feat_slot = nullptr, int *hist_word = nullptr);
// cut points on device: returns the device arrays through out parameters allocated by the callee
struct DeviceCuts {
    float *cut_val = nullptr;
    int *cut_row_ptr = nullptr;
    int *cut_fid = nullptr;
    int n_bins = 0;
    std::vector<long> feature_nnz;  // host: stored values per feature
};
// full_rows: every row stores every column, in order (d_val is a row-major matrix). cells: the matrix that the values come from, where
// its cells are sorted along
struct DenseCells {
    const float *x;
    int n, columns;
    bool minus_zero_is_stored;
};
// Does a cell hold a value? A zero does not; -0 does in double-precision matrices (minus_zero_is_stored, upload_doubles_as_floats).
__host__ __device__ inline bool is_stored(float v, bool minus_zero_is_stored) {
    return v != 0.f || (minus_zero_is_stored && __builtin_signbit(v) != 0);
}
// Are the cells that hold no value sorted along with the others (build_cut_points)? That costs less than grouping the values: on wide
// data, where they would be sorted as 64-bit pairs, up to a quarter of the cells, else up to a 32nd (all passes: 35 M cells of 700
// features 1.9 -> 0.95 ms).
inline bool sorts_cells_along(int n, int F, long nnz) {
    const long all = (long)n * F;
    return nnz > 0 && n >= 1024 && all - nnz <= all / (F > 256 ? 4 : 32);
}
DeviceCuts build_cut_points(hipStream_t s, int F, long nnz, const float *d_val, const int *d_col, int max_num_bin,
                            bool full_rows = false, const DenseCells *cells = nullptr);
// (at most 256 features, full rows, or the cells)
DeviceCuts build_cut_points_by_feature(hipStream_t s, int F, long nnz, const float *d_val, const int *d_col, bool full_rows,
                                       int max_num_bin, const DenseCells *cells = nullptr);

// Tile sums of the device-wide exclusive scan, one pair of arrays per recursion level (grown on demand).
struct ScanScratch {
    struct Level {
        unsigned *sums = nullptr, *scanned = nullptr;
        size_t cap = 0;
    };
    std::vector<Level> levels;
    void release();
};

// out[i] = in[0] + ... + in[i-1] over n 32-bit counters, *d_total (device) = the sum of all of them.
void device_exclusive_scan(hipStream_t s, const unsigned *in, unsigned *out, long n, unsigned *d_total,
                           ScanScratch &sc);

// Buffers of sort_pairs for up to `cap` (64-bit key, 32-bit payload) pairs; allocated once, reused per call.
struct PairSorter {
    long cap = 0, n_tiles = 0;
    unsigned long long *keys[2] = {nullptr, nullptr};
    int *vals[2] = {nullptr, nullptr};
    unsigned *counts = nullptr, *offsets = nullptr, *d_total = nullptr;
    ScanScratch scan;
    void alloc(long n);
    void release();
};
// Stable LSD radix sort (8 bits per pass) of the n pairs in keys[0] / vals[0] by the key bits [0, key_bits),
// ascending. Returns which of the two buffer pairs (0 or 1) holds the result. Stream-ordered; allocates only
// when the scan scratch has to grow (first call).
int sort_pairs(hipStream_t s, PairSorter &ps, long n, int key_bits);

// Bin-major copy of CSR bin ids: sort keys (global bin, payload = row) of every stored value, and the sorted
// pairs split into the two int arrays the root histogram reads. sort_key (may be null): the key a bin sorts by
// (the bin itself stays in the key's high half and is what csc_bin receives).
void launch_csc_keys(hipStream_t s, int n_rows, const int *row_ptr, const int *bin, const int *sort_key,
                     unsigned long long *keys, int *vals);
void launch_bin_sort_keys(hipStream_t s, int n_bins, const int *cut_fid, const int *cut_row_ptr, const uint8_t *in_tables,
                          int *sort_key);
void launch_bin_meta(hipStream_t s, int n_bins, const int *cut_fid, const int *cut_row_ptr, unsigned *meta);
void launch_csc_unpack(hipStream_t s, long nnz, const unsigned long long *keys, const int *vals, int *csc_bin,
                       int *csc_row);

// Pieces of the physical re-ordering of the rows: sort keys (node of a row, payload = its position), gathers
// dst[p] = src[from[p]] of whole rows, the row permutation, and the column-major copy rebuilt from the
// row-major blocks.
void launch_reorder_keys(hipStream_t s, int n, int depth, const int *nid, unsigned long long *keys, int *vals);
void launch_gather_rows(hipStream_t s, int n, int bytes_per_row, const int *from, const void *src, void *dst);
void launch_gather_perm(hipStream_t s, int n, const int *from, const int *perm_old, int *perm_new);
void launch_cols_from_rows(hipStream_t s, int n, int W, int F, int n_blocks, const uint8_t *binmat, size_t block_stride,
                           uint8_t *colmat, size_t col_stride, int bin_bytes);

// Largest of n ints in device memory (synchronises; 0 for n == 0); aborts when one of them is negative.
int device_max_int(hipStream_t s, const int *d_v, long n);

// Host -> device copy of a pageable array, stream-ordered on s; large ones go through pinned staging pieces. The source
// has been read when the call returns.
void upload_large(hipStream_t s, void *dst, const void *src, size_t bytes);
// The same for doubles that the device takes as floats. Zeros of either sign arrive as +0, other values that are too
// small for a float as -0.
void upload_doubles_as_floats(hipStream_t s, float *dst, const double *src, size_t count);
// Several arrays at once: the threads convert and copy one while another crosses PCIe.
class UploadSet {
   public:
    void add(void *dst, const void *src, size_t bytes);
    void add_doubles(float *dst, const double *src, size_t count);
    // Column indices, which cross PCIe as bytes or 16-bit words where they all fit; anything else (negative ones too)
    // arrives as it is.
    void add_columns(int *dst, const int *src, size_t count);
    // an array that another thread is still making: source() waits for it; it is sent last
    void add_late(void *dst, size_t bytes, std::function<const void *()> source);
    void send(hipStream_t s);  // once
    // The arrays one after the other instead. arrived(j) is called for the j-th one in their order, by one thread at a time, as
    // soon as what s gets next runs after its copy.
    void send_in_order(hipStream_t s, const std::function<void(size_t)> &arrived);

   private:
    struct Job {
        void *dst;
        size_t bytes;
        std::function<const void *()> source;                              // the bytes as they are, or:
        std::function<void(char *to, size_t offset, size_t length)> fill;  // writes bytes [offset, offset + length) of them
        bool late;
    };
    friend void send_jobs(hipStream_t s, const std::vector<Job> &jobs, int threads, const std::function<void(size_t)> *arrived);
    struct Columns {
        int *dst;
        const int *src;
        size_t count;
        int width;  // bytes of the narrow form
        void *narrow;
        std::shared_ptr<std::atomic<bool>> fits;
        size_t job;
    };
    static void widen(hipStream_t s, const Columns &c);
    void release_narrow(hipStream_t s);
    template <typename Narrow>
    bool add_narrow(int *dst, const int *src, size_t count);
    std::vector<Job> jobs_;
    std::vector<Columns> columns_;
};
// Device -> pageable host memory after what is queued on s; the bytes are there when the call returns. other: a second stream of
// the caller's.
void download_large(hipStream_t s, hipStream_t other, void *dst, const void *src, size_t bytes);
// The conversion alone, for arrays that the device reads from host memory.
void doubles_to_floats(float *to, const double *from, size_t count);
// A pinned block of kPinnedBytes that the device can read and write directly; kept for later calls.
constexpr size_t kPinnedBytes = (size_t)4 << 20;
void *pinned_acquire();
void pinned_release(void *p);  // the work that uses it is done
void release_transfer_memory();  // the pinned pieces that are kept for later copies

// CSR form of a dense row-major matrix [n][columns] on the device: the stored values are those that are not zero
// (NaN is stored); with minus_zero_is_stored -0 is a stored zero (upload_doubles_as_floats).
struct DeviceCsr {
    float *val = nullptr;
    int *col = nullptr;
    int *row_ptr = nullptr;
    long nnz = 0;
    int n_features = 1;  // largest column with a stored value + 1, at least 1
    float *cells = nullptr;  // see dense_to_csr
};
// Takes `x` over: it becomes the value array when every cell is stored, is handed back as `cells` where cut points are made of them
// (for_cuts, sorts_cells_along), else it is freed. Synchronises.
DeviceCsr dense_to_csr(hipStream_t s, int n, int columns, float *x, bool minus_zero_is_stored, bool for_cuts = false);

// Prediction of the n rows that row_ptr addresses (entry offsets into col / val); out[t * out_stride + i] for
// class tree t and row i, out_stride = 0 means n (a slice of a larger row set passes the whole set's size); adds to out.
// `packed` (optional): the same nodes as 16-byte records (launch_pack_model); with them the trees are walked from LDS.
// For the models that launch_score's records do not describe, and for the entry point that allocates nothing.
void launch_predict(hipStream_t s, int n, int F, const int *row_ptr, const int *col, const float *val,
                    const TreeNode *model, int n_iter, int n_class_trees, int n_nodes, float lr, float base_score,
                    float *out, size_t out_stride = 0, const struct PackedNode *packed = nullptr);
// What a traversal reads of a node, in one 16-byte record.
struct PackedNode {
    float split_value, base_weight;
    unsigned children;  // left | right << 16 (a tree has at most 2^15 - 1 nodes)
    unsigned meta;      // split feature (24 bits, all ones: not a feature of the data) | default_right << 30 | leaf << 31
};
void launch_pack_model(hipStream_t s, const TreeNode *model, long n_total, int n_nodes, PackedNode *packed);

// A model as the scoring kernels read it. The features that its splits use are numbered 0 .. n_used - 1 (ascending);
// a row is spread into keys of these slots, whatever the number of columns of the data. Slot n_used is the leaves' (its
// key is zero), slot n_used + 1 that of features no data can have (always missing).
// Records of eight bytes for models whose trees keep the two children of a node side by side and below it (every tree
// the trainer builds, and the reference's: heap order):
//   x: a split: key(threshold) + (default left ? 1 : 0) - 1, so that "goes right" is `value key + that one > x`;
//      a leaf: the bits of its weight
//   y: slot of the split feature (15 bits; a leaf: slot n_used, whose key never exceeds x)
//      | byte offset of the left child in the tree << 15 (16 bits; a leaf: of the leaf itself)
//      | default left << 31 (a leaf: 0)
// A leaf therefore walks to itself, and a walk of `depth` steps needs no test for the end.
// The model is stored round by round; the records class by class, so that the trees a workgroup stages together
// (consecutive rounds of one class) are one contiguous run.
struct ScoreModel {
    const uint2 *records = nullptr;  // [n_class][n_iter][n_nodes]
    const int *used = nullptr;       // [n_used] feature of every slot
    const int *slot_of = nullptr;    // [n_features + 1] slot of a feature, -1: not used
    int n_used = 0, n_slots = 0, leaf_slot = 0, n_features = 0;
    int n_iter = 0, n_class = 0, n_nodes = 0, depth = 0;
};
struct ScoreRows {
    int n = 0;
    const float *x = nullptr;  // dense [n][columns], else the CSR arrays
    int columns = 0;
    bool minus_zero_is_stored = false;
    const int *row_ptr = nullptr, *col = nullptr;
    const float *val = nullptr;
};
// Scores of the rows: out[t * out_stride + i] is set. narrow: the reference's shared-memory path (at most 96 features in
// the data: double sums, a stored +inf or NaN counts as missing), else its global-memory path (float sums).
// false: the rows' keys fit no kernel's LDS and nothing was launched.
bool launch_score(hipStream_t s, const ScoreRows &rows, const ScoreModel &model, bool narrow, float lr, float base_score,
                  float *out, size_t out_stride);
int score_slice_rows(const ScoreModel &m);  // rows that fill the chip once, in a launch of their own
int score_least_rows(const ScoreModel &m);  // the fewest that k_score_rows serves
// k_score_rows has room for the model's keys; it then serves score_least_rows rows and more.
bool score_rows_fit(const ScoreModel &model);
// Below this many rows k_score_group takes them (see there); with several classes, which k_score_rows shares out, below their part of
// it: the same number of walks of one class. Whole calls with k_score_group and k_score_rows, us: 22 k x 28, 3 x 33 trees of depth 8
// 225, 177; 13 200 rows, 5 x 20 169, 143; 30 k 299, 212; 8200 rows, 8 x 12 123, 113; 30 k one-hot rows, 6 x 15 310, 278.
constexpr int kScoreGroupRows = 65536;
void launch_predict_transform(hipStream_t s, int kind, int n, int num_class, const float *label, float *y);

}  // namespace tgbm
