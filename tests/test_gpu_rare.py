"""Rare features of the sparse layout: the filtered search (k_sparse_rare_filter, k_sparse_rare_search) against the complete
(bin, node) tables (TGBM_SPARSE_SORTED=0: every feature through them), byte for byte, at the edges of its tiles."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    import thundergbm_amd
    thundergbm_amd.load()
    return thundergbm_amd


def _by_feature(counts, n, seed):
    """CSR of features with the given numbers of stored values, in random rows."""
    rng = np.random.default_rng(seed)
    rows = np.concatenate([rng.choice(n, k, replace=False) for k in counts])
    cols = np.repeat(np.arange(len(counts), dtype=np.int32), counts)
    order = np.lexsort((cols, rows))
    rp = np.zeros(n + 1, np.int64)
    np.cumsum(np.bincount(rows, minlength=n), out=rp[1:])
    val = np.exp(rng.standard_normal(len(rows))).astype(np.float32)
    z = np.zeros(n)
    w = rng.standard_normal(len(counts)) * (rng.random(len(counts)) < 0.3)
    np.add.at(z, rows[order], w[cols[order]] * val)
    return val, rp.astype(np.int32), cols[order], z + 0.3 * rng.standard_normal(n)


SHAPES = {
    "single_values": ([1] * 5000 + [2] * 3000, 9000),              # more features than a tile takes
    "tile_edges": ([4096, 4097, 4095, 1, 4096, 2048, 2048, 1, 4097], 5000),
    "two_tiles_a_group": ([20000] * 3 + [4000, 3000] + [190] * 11500, 60000),
    "everything_rare": ([300] * 60, 2000),                         # the tables publish next to nothing
}


# The most frequent features go to tables whatever they hold (kRareExempt, kRareLeast): shapes around that rule, and around a
# search with a value per thread.
FREQUENT = {
    "full_tiles": ([4500] * 128 + [4096, 4097, 4095, 1, 4096, 2048, 2048, 1], 5000),
    "few_rows": ([257] * 60 + [256, 255, 1, 256, 256, 128, 128, 257, 2] * 8, 300),
    "tiles_around_512": ([900] * 128 + [700, 512, 513, 1, 511] * 6, 1000),
    "one_feature_more": ([400] * 129 + [400, 300], 600),
    "few_values": ([3] * 20, 50),
    "only_rare": ([250] * 70, 2000),                               # the tables publish next to nothing
}
RARE_VALUES = {  # (feature 0 owns bin 0 and goes to a table whatever it holds)
    "full_tiles": 4096 + 4095 + 1 + 4096 + 2048 + 2048 + 1, "few_rows": (256 + 255 + 1 + 256 + 256 + 128 + 128 + 2) * 8,
    "tiles_around_512": (700 + 512 + 513 + 1 + 511) * 6, "one_feature_more": 129 * 400 + 300, "few_values": 19 * 3, "only_rare": 69 * 250,
}
OPTIONS = pytest.mark.parametrize("objective,kw", [
    ("reg:linear", {}), ("binary:logistic", {"min_child_weight": 5.0}), ("multi:softmax", {"num_class": 3}),
    ("reg:linear", {"lambda_": 0.0, "min_child_weight": 0.0, "sampled": True})])


@pytest.mark.parametrize("shape", sorted(FREQUENT))
@OPTIONS
def test_features_at_the_edge_of_rare_equal_tables(T, shape, objective, kw):
    val, rp, col, z = _by_feature(*FREQUENT[shape], 5)
    compare(T, val, rp, col, (z - np.median(z)) / z.std(), objective, kw, RARE_VALUES[shape])


@pytest.mark.parametrize("shape", sorted(SHAPES))
@OPTIONS
def test_rare_features_equal_tables(T, shape, objective, kw):
    counts, n = SHAPES[shape]
    val, rp, col, z = _by_feature(counts, n, 5)
    compare(T, val, rp, col, z, objective, kw)


def compare(T, val, rp, col, z, objective, kw, rare_values=None):
    kw = dict(kw)
    sampled = kw.pop("sampled", False)
    y = (z if objective == "reg:linear" else np.digitize(z, [-0.5, 0.5][: 2 if "multi" in objective else 1])).astype(np.float32)
    runs = []
    os.environ["TGBM_LAYOUT"] = "sparse"
    try:
        for rare in ("1", "0"):
            os.environ["TGBM_SPARSE_SORTED"] = rare
            ctypes.CDLL(None).srand(7)
            s = T.Session(val, rp, col, y, objective=objective, depth=7, n_trees=3, max_num_bin=63, learning_rate=0.5, **kw)
            assert s.info("sparse_pass") == 1
            assert rare == "1" or s.info("sparse_rare_values") == 0
            assert rare == "0" or rare_values is None or s.info("sparse_rare_values") == rare_values
            if sampled:
                s.set_option("bagging", 1)
                s.set_option("column_sampling_rate", 0.5)
            s.boost(3)
            runs.append((s.model().tobytes(), s.y_pred().tobytes()))
            s.close()
    finally:
        del os.environ["TGBM_SPARSE_SORTED"], os.environ["TGBM_LAYOUT"]
    assert runs[0] == runs[1]


# Values brought to by blocks of 32 768 rows (TGBM_SPARSE_SPREAD) against values that look their rows up: rows at the edges of blocks,
# a block without values, a task's last group of places, more than 128 nodes in a level, class trees built together.
@pytest.mark.parametrize("n,depth", [(300, 4), (32768, 3), (32769, 6), (100003, 10)])
@pytest.mark.parametrize("objective,kw", [("reg:linear", {}), ("binary:logistic", {"min_child_weight": 0.0}), ("multi:softmax", {"num_class": 3})])
def test_spread_values_equal_looked_up_ones(T, n, depth, objective, kw):
    rng = np.random.default_rng(n)
    counts = np.minimum(n // 2, np.concatenate([[6000] * 3, rng.integers(1, 900, 200), [1] * 2100, [4095, 4096, 2, 3, 4, 5]]))
    val, rp, col, z = _by_feature([int(k) for k in counts], n, 5)
    if n > 65536:  # (nothing is stored in the rows of the second block)
        rp = rp.astype(np.int64)
        keep = np.ones(len(col), bool)
        keep[rp[32768]:rp[65536]] = False
        cut = np.concatenate([[0], np.cumsum(keep)])
        val, col, rp = val[keep], col[keep], cut[rp].astype(np.int32)
    y = (z if objective == "reg:linear" else np.digitize(z, [-0.5, 0.5][: 2 if "multi" in objective else 1])).astype(np.float32)
    runs = []
    os.environ["TGBM_LAYOUT"] = "sparse"
    try:
        for spread in ("1", "0"):
            os.environ["TGBM_SPARSE_SPREAD"] = spread
            s = T.Session(val, rp, col, y, objective=objective, depth=depth, n_trees=3, max_num_bin=63, learning_rate=0.5, **kw)
            assert s.info("sparse_spread_blocks") == (-(-n // 32768) if spread == "1" else 0)
            s.boost(2)
            got = [s.model().tobytes(), s.y_pred().tobytes()]
            if s.tree_per_rounds == 1:  # (stage by stage the levels leave their nodes' histograms too)
                s.gradient()
                s.tree_init()
                for level in range(depth):
                    s.find_split(level)
                    if level < 5:
                        got.append(s.level_hist(level).tobytes())
                    s.partition(level)
                s.finish_tree()
                got.append(s.model().tobytes())
            runs.append(got)
            s.close()
    finally:
        os.environ.pop("TGBM_SPARSE_SPREAD", None)
        del os.environ["TGBM_LAYOUT"]
    assert runs[0] == runs[1]


# The pass over the tables: bins of a lane (up to 64 bins or up to 255), the pairs as words or as pairs, copied to the values or fetched by
# row, the nodes brought to the values or looked up; levels whose tables share a CU and levels whose don't; features in chunks.
@pytest.mark.parametrize("bins", [31, 255])
@pytest.mark.parametrize("objective", ["reg:linear", "binary:logistic"])
def test_tables_whatever_form_their_values_have(T, objective, bins):
    n = 40000
    counts = [n - 1, 33000, 32769, 9000, 5000, 5001, 5002, 5003] + [300] * 60 + [5] * 40
    val, rp, col, z = _by_feature(counts, n, 7)
    y = (z if objective == "reg:linear" else np.digitize(z, [-0.5])).astype(np.float32)
    runs = []
    os.environ["TGBM_LAYOUT"] = "sparse"
    try:
        for spread, word, copy in [("0", "1", "1"), ("1", "1", "1"), ("0", "0", "1"), ("1", "0", "1"), ("0", "1", "0"), ("1", "1", "0"), ("1", "0", "0")]:
            os.environ.update(TGBM_SPARSE_SPREAD=spread, TGBM_GH_WORD=word, TGBM_SPARSE_GH_COPY=copy)
            s = T.Session(val, rp, col, y, objective=objective, depth=7, n_trees=2, max_num_bin=bins, learning_rate=0.5)
            s.boost(2)
            runs.append((s.model().tobytes(), s.y_pred().tobytes()))
            s.close()
    finally:
        for key in ("TGBM_LAYOUT", "TGBM_SPARSE_SPREAD", "TGBM_GH_WORD", "TGBM_SPARSE_GH_COPY"):
            os.environ.pop(key, None)
    assert all(r == runs[0] for r in runs)


# Values of frequent features that several workgroups of the set-up give their places: a part's edge inside a group of four places, at a row
# block's edge and next to a block without values; the levels' histograms against the bins themselves.
@pytest.mark.parametrize("n", [40001, 100003])
def test_frequent_features_in_parts(T, n):
    counts = [min(k, n - 1) for k in (8191, 8192, 8193, 16384, 16390, 33000, n - 1, 70000)] + [900] * 130 + [20] * 10
    val, rp, col, z = _by_feature(counts, n, 11)
    if n > 65536:  # (nothing is stored in the rows of the second block)
        keep = np.ones(len(col), bool)
        keep[rp[32768]:rp[65536]] = False
        rp = np.concatenate([[0], np.cumsum(keep)])[rp].astype(np.int32)
        val, col = val[keep], col[keep]
    runs = []
    os.environ["TGBM_LAYOUT"] = "sparse"
    try:
        for spread in ("1", "0"):
            os.environ["TGBM_SPARSE_SPREAD"] = spread
            s = T.Session(val, rp, col, z.astype(np.float32), depth=5, n_trees=3, max_num_bin=63, learning_rate=0.5)
            bins = s.global_bin_ids(rp, col)[0]
            gh = np.ones((n, 2), np.float32)
            gh[:, 0] = np.arange(n) % 7 - 3  # (whole numbers: the histograms are exact)
            s.set("gh", gh)
            s.tree_init(0)
            s.find_split(0)
            row = np.repeat(np.arange(n), np.diff(rp))
            want = np.stack([np.bincount(bins, gh[row, k], minlength=s.n_bins) for k in (0, 1)], 1)
            assert np.array_equal(s.level_hist(0)[0], want)
            s.close()
            s = T.Session(val, rp, col, z.astype(np.float32), depth=5, n_trees=3, max_num_bin=63, learning_rate=0.5)
            s.boost(3)
            runs.append((s.model().tobytes(), s.y_pred().tobytes()))
            s.close()
    finally:
        os.environ.pop("TGBM_SPARSE_SPREAD", None)
        del os.environ["TGBM_LAYOUT"]
    assert runs[0] == runs[1]


# Spread values where columns are sampled (their segments and values take no part, in tables with kept records and in the filter) and rows are
# resampled (pairs instead of words), against looked-up values and against tables for every feature; 31 and 255 bins (one bin of a lane, four).
@pytest.mark.parametrize("bagging", [0, 1])
@pytest.mark.parametrize("objective,kw", [("reg:linear", {}), ("binary:logistic", {"min_child_weight": 0.0}), ("multi:softmax", {"num_class": 3})])
@pytest.mark.parametrize("bins", [31, 255])
def test_spread_values_of_sampled_columns(T, bins, objective, kw, bagging):
    n = 40000
    counts = [n - 1, 33000, 32769, 9000, 5000] + [700] * 130 + [300] * 60 + [4, 5, 1] * 20
    val, rp, col, z = _by_feature(counts, n, 3)
    y = (z if objective == "reg:linear" else np.digitize(z, [-0.5, 0.5][: 2 if "multi" in objective else 1])).astype(np.float32)
    runs = []
    os.environ["TGBM_LAYOUT"] = "sparse"
    try:
        for spread, rare in (("1", "1"), ("0", "1"), ("1", "0")):
            os.environ.update(TGBM_SPARSE_SPREAD=spread, TGBM_SPARSE_SORTED=rare)
            ctypes.CDLL(None).srand(7)
            s = T.Session(val, rp, col, y, objective=objective, depth=7, n_trees=3, max_num_bin=bins, learning_rate=0.5, **kw)
            assert s.info("sparse_spread_blocks") == (2 if spread == "1" else 0)
            assert (s.info("sparse_rare_values") > 0) == (rare == "1")
            s.set_option("bagging", bagging)
            s.set_option("column_sampling_rate", 0.5)
            s.boost(3)
            runs.append((s.model().tobytes(), s.y_pred().tobytes()))
            s.close()
    finally:
        for key in ("TGBM_LAYOUT", "TGBM_SPARSE_SPREAD", "TGBM_SPARSE_SORTED"):
            os.environ.pop(key, None)
    assert runs[0] == runs[1] and runs[0] == runs[2]
