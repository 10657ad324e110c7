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
