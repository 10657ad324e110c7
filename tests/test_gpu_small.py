"""Small data: the levels in one launch each (k_small_level, k_map_end) against the launches of larger data (TGBM_SMALL=0), byte
for byte, at the edges of their range."""
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


def _table(n, F, filled, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, F)).astype(np.float32)
    X[rng.random((n, F)) >= filled] = 0
    rp = np.zeros(n + 1, np.int32)
    np.cumsum((X != 0).sum(1), out=rp[1:])
    r, c = np.nonzero(X)
    z = X[:, 0] - 2 * np.abs(X[:, F // 2]) + (X[:, -1] > 0.3) + 0.3 * rng.standard_normal(n)
    return (X[r, c], rp, c.astype(np.int32)), z


CASES = [
    # rows, columns, share of stored values, bins, depth, objective
    (12288, 28, 1.0, 255, 8, "reg:linear"), (12287, 28, 0.6, 255, 6, "binary:logistic"), (8192, 64, 0.9, 63, 7, "reg:linear"),
    (8193, 40, 0.7, 255, 7, "binary:logistic"), (10241, 9, 1.0, 31, 9, "multi:softmax"), (12288, 100, 0.9, 255, 5, "reg:linear"),
    (8192, 11, 0.8, 1024, 7, "binary:logistic"), (4097, 5, 1.0, 700, 6, "reg:linear"),
    (4097, 100, 1.0, 255, 5, "binary:logistic"), (3000, 7, 0.5, 1024, 6, "reg:linear"), (1025, 3, 1.0, 16, 10, "reg:logistic"),
    (5000, 12, 1.0, 255, 6, "multi:softmax"), (40, 5, 0.7, 255, 4, "reg:linear"), (2, 2, 1.0, 255, 2, "reg:linear"),
    (600, 4, 1.0, 255, 1, "reg:linear"),
]


@pytest.mark.parametrize("n,F,filled,bins,depth,objective", CASES)
@pytest.mark.parametrize("sampled", [False, True])
def test_small_levels_equal_large_ones(T, n, F, filled, bins, depth, objective, sampled):
    (val, rp, col), z = _table(n, F, filled, n)
    y = z.astype(np.float32)
    kw = {}
    if objective == "multi:softmax":
        y, kw["num_class"] = np.digitize(z, [-1, 0, 1]).astype(np.float32), 4
    elif "logistic" in objective:
        y = (z > np.median(z)).astype(np.float32)
    runs = []
    try:
        for small in ("1", "0"):
            os.environ["TGBM_SMALL"] = small
            ctypes.CDLL(None).srand(3)
            s = T.Session(val, rp, col, y, objective=objective, depth=depth, n_trees=5, max_num_bin=bins, learning_rate=0.5,
                          gamma=0.5, **kw)
            assert s.info("small_levels") == int(small)
            if sampled:
                s.set_option("bagging", 1)
                s.set_option("column_sampling_rate", 0.4)
            s.boost(3)
            s.boost(2)
            runs.append((s.model().tobytes(), s.y_pred().tobytes(), s.nid().tobytes(), np.round(s.metric_log(), 5).tobytes(),
                         s.nodes().tobytes()))
            s.close()
    finally:
        del os.environ["TGBM_SMALL"]
    assert runs[0] == runs[1]


@pytest.mark.parametrize("n,bins,small", [(12288, 255, True), (12289, 255, False), (8192, 1024, True), (8193, 1024, False)])
def test_where_the_range_ends(T, n, bins, small):
    (val, rp, col), z = _table(n, 5, 1.0, n)
    s = T.Session(val, rp, col, z.astype(np.float32), depth=6, n_trees=1, max_num_bin=bins)
    assert s.info("wide_eval") == int(bins > 255)
    assert s.info("small_levels") == int(small) and (s.info("split_hist_rows") > 0) == (not small)
    s.close()
