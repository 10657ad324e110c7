"""The level kernels of the dense layout (thundergbm_amd/csrc/level_kernels.hip): what boost() runs in fewer launches
against the stages one by one, at the edges of the work items and of the nodes a workgroup looks at together."""
import ctypes
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import datasets as D  # noqa: E402

pytestmark = pytest.mark.gpu


def one_by_one(s, rounds, depth, K):
    for _ in range(rounds):
        s.gradient()
        for k in range(K):
            s.tree_init(k)
            for level in range(depth):
                s.find_split(level)
                s.partition(level)
            s.finish_tree(k)


@pytest.mark.parametrize("n,F,depth,bins,objective", [
    (1, 1, 1, 255, "reg:linear"), (2047, 3, 2, 255, "reg:linear"), (2048, 5, 4, 16, "binary:logistic"),
    (2049, 130, 5, 255, "reg:linear"), (20_480, 9, 8, 255, "binary:logistic"), (20_481, 4, 11, 64, "reg:linear"),
    (5000, 12, 6, 1000, "reg:linear"), (4500, 8, 5, 255, "multi:softmax"), (300_000, 6, 9, 255, "reg:logistic")])
def test_boost_equals_the_stages(n, F, depth, bins, objective):
    import thundergbm_amd as T
    rng = np.random.default_rng(n + F)
    X = rng.standard_normal((n, F)).astype(np.float32)
    X[rng.random((n, F)) < 0.1] = 0
    X[0, 0] = 1.0
    z = X[:, 0] + np.abs(X[:, F // 2]) + 0.3 * rng.standard_normal(n)
    K = 3 if objective.startswith("multi") else 1
    y = z if objective == "reg:linear" else (np.digitize(z, [0, 1]) if K > 1 else z > 0.5)
    y = np.asarray(y, np.float32)
    val, rp, col = D.dense_to_csr(X)
    models, maps, preds = [], [], []
    for stages in (False, True):
        s = T.Session(val, rp, col, y, depth=depth, n_trees=3, learning_rate=0.5, max_num_bin=bins, objective=objective,
                      min_child_weight=0.5)
        if stages:
            one_by_one(s, 3, depth, K)
        else:
            s.boost(3)
        models.append(s.model().tobytes())
        maps.append(s.nid())
        preds.append(s.y_pred())
        s.close()
    assert models[0] == models[1]
    assert np.array_equal(maps[0], maps[1])
    assert np.array_equal(preds[0], preds[1])


@pytest.mark.parametrize("n", [256 * 2048 + 1, 1_300_001, (1 << 24) - 1, 1 << 24])
def test_rows_of_nodes_of_many_items(n):
    """Nodes of more work items than a workgroup has threads, below and above the rows from which on their counts are added up
    by groups: every node holds the rows that its path leads there (squared loss: the hessians count them, exactly up to
    2^24)."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    X = rng.integers(1, 1000, (n, 2)).astype(np.float32)
    y = (np.floor(X[:, 0] / 100) + (X[:, 1] > 700) * (X[:, 0] > 300) + 0.1 * rng.standard_normal(n)).astype(np.float32)
    s = T.Session(X.reshape(-1), np.arange(0, 2 * n + 1, 2, dtype=np.int32), np.tile(np.arange(2, dtype=np.int32), n), y,
                  depth=5, n_trees=2, learning_rate=0.5, gamma=0.0)
    s.boost(2)
    for tree in s.model().reshape(2, -1):
        node = np.zeros(n, np.int64)
        for _ in range(6):
            rows = np.bincount(node, minlength=len(tree))
            at = np.unique(node)
            assert np.array_equal(tree["sum_h"][at], rows[at])
            inner = ~tree["is_leaf"][node].astype(bool)
            left = X[np.arange(n), np.maximum(tree["split_fid"][node], 0)] < tree["split_value"][node]
            node = np.where(inner, np.where(left, tree["lch"][node], tree["rch"][node]), node)
    assert np.array_equal(s.nid(), node)
    s.close()


@pytest.mark.parametrize("items,n,F,depth,bins,objective,missing", [
    (1, 16_385, 4, 8, 255, "binary:logistic", 0.0), (1, 30_000, 3, 10, 16, "reg:linear", 0.3), (1, 20_480, 30, 5, 63, "binary:logistic", 0.1),
    (1, 65_535, 9, 8, 1000, "reg:linear", 0.1), (2, 65_536, 21, 7, 255, "multi:softmax", 0.1), (2, 240_000, 28, 8, 255, "reg:logistic", 0.0),
    (2, 70_001, 9, 8, 1000, "reg:linear", 0.1), (2, 500_001, 28, 8, 255, "binary:logistic", 0.05), (2, 50_000, 260, 6, 255, "reg:linear", 0.0),
    (2, 1_048_575, 16, 7, 255, "reg:linear", 0.0), (4, 1_000_001, 28, 7, 255, "binary:logistic", 0.0), (4, 70_001, 400, 5, 255, "reg:linear", 0.1),
    (4, 300_001, 28, 6, 1000, "reg:linear", 0.1)])
def test_lists_and_histograms_in_one_launch(items, n, F, depth, bins, objective, missing, monkeypatch):
    """k_split_hist against the scatter and histogram launches: 1, 2 and 4 partition items a workgroup, records with and
    without gradient words, 16-bit bins, several blocks, class trees, sorted rows (all rows of a child in one workgroup)."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, F)).astype(np.float32)
    X = X[np.argsort(X[:, 0])]
    X[rng.random((n, F)) < missing] = 0
    z = X[:, 0] + np.abs(X[:, F // 2]) + 0.3 * rng.standard_normal(n)
    y = z if objective == "reg:linear" else (np.digitize(z, [0, 1]) if objective.startswith("multi") else z > 0.5)
    val, rp, col = D.dense_to_csr(X)
    out = []
    for switch in ("1", "0"):
        monkeypatch.setenv("TGBM_SPLIT_HIST", switch)
        s = T.Session(val, rp, col, np.asarray(y, np.float32), depth=depth, n_trees=3, learning_rate=0.5, max_num_bin=bins,
                      objective=objective)
        assert s.info("split_hist_rows") == (2048 * items if switch == "1" else 0)
        s.boost(3)
        out.append((s.model().tobytes(), s.nid().tobytes(), s.y_pred().tobytes(), s.metric_log().tobytes()))
        s.close()
    same = [a == b for a, b in zip(*out)]
    assert all(same), same


@pytest.mark.parametrize("n,depth,bins,objective,rate", [
    (1_200, 6, 1024, "reg:linear", 1.0), (8_000, 7, 1024, "binary:logistic", 1.0), (8_192, 5, 513, "reg:linear", 0.5),
    (5_000, 6, 1500, "reg:linear", 1.0), (6_000, 4, 300, "multi:softmax", 1.0)])
def test_merge_and_search_of_wide_features_in_one_launch(n, depth, bins, objective, rate, monkeypatch):
    """k_merge_eval_wide (TGBM_SMALL=0) against k_eval_split_wide after k_small_level: columns of 1 .. `bins` values, 0 to 4
    quarters of 256 bins full or with a remainder, ties between columns, features past the one launch's bins (1500)."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    counts = [c for c in (1, 2, 255, 256, 257, 512, 513, 768, 1023, 1024, 1025, 1500) if c <= bins] + [256]
    X = np.stack([rng.permutation(np.arange(n) % c) + 1 for c in counts], 1).astype(np.float32)
    X[:, -1] = X[:, counts.index(256)]
    X[rng.random(X.shape) < 0.1] = 0
    z = X[:, 2] / 255 + np.abs(X[:, -2] / counts[-2] - 0.5) + 0.3 * rng.standard_normal(n)
    y = z if objective == "reg:linear" else (np.digitize(z, [0.7, 1.0]) if objective.startswith("multi") else z > 0.8)
    val, rp, col = D.dense_to_csr(X)
    out = []
    for small in ("1", "0"):
        monkeypatch.setenv("TGBM_SMALL", small)
        ctypes.CDLL(None).srand(3)
        s = T.Session(val, rp, col, np.asarray(y, np.float32), depth=depth, n_trees=3, learning_rate=0.5, max_num_bin=bins,
                      objective=objective)
        assert s.info("wide_eval") == 1
        if rate < 1:
            s.set_option("column_sampling_rate", rate)
        s.boost(3)
        out.append((s.model().tobytes(), s.nid().tobytes(), s.y_pred().tobytes(), np.round(s.metric_log(), 5).tobytes()))
        s.close()
    assert out[0] == out[1]


@pytest.mark.parametrize("n,groups,numbers,depth,objective,rate", [
    (1_600, (9, 16, 41), 5, 6, "binary:logistic", 1.0), (7_000, (3, 120), 17, 7, "reg:linear", 0.4), (8_192, (40,), 0, 5, "reg:linear", 1.0),
    (3_000, (6, 7, 8, 9), 30, 6, "multi:softmax", 1.0), (2_500, (), 70, 4, "reg:linear", 1.0), (257, (5,), 2, 10, "reg:logistic", 1.0)])
def test_search_of_few_rows_with_the_lists(n, groups, numbers, depth, objective, rate, monkeypatch):
    """k_small_level with the next level's split search in it against the launches of larger data: columns that hold a one-hot
    group of features, columns without a value, parts of 4, 8 and 16 columns and wider ones, class trees, sampled columns."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    hot = [np.eye(g, dtype=np.float32)[rng.integers(0, g, n)] for g in groups]
    X = np.concatenate(hot + [rng.standard_normal((n, numbers)).astype(np.float32)], 1)
    X[:, X.shape[1] // 2] = 0
    X[rng.random(n) < 0.05] = 0
    z = X @ rng.standard_normal(X.shape[1]) / 3 + 0.3 * rng.standard_normal(n)
    y = z if objective == "reg:linear" else (np.digitize(z, [-0.3, 0.3]) if objective.startswith("multi") else z > 0)
    val, rp, col = D.dense_to_csr(X)
    out = []
    for small in ("1", "0"):
        monkeypatch.setenv("TGBM_SMALL", small)
        ctypes.CDLL(None).srand(3)
        s = T.Session(val, rp, col, np.asarray(y, np.float32), depth=depth, n_trees=4, learning_rate=0.5, objective=objective)
        if rate < 1:
            s.set_option("column_sampling_rate", rate)
        s.boost(3)
        s.boost(1)
        out.append((s.model().tobytes(), s.nid().tobytes(), s.y_pred().tobytes(), np.round(s.metric_log(), 5).tobytes()))
        s.close()
    assert out[0] == out[1]


@pytest.mark.parametrize("n,objective,bins,empty,descending", [
    (3_000, "reg:linear", 1024, 8, False), (20_000, "binary:logistic", 1024, 8, False), (70_000, "multi:softmax", 1024, 8, False),
    (20_000, "reg:linear", 255, 64, True)])
@pytest.mark.parametrize("route", ["boost", "launches", "stages"])
def test_first_block_without_bins(n, objective, bins, empty, descending, route, monkeypatch):
    """The first feature block stores an item's scales and the rows' sums for all of them. Its columns may hold no value at all
    (16-bit bins and rows whose columns do not ascend are not bundled): the same data with those columns last."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    F = 37 if bins > 255 else 90
    X = rng.permuted(np.tile(np.arange(n) % 1000 + 1, (F, 1)), axis=1).T.astype(np.float32)
    X[rng.random((n, F)) < 0.3] = 0  # (no column is stored in every row)
    X[:, :empty] = 0
    z = X[:, empty] / 500 + np.abs(X[:, -1] / 500 - 1) + 0.3 * rng.standard_normal(n)
    K = 3 if objective.startswith("multi") else 1
    y = z if objective == "reg:linear" else (np.digitize(z, [0.8, 1.4]) if K > 1 else z > 1)
    if route == "launches":
        monkeypatch.setenv("TGBM_SPLIT_HIST", "0")
        monkeypatch.setenv("TGBM_SMALL", "0")
    out = []
    for shift in (0, empty):
        val, rp, col = D.dense_to_csr(np.roll(X, -shift, axis=1))
        if descending:
            order = np.lexsort((-col, np.repeat(np.arange(n), np.diff(rp))))
            val, col = val[order], col[order]
        s = T.Session(val, rp, col, np.asarray(y, np.float32), depth=6, n_trees=3, learning_rate=0.5, max_num_bin=bins, objective=objective)
        assert shift > 0 or s.info("dense_W") == empty
        if route == "stages":
            one_by_one(s, 3, 6, K)
        else:
            s.boost(3)
        model = s.model()
        model["split_fid"][model["split_fid"] >= 0] += shift
        out.append((model.tobytes(), s.y_pred().tobytes(), s.nid().tobytes()))
        s.close()
    assert np.any(model["split_fid"] >= empty)
    same = [a == b for a, b in zip(*out)]  # (a failed comparison of the bytes themselves is printed for minutes)
    assert all(same), same


@pytest.mark.parametrize("n,F", [(500_001, 28), (60_000, 300)])
def test_work_items_of_the_stages(n, F):
    """boost() halves the root's work items where the levels below are built by k_split_hist. Stage by stage they are
    k_hist_dense's, which wants two workgroups per CU."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, F)).astype(np.float32)
    y = X[:, 0] + np.abs(X[:, 1])
    s = T.Session(*D.dense_to_csr(X), y, depth=6, n_trees=2, learning_rate=0.5)
    target = 512 // s.info("dense_blocks")
    items = []
    for step in (lambda: s.boost(1), lambda: one_by_one(s, 1, 6, 1)):
        step()
        chunk, count = s.get("ctl", np.int32).reshape(-1, 4)[0][:2]
        assert count == -(-n // chunk)
        items.append(count)
    s.close()
    assert items[0] <= target // 2 < items[1] <= target


@pytest.mark.parametrize("n,F,bins,depth,K,served", [(60_000, 100, 16, 8, 1, True), (60_000, 100, 16, 11, 1, False),
                                                     (60_000, 400, 255, 6, 8, False), (1_048_576, 70, 8, 5, 1, False)])
def test_room_for_runs_where_there_are_runs(n, F, bins, depth, K, served, monkeypatch):
    """The workgroups of k_split_hist store more histograms than the other launches' work items where the features have few bins:
    room for them is taken where that kernel serves the data, and is enough there."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n + K)
    X = rng.integers(1, bins, (n, F)).astype(np.float32) if bins < 255 else rng.standard_normal((n, F)).astype(np.float32)
    z = X[:, 0] + 2 * np.abs(X[:, 1])
    y = z if K == 1 else np.digitize(z, np.quantile(z, np.arange(1, K) / K))
    kw = dict(depth=depth, n_trees=1, max_num_bin=bins, objective="reg:linear" if K == 1 else "multi:softmax", num_class=K)
    room = []
    for switch in ("1", "0"):
        monkeypatch.setenv("TGBM_SPLIT_HIST", switch)
        s = T.Session(X.reshape(-1), np.arange(0, n * F + 1, F, dtype=np.int32), np.tile(np.arange(F, dtype=np.int32), n), y.astype(np.float32), **kw)
        room.append(s.info("partial_histograms"))
        rows = s.info("split_hist_rows")
        assert (rows > 0) == (served and switch == "1")
        if rows:
            assert 2 * room[0] >= n // rows + 2 ** (depth - 2) + 1
        s.close()
    assert served or room[0] == room[1]


@pytest.mark.parametrize("n,switch,own", [(5_000, "TGBM_SMALL", False), (40_000, "TGBM_SPLIT_HIST", False), (40_000, "TGBM_SPLIT_HIST", True)])
def test_profile_counts_histogram_launches(n, switch, own, monkeypatch):
    """Levels whose histograms are built by the partition's launch have no histogram launch, time or bytes of their own."""
    import thundergbm_amd as T
    monkeypatch.setenv(switch, "0" if own else "1")
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 12)).astype(np.float32)
    s = T.Session(*D.dense_to_csr(X), X[:, 0] + np.abs(X[:, 1]), depth=5, n_trees=3)
    s.set_profiling(True)
    s.boost(3)
    hist = s.phase_profile()["hist"]
    s.close()
    assert hist["root"]["launches"] == 3 and hist["root"]["bytes"] == 3 * n * (12 + 8)
    assert hist["below_root"]["launches"] == (12 if own else 0)
    assert (hist["below_root"]["bytes"] > 0) == own and (hist["below_root"]["ms"] > 0) == own


@pytest.mark.parametrize("n,objective", [(60_000, "reg:linear"), (80_001, "binary:logistic")])
def test_merge_and_search_of_many_items_of_wide_features(n, objective):
    """k_merge_eval_wide with sixteen wavefronts, for more than eight work items a pair, 1 to 4 quarters of 256 bins (three leave a
    wavefront without any), against k_hist_merge and k_eval_split_wide: a column of more than kMergeWideBins bins sends all of them
    there. No split of it leaves enough rows on both sides."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    counts = [256, 257, 512, 513, 700, 768, 769, 1023, 1024]
    X = np.zeros((n, len(counts) + 1), np.float32)
    for f, c in enumerate(counts):
        X[:, f] = rng.permutation(np.arange(n) % c) + 1
    X[rng.random(X.shape) < 0.1] = 0
    X[:, -1] = 0
    X[rng.choice(n, 1_500, replace=False), -1] = np.arange(1_500) + 1
    z = X[:, 4] / 700 + np.abs(X[:, 7] / 1023 - 0.5) + X[:, 0] / 256 * (X[:, 3] > 200) + 0.3 * rng.standard_normal(n)
    y = (z if objective == "reg:linear" else z > 1).astype(np.float32)
    out = []
    for columns in (len(counts), len(counts) + 1):
        s = T.Session(*D.dense_to_csr(X[:, :columns]), y, depth=5, n_trees=3, learning_rate=0.5, max_num_bin=1_500, objective=objective,
                      min_child_weight=1_501 if objective == "reg:linear" else 376)
        bins = np.diff(s.cuts()[1])
        assert bins[:len(counts)].tolist() == counts and (columns == len(counts) or bins[-1] == 1_500)
        assert s.info("split_hist_rows") > 0 and n // s.info("split_hist_rows") > 8
        s.boost(3)
        out.append((s.model().tobytes(), s.nid().tobytes(), s.y_pred().tobytes()))
        assert len(np.unique(s.model()["split_fid"])) > 3
        s.close()
    same = [a == b for a, b in zip(*out)]
    assert all(same), same


@pytest.mark.parametrize("n,F,per_row,objective", [(120_000, 2_823, 20, "binary:logistic"), (540_000, 6, 0, "multi:softmax")])
def test_root_of_drained_items(n, F, per_row, objective, monkeypatch):
    """k_merge_eval at the root where the work items have more rows than the LDS adds up packed (few items: many feature blocks or
    classes) and no feature is stored in every row, against k_hist_merge and k_eval_split (an arena that is too small for the last level)."""
    import thundergbm_amd as T
    monkeypatch.setenv("TGBM_LAYOUT", "dense")
    rng = np.random.default_rng(n)
    if per_row:
        col = np.minimum(F * rng.random((n, per_row)) ** 3, F - 1).astype(np.int32)
        col.sort(axis=1)
        keep = np.ones(col.shape, bool)
        keep[:, 1:] = col[:, 1:] != col[:, :-1]
        rp = np.concatenate([[0], np.cumsum(keep.sum(1))]).astype(np.int32)
        z = 0.3 * (col % 7 == 0).sum(1) - 0.2 * (col < 40).sum(1) + 0.5 * rng.standard_normal(n)
        col = col[keep]
        val = np.exp(rng.standard_normal(col.size)).astype(np.float32)
    else:
        X = rng.standard_normal((n, F)).astype(np.float32)
        X[rng.random(X.shape) < 0.1] = 0
        z = X[:, 0] + np.abs(X[:, 1])
        val, rp, col = D.dense_to_csr(X)
    K = 8 if objective.startswith("multi") else 1
    y = np.digitize(z, np.quantile(z, np.arange(1, K) / K)) if K > 1 else z > np.median(z)
    out = []
    for nodes in (None, None, "4"):
        if nodes:
            monkeypatch.setenv("TGBM_HIST_ARENA_NODES", nodes)
        s = T.Session(val, rp, col, y.astype(np.float32), depth=4, n_trees=2, learning_rate=0.3, objective=objective, num_class=K)
        s.boost(2)
        out.append((s.model().tobytes(), s.nid().tobytes(), s.y_pred().tobytes()))
        if nodes is None:
            chunk, items = s.get("ctl", np.int32).reshape(-1, 4)[0][:2]
            assert chunk > 8192 and items <= 64
        s.close()
    same = [[a == b for a, b in zip(o, out[-1])] for o in out[:-1]]
    assert np.all(same), same


# Pairs that fill the fields of a packed bin (every row at the largest gradient of one sign, every hessian at the largest, all in one
# bin), at the ends of what an item adds before it is drained (8192 rows with float hessians, 32 768 with whole ones), and one row.
@pytest.mark.parametrize("n", [1, 2, 8191, 8192, 8193, 32769])
@pytest.mark.parametrize("g,h", [(-0.7366291, 0.19483), (1.0, 0.2499999), (3.1e8, 1.0), (-1e-12, 1e-16), (5.0, 3.0)])
def test_pairs_that_fill_their_fields(n, g, h):
    import parity as P
    import thundergbm_amd as T
    X = np.ones((n, 2), np.float32)
    X[:, 1] = np.arange(n) % 3 + 1
    val, rp, col = D.dense_to_csr(X)
    s = T.Session(val, rp, col, np.arange(n).astype(np.float32), depth=2, n_trees=1, objective="reg:linear")
    gh = np.empty((n, 2), np.float32)
    gh[:] = g, h
    s.set("gh", gh)
    s.tree_init(0)
    s.find_split(0)
    q = P.node_quantum(s.quant(), n, False)
    got = s.level_hist(0)[0]
    one = np.rint(gh[0].astype(np.float64) / q) * q
    want = np.bincount(s.global_bin_ids(rp, col)[0], minlength=s.n_bins)[:, None] * one
    assert np.array_equal(got, want)  # (the steps are powers of two and the sums integers below 2^53 of them)
    s.close()


# Class trees whose rows walk them at the end (655 360 rows of all trees on) against the launches that keep row lists, byte for byte: records
# of 4, 8, 16 and 32 bytes, features that share a column, missing values, trees that stop early, an odd number of rows.
# (width: of the records, 0 where the rows are one or two too few)
@pytest.mark.parametrize("n,F,K,depth,hot,width", [
    (163_840, 3, 4, 8, 0, 4), (163_839, 3, 4, 8, 0, 0), (218_455, 7, 3, 6, 0, 8), (131_073, 13, 5, 4, 0, 16), (93_623, 31, 7, 8, 0, 32),
    (131_072, 6, 5, 1, 0, 8), (120_001, 8, 6, 7, 60, 16), (220_000, 2, 3, 10, 30, 4)])
def test_class_trees_are_walked(n, F, K, depth, hot, width, monkeypatch):
    import thundergbm_amd as T
    rng = np.random.default_rng(n + F)
    X = np.zeros((n, F + hot), np.float32)
    X[:, :F] = rng.standard_normal((n, F)).astype(np.float32)
    X[:, :F][rng.random((n, F)) < 0.15] = 0
    group = rng.integers(0, hot + 1, n)
    if hot:
        X[np.arange(n)[group < hot], F + group[group < hot]] = 1
    z = X[:, 0] + np.abs(X[:, F - 1]) + 0.2 * (group % 5) + 0.3 * rng.standard_normal(n)
    y = np.digitize(z, np.quantile(z, np.arange(1, K) / K)).astype(np.float32)
    val, rp, col = D.dense_to_csr(X)
    out = []
    for switch in ("1", "0"):
        monkeypatch.setenv("TGBM_SPLIT_HIST", switch)
        s = T.Session(val, rp, col, y, depth=depth, n_trees=2, learning_rate=0.4, objective="multi:softmax", num_class=K, gamma=2.0)
        assert (s.info("split_hist_rows") > 0) == (switch == "1")
        assert s.info("class_walk") == (width if switch == "1" else 0)
        s.boost(2)
        out.append((s.model().tobytes(), s.nid().tobytes(), s.y_pred().tobytes()))
        s.close()
    same = [a == b for a, b in zip(*out)]
    assert all(same), same
