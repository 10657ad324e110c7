"""Dense arrays given to the estimators: the device makes the CSR form of them (prep_kernels.hip, transfer.hip); the CSR
matrix that scipy makes of the same array is the reference."""
import os
import sys

import numpy as np
import pytest
import scipy.sparse as sp

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu


def matrix(n, F, dtype, filled, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, F)).astype(dtype) if np.dtype(dtype).kind == "f" else rng.integers(-3, 4, (n, F)).astype(dtype)
    X[rng.random((n, F)) >= filled] = 0
    if filled < 1 and np.dtype(dtype).kind == "f":
        X[rng.random((n, F)) < 0.05] = -0.0
        X[:, F // 2] = np.where(rng.random(n) < 0.3, 1e-60, X[:, F // 2])  # (a stored zero when it becomes a float32)
        X[:, -1] = 0  # (no feature at all)
    y = X[:, 0].astype(np.float64) - (X[:, min(1, F - 1)] > 0) + 0.1 * rng.standard_normal(n)
    return X, y.astype(np.float32)


def trees_of(m):
    return [np.concatenate([np.asarray(t[k]).reshape(-1) for t in m.get_trees()]).tobytes()
            for k in ("children_left", "children_default", "feature", "threshold", "value", "node_sample_weight")]


@pytest.mark.parametrize("n,F,dtype,filled", [
    (1, 3, "float32", 1.0), (17, 15, "float32", 1.0), (300, 16, "float64", 0.7), (4097, 17, "float32", 0.5),
    (5000, 33, "float64", 1.0), (2500, 40, "int64", 0.8), (1200, 130, "float32", 0.9),
    (190_000, 17, "float32", 0.99), (110_000, 31, "float64", 0.9)])  # (the last two go through the pinned pieces)
def test_dense_fit_equals_csr_fit(n, F, dtype, filled):
    import thundergbm_amd as T
    X, y = matrix(n, F, dtype, filled, seed=n + F)
    kw = dict(depth=5, n_trees=4, learning_rate=0.5, verbose=0)
    a = T.TGBMRegressor(**kw).fit(X, y)
    b = T.TGBMRegressor(**kw).fit(sp.csr_matrix(X), y)
    assert trees_of(a) == trees_of(b)
    assert a.group_label == b.group_label and a.num_class == b.num_class


def test_dense_fit_of_classes_and_groups_equals_csr_fit():
    import thundergbm_amd as T
    X, y = matrix(6000, 20, "float32", 0.9, seed=3)
    yc = np.digitize(y, [-1, 0, 1]).astype(np.float32) * 2
    for objective, labels, groups in (("multi:softmax", yc, None), ("binary:logistic", (y > 0).astype(np.float32), None),
                                      ("rank:pairwise", yc, np.full(60, 100, np.int32))):
        kw = dict(depth=4, n_trees=3, objective=objective, verbose=0)
        m = [T.TGBMClassifier(**kw) for _ in range(2)]
        import ctypes
        for mm, XX in zip(m, (X, sp.csr_matrix(X))):
            ctypes.CDLL(None).srand(5)
            mm.fit(XX, labels, groups=groups)
        assert trees_of(m[0]) == trees_of(m[1]), objective
        assert m[0].group_label == m[1].group_label and m[0].num_class == m[1].num_class


@pytest.mark.parametrize("n,F,used,classes,depth,n_iter", [
    (1, 3, 3, 1, 1, 1), (1, 40, 40, 1, 6, 300), (257, 20, 20, 4, 4, 70), (1025, 50, 50, 1, 8, 11), (3000, 97, 97, 1, 5, 9),
    (1500, 700, 300, 3, 6, 20)])
def test_scoring_kernels_agree(n, F, used, classes, depth, n_iter):
    """Dense rows and their CSR form, a thread per row and a group of lanes per row, and the walk of the 48-byte nodes:
    the same bits, below and above the 96 features where the sums change from double to float."""
    import ctypes as C
    import datasets as D
    import thundergbm_amd as T
    L = T.load()
    rng = np.random.default_rng(n + F)
    X = rng.standard_normal((4000, F)).astype(np.float32)
    X[:, used:] *= 1e-3
    X[rng.random(X.shape) < 0.1] = 0
    z = X[:, :used] @ rng.standard_normal(used)
    y = np.digitize(z, np.quantile(z, np.linspace(0, 1, classes + 1)[1:-1])).astype(np.float32) if classes > 1 else z
    m = (T.TGBMClassifier if classes > 1 else T.TGBMRegressor)(
        depth=depth, n_trees=n_iter, learning_rate=0.3, verbose=0, objective="multi:softprob" if classes > 1 else "reg:linear")
    m.fit(X, y)
    Xt = rng.standard_normal((n, F)).astype(np.float64)
    Xt[rng.random(Xt.shape) < 0.2] = 0
    Xt.reshape(-1)[::37] = np.inf
    Xt.reshape(-1)[1::41] = np.nan
    Xt.reshape(-1)[2::43] = -1e-70
    csr = sp.csr_matrix(Xt)
    want, got = None, {}
    val, rp, col = csr.data.astype(np.float32), csr.indptr.astype(np.int32), csr.indices.astype(np.int32)
    p = lambda a: a.ctypes.data_as(C.c_void_p)
    try:
        for name, env in (("nodes", {"TGBM_PREDICT_TPS": "0"}), ("rows", {"TGBM_PREDICT_GROUP": "0"}),
                          ("group", {"TGBM_PREDICT_GROUP": "1"}), ("default", {})):
            os.environ.update(env)
            raw = np.zeros(n * m.tree_per_iter, np.float32)
            L.tgbm_predict_raw(n, p(val), p(rp), p(col), m.model, n_iter, m.tree_per_iter, 0.3, 0.25, p(raw))
            got[name] = (raw, m.predict(Xt).copy(), m.predict(csr).copy(), m.predict(Xt.astype(np.float32)).copy())
            for k in env:
                os.environ.pop(k)
    finally:
        for k in ("TGBM_PREDICT_TPS", "TGBM_PREDICT_GROUP"):
            os.environ.pop(k, None)
    want = got["nodes"]
    for name, outs in got.items():
        for a, b in zip(outs, want):
            assert np.array_equal(a, b, equal_nan=True), name
        assert np.array_equal(outs[1], outs[2], equal_nan=True), name
