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
