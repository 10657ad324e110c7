"""Scoring calls that go up in slices of rows, several copies at once, and come back through pinned pieces
(thundergbm_amd/csrc/predictor.hip, transfer.hip) against the same rows scored a few at a time."""
import os
import sys

import numpy as np
import pytest
import scipy.sparse as sp

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))

pytestmark = pytest.mark.gpu


def piecewise(m, X, rows, classes=1):
    """(the C call returns class after class)"""
    parts = [np.asarray(m.predict(X[i:i + rows])).reshape(classes, -1) for i in range(0, X.shape[0], rows)]
    return np.concatenate(parts, axis=1).reshape(-1)


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("n,objective", [(262_145, "reg:linear"), (650_003, "reg:linear"), (300_001, "multi:softprob")])
def test_dense_rows_in_slices(n, objective, dtype):
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 28)).astype(dtype)
    X[rng.random(n) < 0.1] = 0
    y = X[:4000, 0] + np.abs(X[:4000, 1])
    classes = 3 if objective.startswith("multi") else 1
    if objective == "reg:linear":
        m = T.TGBMRegressor(depth=5, n_trees=6, learning_rate=0.4, verbose=0).fit(X[:4000], y)
    else:
        m = T.TGBMClassifier(depth=5, n_trees=6, learning_rate=0.4, verbose=0, objective=objective).fit(X[:4000], np.digitize(y, [0.5, 1]))
    assert np.asarray(m.predict(X)).reshape(-1).tobytes() == piecewise(m, X, 40_000, classes).tobytes()


@pytest.mark.parametrize("n,F,far", [(600_001, 250, None), (600_001, 3_000, None), (500_000, 3_000, 70_000), (400_000, 90, 200)])
def test_sparse_rows_in_slices(n, F, far):
    """Column indices that cross as bytes, as words, and with one in the middle that fits neither (`far`); 100 000 rows with
    next to nothing in them."""
    import thundergbm_amd as T
    rng = np.random.default_rng(n + F)
    counts = rng.integers(0, 30, n)
    counts[100_000:250_000] = 0
    counts[100_000:250_000:1000] = 1
    rp = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    col = np.sort(rng.integers(0, F, (n, 30)), axis=1)
    keep = np.arange(30)[None, :] < counts[:, None]
    col = col[keep].astype(np.int32)
    col[rp[100_000:250_000:1000]] = F - 1  # (every part has a column past the narrow ones, see below)
    val = rng.standard_normal(col.size).astype(np.float32)
    if far is not None:
        last = rp[n // 2 + 60_000] - 1  # (the last stored value of some row)
        col[last] = far
    width = (far or F - 1) + 1
    X = sp.csr_matrix((val, col, rp), shape=(n, width))
    y = np.asarray(X[:5000].sum(1)).ravel()
    m = T.TGBMRegressor(depth=6, n_trees=8, learning_rate=0.4, verbose=0).fit(X[:5000], y)
    whole = np.asarray(m.predict(X)).reshape(-1)
    # (the type of the sums hangs on the data's largest column, as in the reference: double up to 96 columns)
    part = piecewise(m, X, 30_000)
    assert np.allclose(whole, part, rtol=2e-6, atol=2e-6)
    if F > 96:
        assert whole.tobytes() == part.tobytes()


# Several classes: the ends of k_score_group's range (65 536 rows through the classes), of the launches that share the classes out
# (2048 workgroups of 256 rows) and of one slice (1024 workgroups through the classes), against k_score_group, which gives the same bits.
@pytest.mark.parametrize("classes,n", [
    (3, 21_845), (3, 21_846), (5, 13_108), (7, 9_363), (3, 174_762), (3, 174_763), (5, 209_716), (8, 66_000), (3, 262_144), (3, 524_289)])
def test_classes_are_shared_out(classes, n, monkeypatch):
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    X = rng.standard_normal((n, 3)).astype(np.float32)
    X[rng.random((n, 3)) < 0.1] = 0
    y = rng.integers(0, classes, 2000)
    m = T.TGBMClassifier(depth=4, n_trees=3, verbose=0, objective="multi:softprob").fit(X[:2000], y)
    assert m.num_class == classes
    got = np.asarray(m.predict(X))
    monkeypatch.setenv("TGBM_PREDICT_GROUP", "1")
    assert got.tobytes() == np.asarray(m.predict(X)).tobytes()
