"""Host arrays on their way to the device: labels grouped into classes, column indices narrowed for the transfer."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import datasets as D  # noqa: E402

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("values", [[0, 1, 2], [-3, 5, 70], [1, 100_000, 2_000_000], [0.5, 1, 2, 7]])
@pytest.mark.parametrize("n", [999, 300_001])
def test_labels_become_classes(values, n):
    import thundergbm_amd as T
    rng = np.random.default_rng(n)
    X = rng.random((n, 2), dtype=np.float32) + 0.1
    y = rng.choice(np.asarray(values, np.float32), n)
    y[: len(values)] = values
    val, rp, col = D.dense_to_csr(X)
    s = T.Session(val, rp, col, y, depth=1, n_trees=1, objective="multi:softmax", max_num_bin=16)
    labels = np.unique(np.trunc(np.asarray(values, np.float32)))
    assert np.array_equal(s.labels(), labels)
    want = np.zeros(n, np.float32)
    for k, v in enumerate(labels):
        want[y == v] = k
    assert np.array_equal(s.y(), want)
    s.close()


@pytest.mark.parametrize("last", [200, 255, 256, 65_535])
def test_narrowed_column_indices_arrive_whole(last):
    """Enough indices for the pinned pieces; the largest index sits in the middle, where a look at the ends misses it."""
    import thundergbm_amd as T
    n, k = 1_300_003, 10
    rng = np.random.default_rng(last)
    col = np.sort(rng.integers(0, 20, (n, k)) * 10 + np.arange(k), axis=1).astype(np.int32)
    col[n // 2, -1] = last
    rp = (np.arange(n + 1) * k).astype(np.int32)
    val = rng.random(n * k, dtype=np.float32) + 0.5
    y = rng.random(n, dtype=np.float32)
    s = T.Session(val, rp, col.reshape(-1), y, depth=2, n_trees=1, max_num_bin=8)
    assert s.F == last + 1
    _, crp, _ = s.cuts()
    stored = np.diff(crp) > 0
    assert np.array_equal(np.flatnonzero(stored), np.unique(col))
    s.close()
