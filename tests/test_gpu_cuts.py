"""Cut points sorted by feature (thundergbm_amd/csrc/cut_kernels.hip) and bins searched in LDS against a plain selection, at the
edges of their tiles."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _expected(X, stored, max_bin):
    cuts, ptr = [], [0]
    for f in range(X.shape[1]):
        u = np.unique(X[stored[:, f], f] + np.float32(0))
        step = len(u) // max_bin
        c = u if step == 0 else u[::step][:max_bin]
        cuts.append(c)
        ptr.append(ptr[-1] + len(c))
    return np.concatenate(cuts), np.array(ptr)


@pytest.mark.parametrize("n,F,filled,max_bin", [
    (1, 3, 1.0, 255), (4096, 2, 1.0, 255), (4097, 256, 1.0, 63), (8191, 255, 0.5, 255), (5000, 257, 0.7, 31), (70000, 5, 0.9, 255),
    (12289, 17, 1.0, 1024), (3000, 300, 1.0, 255)])
@pytest.mark.parametrize("dense", [False, True])
def test_cut_points(n, F, filled, max_bin, dense):
    import thundergbm_amd as T
    rng = np.random.default_rng(n + F)
    X = rng.standard_normal((n, F)).astype(np.float32)
    X[:, ::3] = np.round(X[:, ::3] * 4) / 4 + np.float32(0.125)  # few distinct values
    if filled < 1:
        X[rng.random((n, F)) >= filled] = 0
        X[:, F // 2] = 0  # a column without values
        X[0, F - 1] = 1
    y = X[:, 0] + 1
    want, ptr = _expected(X, X != 0, max_bin)
    if dense:
        m = T.TGBMRegressor(depth=3, n_trees=1, max_num_bin=max_bin, verbose=0).fit(X, y)
        v = m.get_trees()[0]
        walk = [0]  # every split is at a cut point, or below all of them
        for i in walk:
            if v["children_left"][i] >= 0:
                c = want[ptr[v["feature"][i]]:ptr[v["feature"][i] + 1]]
                assert v["threshold"][i] in c or v["threshold"][i] < c[0]
                walk += [v["children_left"][i], v["children_right"][i]]
        return
    rp = np.zeros(n + 1, np.int32)
    np.cumsum((X != 0).sum(1), out=rp[1:])
    r, c = np.nonzero(X)
    s = T.Session(X[r, c], rp, c.astype(np.int32), y, depth=3, n_trees=1, max_num_bin=max_bin)
    cv, crp, cf = s.cuts()
    assert np.array_equal(cv, want) and np.array_equal(crp, ptr)
    assert np.array_equal(cf, np.repeat(np.arange(F), np.diff(ptr)))
    ids, _ = s.global_bin_ids(rp, c.astype(np.int32))
    per = [np.clip(np.searchsorted(want[ptr[f]:ptr[f + 1]], X[:, f], side="right"), 0, max(ptr[f + 1] - ptr[f] - 1, 0)) + ptr[f] for f in range(F)]
    assert np.array_equal(ids, np.stack(per, 1)[r, c])
    s.close()


# Segments that one workgroup sorts: 2, 4, 8 and 16 keys a thread, and the first ones that are too long for it; features that
# share a value or none.
@pytest.mark.parametrize("n,F,filled,max_bin", [
    (2048, 3, 1.0, 255), (2049, 9, 1.0, 255), (2500, 119, 0.1, 255), (8192, 2, 1.0, 1024), (8193, 33, 0.99, 255), (16384, 5, 1.0, 63),
    (16385, 5, 1.0, 63), (16500, 300, 0.98, 255), (64, 256, 0.4, 2), (65, 1, 1.0, 255)])
@pytest.mark.parametrize("dense", [False, True])
def test_cut_points_of_short_segments(n, F, filled, max_bin, dense):
    test_cut_points(n, F, filled, max_bin, dense)


# Dense cells of which some hold no value, sorted along with the values or not (at most a quarter of them on wide data, a 32nd else; 1024
# rows), and bins by runs of features (16 384 cut points a run), against the same values as CSR.
@pytest.mark.parametrize("n,F,filled,max_bin", [
    (1023, 257, 0.99, 31), (1024, 257, 0.99, 31), (4096, 300, 0.76, 63), (4097, 300, 0.74, 63), (5000, 40, 0.98, 255), (5000, 40, 0.95, 255),
    (3000, 130, 0.97, 255), (4100, 260, 0.9, 300), (2049, 64, 1.0, 255)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_cells_without_values(n, F, filled, max_bin, dtype):
    import scipy.sparse as sp
    import thundergbm_amd as T
    rng = np.random.default_rng(n + F)
    X = rng.standard_normal((n, F)).astype(dtype)
    X[:, ::3] = np.round(X[:, ::3] * 4) / 4
    X[rng.random((n, F)) >= filled] = 0
    X[:, F // 2] = 0
    X[5, 3], X[6, 3], X[7, 4] = np.inf, -np.inf, -0.0
    if dtype == np.float64:
        X[8, 5] = 1e-60  # (stored, and zero as a float)
    y = (X[:, 0] + np.abs(X[:, 1]) - X[:, F - 1]).astype(np.float32)
    runs = []
    for data in (X, sp.csr_matrix(X)):
        m = T.TGBMRegressor(depth=4, n_trees=3, max_num_bin=max_bin, verbose=0).fit(data, y)
        runs.append([{k: v.tobytes() for k, v in t.items()} for t in m.get_trees()] + [m.predict(data).tobytes()])
    assert runs[0] == runs[1]


# Bins by runs of features (two here) and by each value's own search: rows with fewer and with more than four values a run.
@pytest.mark.parametrize("filled", [0.035, 0.045])
def test_bins_of_rows_with_few_values(filled, monkeypatch):
    monkeypatch.setenv("TGBM_LAYOUT", "dense")
    test_cut_points(6000, 200, filled, 200, False)
