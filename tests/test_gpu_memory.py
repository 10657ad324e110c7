"""Device memory that is kept between calls (thundergbm_amd/csrc/device_memory.hip)."""
import os
import sys
import threading

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import datasets as D  # noqa: E402

pytestmark = pytest.mark.gpu


def test_calls_share_and_return_kept_memory():
    """Sessions of two threads at once, of different sizes, then again after everything kept went back to the driver:
    the same models each time."""
    import thundergbm_amd as T
    L = T.load()
    D.warm_up(T)
    data = []
    for n, F in ((3000, 5), (777, 40)):
        X, y = D.config1(n, F, seed=n)
        data.append(D.dense_to_csr(X) + (y,))

    def train(i):
        val, rp, col, y = data[i]
        s = T.Session(val, rp, col, y, depth=5, n_trees=6, learning_rate=0.5)
        s.boost(6)
        m = s.model().tobytes()
        s.close()
        return m

    alone = [train(0), train(1)]
    got = {}

    def loop(i):
        got[i] = [train(i) for _ in range(5)]

    threads = [threading.Thread(target=loop, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    L.tgbm_release_memory()
    for i in (0, 1):
        assert all(m == alone[i] for m in got[i])
        assert train(i) == alone[i]


def test_an_idle_process_holds_little_and_can_give_it_back():
    import ctypes as C
    import thundergbm_amd as T
    D.warm_up(T)
    hip = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))

    def memory():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value, total.value

    X, y = D.config1(400_000, 20, seed=1)
    val, rp, col = D.dense_to_csr(X)

    def train():
        s = T.Session(val, rp, col, y, depth=6, n_trees=2)
        s.boost(2)
        s.close()

    train()
    T.release_memory()
    free, total = memory()
    train()
    kept = free - memory()[0]
    assert 0 < kept <= total // 32
    T.release_memory()
    assert free - memory()[0] < kept // 4


@pytest.mark.parametrize("filled,more", [(0.9, 0.5), (0.99, 1.5)])
def test_a_dense_matrix_goes_once_its_values_are_grouped(filled, more):
    """Beside what the same data takes as CSR a dense call needs its matrix: with empty cells past a 32nd (of up to 256 columns) until the
    values are grouped, when its block becomes one of the sort's, else until the cells are sorted."""
    import ctypes as C
    import scipy.sparse as sp
    import thundergbm_amd as T
    D.warm_up(T)
    hip = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))

    def free():
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    rng = np.random.default_rng(3)
    X = rng.standard_normal((400_000, 40)).astype(np.float32)
    X[rng.random(X.shape) >= filled] = 0
    y = X[:, 0] + X[:, 1] ** 2

    def kept(data):  # (the blocks of a call are kept until they are given back: the most that it held at a time, by size)
        T.release_memory()
        before = free()
        T.TGBMRegressor(depth=3, n_trees=1).fit(data, y)
        return before - free()

    as_csr = sp.csr_matrix(X)
    kept(as_csr)
    extra = kept(X) - kept(as_csr)
    assert extra < more * X.nbytes, extra


@pytest.mark.parametrize("spread", ["1", "0"])
def test_sparse_sessions_hold_a_value_once(spread, monkeypatch):
    """A session of the sparse level pass: its values have places of their own, and the copy that those are made of goes. A value of a
    frequent feature takes 4 bytes as a bin, 18 in its place (14 looked up) and 1/0.6 in a byte column here, the copy 8."""
    import ctypes as C
    import thundergbm_amd as T
    D.warm_up(T)
    hip = C.CDLL(next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64" in line))

    def free():
        T.release_memory()
        f, t = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(f), C.byref(t)) == 0
        return f.value

    monkeypatch.setenv("TGBM_LAYOUT", "sparse")
    monkeypatch.setenv("TGBM_SPARSE_SPREAD", spread)
    rng = np.random.default_rng(1)
    n, F = 300_000, 40
    X = np.exp(rng.standard_normal((n, F))).astype(np.float32)
    X[rng.random(X.shape) >= 0.6] = 0
    val, rp, col = D.dense_to_csr(X)
    before = free()
    s = T.Session(val, rp, col, X[:, 0] + X[:, 1], depth=3, n_trees=2, max_num_bin=15)
    assert s.info("sparse_pass") == 1 and s.info("sparse_spread_blocks") == (10 if spread == "1" else 0)
    held = (before - free()) / len(val)
    s.boost(2)
    s.close()
    rows = 40 * n / len(val)  # (what a row takes itself: labels, predictions, pairs, nodes, words)
    assert held < 4 + (18 if spread == "1" else 14) + 1 / 0.6 + rows + 4, held
