"""Deep trees in the dense layout: levels of so many nodes that one launch plans their work items (k_plan_level)."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
import datasets as D  # noqa: E402
import parity as P  # noqa: E402
import test_gpu_edge as E  # noqa: E402
from test_gpu_edge import T, _default_layout  # noqa: E402,F401  (fixtures)

pytestmark = pytest.mark.gpu

DEEP = dict(gamma=0.0, min_child_weight=0.05)
CASES = {
    # name: (rows, features, longest row, objective, targets, options, layout)
    "depth11": (4000, 5, 5, "reg:linear", "reg", dict(DEEP, depth=11, max_num_bin=255), "dense"),
    "depth12": (9000, 7, 6, "binary:logistic", "bin", dict(DEEP, depth=12, max_num_bin=64), "dense"),
    "depth13": (20000, 6, 6, "reg:linear", "reg", dict(DEEP, depth=13, max_num_bin=255), "dense"),
    "depth14": (12000, 4, 4, "reg:logistic", "prob", dict(DEEP, depth=14, max_num_bin=33), "dense"),
    "few_rows": (40, 3, 3, "reg:linear", "reg", dict(DEEP, depth=14, max_num_bin=16), "dense"),
    "classes": (5000, 6, 6, "multi:softmax", "multi", dict(DEEP, depth=12, max_num_bin=32), "dense"),
    "bins_of_16_bits": (6000, 5, 5, "reg:linear", "reg", dict(DEEP, depth=12, max_num_bin=64), "dense-16"),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_deep_trees_match_the_oracle(T, name):  # noqa: F811
    margins = P.Margins("deep/" + name)
    E.run_case(T, CASES[name], 77, margins)
    margins.report()


@pytest.mark.parametrize("cap", ["4", "256", "512", "1024"])
def test_deep_levels_in_batches_of_nodes(T, cap):  # noqa: F811
    """A capped arena builds single nodes below the levels that fit: planned from fewer levels on."""
    rng = np.random.default_rng(3)
    X = rng.standard_normal((15000, 5)).astype(np.float32)
    y = (X[:, 0] + np.abs(X[:, 1]) + 0.3 * rng.standard_normal(15000)).astype(np.float32)
    val, rp, col = D.dense_to_csr(X)
    runs = []
    os.environ["TGBM_LAYOUT"] = "dense"
    for arena in (None, cap):
        if arena is not None:
            os.environ["TGBM_HIST_ARENA_NODES"] = arena
        s = T.Session(val, rp, col, y, depth=12, n_trees=2, learning_rate=0.5, max_num_bin=48, **DEEP)
        s.boost(2)
        runs.append((s.model().tobytes(), s.y_pred().tobytes(), s.nid().tobytes()))
        s.close()
    assert runs[0] == runs[1]
