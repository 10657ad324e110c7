"""What this library is measured on: whole calls of its public entry points, from the arrays that a program has in
host memory (the library takes host data) to the model or the scores that it gets back.

A training pass is `TGBMClassifier` / `TGBMRegressor.fit` on a dense array and `get_trees`, or, where the data is CSR,
one `Session`: upload, cut points, bins, all boosting rounds, the model. A scoring pass is `predict` on a dense array
with a fitted estimator, or `tgbm_predict_raw` on CSR arrays with a model handle. Every pass trains from scratch or
scores afresh; nothing is carried from one to the next.

Rows, columns, values and labels follow the repository's benchmark configurations and its quick-start data set.
"""
import ctypes
import math

import numpy as np
import torch

import thundergbm_amd as T

MODEL_ROWS = 20_000  # rows that the models of the scoring cases are trained on
FIELDS = ("lch", "rch", "gain", "base_weight", "split_fid", "split_value", "default_right", "is_leaf", "is_valid",
          "is_pruned", "sum_g", "sum_h")


def case(name, call, data, rows, features, objective, depth, trees, **more):
    """call: fit / score. data: dense (a float array), csr (the same values as CSR arrays), onehot (CSR: quantised columns
    and one-hot groups of 4 and 40), zipf (CSR: `per_row` draws of a power-law distributed column per row)."""
    c = dict(name=name, call=call, data=data, rows=rows, features=features, objective=objective, depth=depth, trees=trees,
             classes=1, bins=255, rate=0.1, filled=1.0, dtype="float32", per_row=0, group=0, bagging=False, columns=1.0)
    c.update(more)
    return c


def listed():
    return [
        # the quick-start call: a small sparse data set, 40 trees of depth 6 at learning rate 1
        case("fit_quickstart", "fit", "zipf", 1605, 119, "reg:linear", 6, 40, rate=1.0, per_row=14),
        # a first experiment on a small table (benchmark configuration 1)
        case("fit_small_table", "fit", "dense", 10_000, 8, "reg:linear", 6, 40),
        # an ordinary table of numbers as a numpy array through the scikit-learn interface
        case("fit_table", "fit", "dense", 500_000, 28, "binary:logistic", 8, 100),
        # the headline workload (benchmark configuration 2) with all its trees
        case("fit_large", "fit", "csr", 10_000_000, 28, "binary:logistic", 8, 100),
        # wide data with heavy-tailed columns (the shape of benchmark configuration 3, as a double-precision array)
        case("fit_wide", "fit", "dense", 50_021, 700, "reg:linear", 6, 50, dtype="float64"),
        # click data: 100 000 columns, ~35 stored values per row, 63 bins (benchmark configuration 4)
        case("fit_clicks", "fit", "zipf", 1_000_000, 100_000, "binary:logistic", 8, 40, bins=63, per_row=40),
        # numbers and one-hot groups, eight unbalanced classes (benchmark configuration 5)
        case("fit_classes", "fit", "onehot", 500_000, 54, "multi:softmax", 8, 20, classes=8),
        # learning to rank: query groups of about 120 rows
        case("fit_ranking", "fit", "dense", 200_003, 136, "rank:ndcg", 8, 40, group=120),
        # a table with a third of its values missing, resampled rows and columns, many bins
        case("fit_resampled", "fit", "csr", 77_777, 37, "reg:linear", 7, 50, bins=1024, filled=0.66, bagging=True, columns=0.2),
        # one request of a service
        case("score_one_row", "score", "dense", 1, 28, "reg:linear", 6, 100),
        # class probabilities of a table
        case("score_table", "score", "dense", 200_000, 28, "multi:softprob", 8, 40, classes=5),
        # scoring of sparse rows with many columns
        case("score_clicks", "score", "zipf", 500_000, 100_000, "reg:linear", 8, 100, bins=63, per_row=40),
    ]


def spread(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    call = rng.choice(("fit", "fit", "fit", "score"))
    data = rng.choice(("dense", "dense", "csr", "onehot", "zipf"))
    depth, trees = rng.randint(4, 8), rng.randint(10, 100)
    more = dict(rate=rng.choice((0.05, 0.1, 0.3, 1.0)), bins=rng.choice((31, 63, 128, 255, 255, 255, 1024 if data in ("dense", "csr") else 255)))
    least = 1 if call == "score" else 1_000
    if data == "zipf":
        rows, features = spread(rng, least, 1_000_000), spread(rng, 100, 100_000)
        more["per_row"] = min(features // 4, rng.randint(10, 40))
        trees = min(trees, 40)
    elif data == "onehot":
        rows, features = spread(rng, least, 500_000), rng.randint(50, 64)
    elif data == "csr":
        features = spread(rng, 4, 200)
        rows = spread(rng, least, min(10_000_000, 280_000_000 // features))
        more["filled"] = rng.choice((1.0, 1.0, 0.9, 0.5))
    else:
        features = spread(rng, 4, 700)
        rows = spread(rng, least, min(600_000, 30_000_000 // features))
        more["dtype"] = rng.choice(("float32", "float32", "float64"))
        more["filled"] = rng.choice((1.0, 1.0, 0.9))
    kinds = ["reg:linear", "binary:logistic", "reg:logistic"]
    if data in ("dense", "onehot") and rows * features <= 28_000_000:
        kinds += ["multi:softmax" if call == "fit" else "multi:softprob"] + (["rank:ndcg", "rank:pairwise"] if call == "fit" else [])
    objective = rng.choice(kinds)
    if call == "score" and objective == "binary:logistic":
        objective = "reg:logistic"
    if objective.startswith("multi:"):
        more["classes"], trees = rng.randint(3, 8), min(trees, 20)
    if objective.startswith("rank:"):
        more["group"], trees = rng.randint(20, 200), min(trees, 40)
    elif call == "fit" and data != "zipf" and rng.random() < 0.2:
        more["bagging"] = True
    if call == "fit" and data != "zipf" and rng.random() < 0.2:
        more["columns"] = 0.3
    c = case("", call, data, rows, features, objective, depth, trees, **more)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------------------- the inputs


def table(c, rows, gen):
    """Numbers as they come: normal columns, one in twenty heavy-tailed, a quarter derived from others; exact zeros are
    values that are not there."""
    F = c["features"]
    X = torch.randn(rows, F, device="cuda", generator=gen)
    for f in range(3, F, 20):
        X[:, f] /= torch.sqrt(-torch.log(torch.rand(rows, device="cuda", generator=gen).clamp_(1e-7, 0.9999999)))
    base = F - F // 4
    for j in range(F - base):
        a, b = X[:, (2 * j) % base], X[:, (2 * j + 1) % base]
        X[:, base + j] = a * b if j % 2 == 0 else (a - b).abs()
    if c["filled"] < 1:
        X *= torch.rand(rows, F, device="cuda", generator=gen) < c["filled"]
    return X


def one_hot(c, rows, gen):
    F = c["features"]
    q = F - 44
    X = torch.zeros(rows, F, device="cuda")
    X[:, :q] = torch.floor(torch.rand(rows, q, device="cuda", generator=gen) * 3000)
    at = torch.arange(rows, device="cuda")
    for first, width in ((q, 4), (q + 4, 40)):
        X[at, first + torch.randint(0, width, (rows,), device="cuda", generator=gen)] = 1
    return X


def to_csr(X):
    mask = X != 0
    ptr = torch.zeros(X.shape[0] + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(mask.sum(1), 0, out=ptr[1:])
    col = torch.arange(X.shape[1], dtype=torch.int32, device="cuda").expand(X.shape)
    if int(ptr[-1]) == X.numel():
        return X.reshape(-1), ptr.int(), col.reshape(-1)
    return X[mask], ptr.int(), col[mask]


def clicks(c, rows, gen):
    """Columns with power-law frequencies (the few most frequent ones in most rows, most of them in a handful), values
    log-normal; a column drawn twice in a row is stored once."""
    F, k = c["features"], c["per_row"]
    u = torch.rand(rows, k, device="cuda", generator=gen).clamp_(min=1e-6)
    raw = torch.floor(u.double().pow(-10.0)) - 1
    other = torch.randint(0, F, (rows, k), device="cuda", generator=gen)
    raw = torch.where(raw >= F, other.double(), raw).long().sort(1).values
    keep = torch.ones_like(raw, dtype=torch.bool)
    keep[:, 1:] = raw[:, 1:] != raw[:, :-1]
    ptr = torch.zeros(rows + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(keep.sum(1), 0, out=ptr[1:])
    col = raw[keep]
    val = torch.exp(torch.randn(col.numel(), device="cuda", generator=gen))
    return val, ptr.int(), col.int()


def signal(c, values, rows, gen):
    """What the labels hang on: ten columns of a table, or some hundreds of the columns of sparse rows."""
    if isinstance(values, tuple):
        val, ptr, col = values
        w = torch.randn(c["features"], device="cuda", generator=gen)
        w *= (torch.rand(c["features"], device="cuda", generator=gen) < 0.05) | (torch.arange(c["features"], device="cuda") < 20)
        row = torch.repeat_interleave(torch.arange(rows, device="cuda"), (ptr[1:] - ptr[:-1]).long())
        z = torch.zeros(rows, device="cuda", dtype=torch.float64)
        z.index_add_(0, row, (w[col.long()] * torch.log1p(val)).double())  # (in double: the labels hang on the seed alone)
        return (z - z.mean()).float()
    X = values / values.abs().amax(0).clamp(min=1) if c["data"] == "onehot" else values
    z = torch.zeros(rows, device="cuda")
    for f in torch.randperm(c["features"], device="cuda", generator=gen)[:10].tolist():
        z += X[:, f].clamp(-5, 5) * float(torch.randn(1, device="cuda", generator=gen))
    return z + 0.3 * X[:, 0].clamp(-5, 5) * X[:, 1].clamp(-5, 5)


def labels(c, z, gen):
    rows, kind = len(z), c["objective"]
    noise = torch.rand(rows, device="cuda", generator=gen)
    if kind.startswith("multi:"):
        k = c["classes"]
        at = torch.randn(k, device="cuda", generator=gen)
        bias = torch.log(1 / torch.arange(1.0, k + 1, device="cuda"))
        y = (z[:, None] * at + bias - torch.log(-torch.log(torch.rand(rows, k, device="cuda", generator=gen).clamp_(1e-7, 0.9999999)))).argmax(1)
        y[: min(k, rows)] = torch.arange(min(k, rows), device="cuda")
    elif kind.startswith("rank:"):
        y = torch.bucketize(z + torch.randn(rows, device="cuda", generator=gen), torch.tensor([0.0, 1.5, 3.0, 4.5], device="cuda"))
    elif kind.endswith("logistic"):
        y = noise < torch.sigmoid(z)
        y[:2] = torch.tensor([False, True], device="cuda")[:rows]
    else:
        y = z + 0.5 * torch.randn(rows, device="cuda", generator=gen)
    return y.float().cpu().numpy()


def make(c, rows, gen):
    """(the matrix as a program holds it in host memory, labels)."""
    if c["data"] == "zipf":
        values = clicks(c, rows, gen)
    else:
        values = one_hot(c, rows, gen) if c["data"] == "onehot" else table(c, rows, gen)
    y = labels(c, signal(c, values, rows, gen), gen)
    if c["data"] == "dense":
        return values.cpu().numpy().astype(c["dtype"], copy=False), y
    return tuple(t.cpu().numpy() for t in (values if c["data"] == "zipf" else to_csr(values))), y


def groups(c, rows):
    if not c["group"]:
        return None
    rng = np.random.default_rng(rows)
    sizes = rng.integers(c["group"] // 2, c["group"] * 3 // 2 + 1, size=3 * rows // c["group"] + 2)
    ends = np.minimum(np.cumsum(sizes), rows)
    sizes = np.diff(np.concatenate([[0], ends]))
    return sizes[sizes > 0].astype(np.int32)


def estimator(c):
    kind = T.TGBMRegressor if c["objective"].startswith("reg:") else T.TGBMClassifier
    return kind(depth=c["depth"], n_trees=c["trees"], max_num_bin=c["bins"], learning_rate=c["rate"], objective=c["objective"],
                num_class=c["classes"], bagging=int(c["bagging"]), column_sampling_rate=c["columns"], verbose=0)


def session(c, X, y):
    val, ptr, col = X
    s = T.Session(val, ptr, col, y, depth=c["depth"], n_trees=c["trees"], max_num_bin=c["bins"], learning_rate=c["rate"],
                  objective=c["objective"], num_class=c["classes"], groups=groups(c, len(y)))
    if c["bagging"]:
        s.set_option("bagging", 1)
    if c["columns"] < 1:
        s.set_option("column_sampling_rate", c["columns"])
    return s


class Handle:
    """A model handle of the C interface, given back with the state that owns it."""

    def __init__(self, s):
        self.lib, self.h = T.load(), ctypes.c_void_p(s.export_model())

    def __del__(self):
        self.lib.model_free(ctypes.byref(self.h))


def prepare(case, seed):
    c = case
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": c, "seed": seed & 0x7FFFFFFF}
    if c["call"] == "score":
        X, y = make(c, MODEL_ROWS, gen)
        if c["data"] == "dense":
            state["model"] = estimator(c).fit(X, y)
        else:
            s = session(c, X, y)
            s.boost(c["trees"])
            state.update(model=Handle(s), per_round=s.tree_per_rounds, base=s.base_score)
            s.close()
    state["X"], state["y"] = make(c, c["rows"], gen)
    state["groups"] = groups(c, c["rows"])
    return state


# ---------------------------------------------------------------------------------------------------------- one pass


def run(state):
    c, X, y = state["case"], state["X"], state["y"]
    if c["call"] == "score":
        if c["data"] == "dense":
            return state["model"].predict(X)
        val, ptr, col = X
        out = np.zeros(c["rows"] * state["per_round"], np.float32)
        p = [a.ctypes.data_as(ctypes.c_void_p) for a in (val, ptr, col, out)]
        T.load().tgbm_predict_raw(c["rows"], *p[:3], state["model"].h, c["trees"], state["per_round"], c["rate"], state["base"], p[3])
        return out
    if c["bagging"] or c["columns"] < 1 or c["group"]:
        ctypes.CDLL(None).srand(state["seed"])  # these draw from the C library's generator: a program that wants its model again seeds it
    if c["data"] == "dense":
        trees = estimator(c).fit(X, y, groups=state["groups"]).get_trees()
        return {k: np.concatenate([t[k].reshape(-1) for t in trees]) for k in trees[0]}
    s = session(c, X, y)
    s.boost(c["trees"])
    model = s.model()
    out = {k: np.ascontiguousarray(model[k]) for k in FIELDS}
    out["metric"] = s.metric_log()
    s.close()
    return out


def work(case):
    """Every input value read and every result written once; below that, what boosting trees by histograms visits: the rows
    of the root and of the smaller child of every pair - at most half of the rows a level - with a byte (above 255 bins
    two) per stored value, the gradient pair, and two additions per value; scoring: one node per row, tree and level."""
    c = case
    rows, per_round = c["rows"], max(1, c["classes"] if c["classes"] > 2 else 1)
    if c["data"] == "zipf":
        stored = min(c["per_row"], c["features"]) * 0.87
    elif c["data"] == "onehot":
        stored = c["features"] - 42
    else:
        stored = c["features"] * c["filled"]
    if c["data"] == "dense":
        given = rows * c["features"] * (8 if c["dtype"] == "float64" else 4)
    else:
        given = rows * (stored * 8 + 4)
    trees = c["trees"] * per_round
    model = trees * ((2 << c["depth"]) - 1) * 28
    if c["call"] == "score":
        return {"bytes": given + model + rows * per_round * 4, "flops": rows * trees * (c["depth"] + 1)}
    visits = rows * (1 + (c["depth"] - 1) / 2) * trees
    width = 2 if c["bins"] > 255 else 1
    return {"bytes": given + rows * 4 + model + visits * (stored * width + 8) + rows * trees * 16, "flops": visits * stored * 2}


def tolerance(case):
    """32-bit floats from exact or double-precision sums; a split decided by a tie may fall the other way."""
    return {"rel": 1e-5, "differ": 1e-3}
