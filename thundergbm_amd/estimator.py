"""scikit-learn style estimators over the C ABI, with the constructor arguments, method names and
data handling of the reference wrapper (python/thundergbm/thundergbm.py): dense inputs lose their
exact zeros on the way to CSR (zeros are missing values), values go in as float32 with ascending
column indices, classifier predictions come back as the original labels."""
import ctypes as C

import numpy as np
import scipy.sparse as sp
from sklearn.base import BaseEstimator, ClassifierMixin, RegressorMixin

from . import _lib

_PARAMS = ("depth", "n_trees", "n_gpus", "min_child_weight", "lambda_tgbm", "gamma", "max_num_bin", "verbose",
           "column_sampling_rate", "bagging", "n_parallel_trees", "learning_rate", "objective", "num_class",
           "tree_method")


def _csr(X):
    """CSR view of X with float32 values and ascending column indices; the caller's matrix is only copied
    when it has to be changed."""
    if not sp.issparse(X):
        X = sp.csr_matrix(np.asarray(X))
    elif X.format != "csr":
        X = X.tocsr()
    if X.data.dtype != np.float32 or not X.data.flags.c_contiguous:
        X = sp.csr_matrix((np.ascontiguousarray(X.data, dtype=np.float32), X.indices, X.indptr), shape=X.shape)
    if not X.has_sorted_indices:
        X = X.copy()
        X.sort_indices()
    return X


def _dense(X):
    """X as a C-contiguous float32 or float64 matrix for the entry points that take dense data as it is, or None where
    the conversion to CSR has to decide (sparse input, other shapes and types). Types that float32 holds as well as the
    CSR path's own cast go in as float32."""
    if sp.issparse(X):
        return None
    X = np.asarray(X)
    if X.ndim != 2 or X.size == 0 or X.size >= 1 << 32:
        return None
    if X.dtype.kind in "iub" or X.dtype == np.float16:
        X = X.astype(np.float32)
    if X.dtype != np.float32 and X.dtype != np.float64:
        return None
    return np.ascontiguousarray(X)


def _ptr(a):
    return C.c_void_p(a.ctypes.data)


def _stored_label_count(model_path):
    """Number of labels a model file stores (read from its header, nothing else is parsed)."""
    import struct
    with open(model_path, "rb") as f:
        (olen,) = struct.unpack("<i", f.read(4))
        if olen < 0 or olen >= 4096:
            raise ValueError("model file %s: bad objective length" % model_path)
        f.seek(olen + 16, 1)
        raw = f.read(4)
        if len(raw) != 4:
            raise ValueError("model file %s is truncated" % model_path)
        (n_label,) = struct.unpack("<i", raw)
    if n_label < 0:
        raise ValueError("model file %s: bad label count" % model_path)
    return n_label


class TGBMModel(BaseEstimator):
    def __init__(self, depth=6, n_trees=40, n_gpus=1, min_child_weight=1.0, lambda_tgbm=1.0, gamma=1.0,
                 max_num_bin=255, verbose=1, column_sampling_rate=1.0, bagging=0, n_parallel_trees=1,
                 learning_rate=1.0, objective="reg:linear", num_class=1, tree_method="auto"):
        for name in _PARAMS:
            setattr(self, name, locals()[name])
        self.model = None
        self.tree_per_iter = -1
        self.group_label = None

    def __del__(self):
        self._release()

    def _release(self):
        if getattr(self, "model", None) is not None:
            _lib.load().model_free(C.byref(self.model))
            self.model = None

    def fit(self, X, y, groups=None):
        lib = _lib.load()
        self._release()
        dense = _dense(X)
        X = _csr(X) if dense is None else dense
        y = np.ascontiguousarray(y, dtype=np.float32)
        if X.shape[0] != len(y):
            raise ValueError("X and y have different numbers of rows")
        if dense is not None:
            return self._fit_dense(lib, X, y, groups)
        indptr = np.ascontiguousarray(X.indptr, dtype=np.int32)
        indices = np.ascontiguousarray(X.indices, dtype=np.int32)
        n_labels = len(np.unique(y))
        group_label = (C.c_float * max(n_labels, 1))()
        n_class = (C.c_int * 1)(self.num_class)
        per_iter = (C.c_int * 1)(0)
        self.model = C.c_void_p(None)
        grp = None if groups is None else np.ascontiguousarray(groups, dtype=np.int32)
        lib.sparse_train_scikit(X.shape[0], _ptr(X.data), _ptr(indptr), _ptr(indices), _ptr(y), self.depth,
                                self.n_trees, self.n_gpus, self.min_child_weight, self.lambda_tgbm, self.gamma,
                                self.max_num_bin, self.verbose, self.column_sampling_rate, int(self.bagging),
                                self.n_parallel_trees, self.learning_rate, self.objective.encode("utf-8"),
                                C.cast(n_class, C.c_void_p), self.tree_method.encode("utf-8"),
                                C.cast(C.byref(self.model), C.c_void_p), C.cast(per_iter, C.c_void_p),
                                C.cast(group_label, C.c_void_p), None if grp is None else _ptr(grp),
                                0 if grp is None else len(grp))
        self.num_class = n_class[0]
        self.tree_per_iter = per_iter[0]
        self.group_label = [group_label[i] for i in range(n_labels)]
        if not self.model:
            raise RuntimeError("The model returned is empty!")
        return self

    def _fit_dense(self, lib, X, y, groups):
        group_label = np.zeros(len(y), dtype=np.float32)
        n_labels = C.c_int(0)
        n_class = C.c_int(self.num_class)
        per_iter = C.c_int(0)
        self.model = C.c_void_p(None)
        grp = None if groups is None else np.ascontiguousarray(groups, dtype=np.int32)
        lib.tgbm_train_dense(X.shape[0], X.shape[1], _ptr(X), int(X.dtype == np.float64), _ptr(y), self.depth,
                             self.n_trees, self.n_gpus, self.min_child_weight, self.lambda_tgbm, self.gamma,
                             self.max_num_bin, self.verbose, self.column_sampling_rate, int(self.bagging),
                             self.n_parallel_trees, self.learning_rate, self.objective.encode("utf-8"),
                             C.byref(n_class), self.tree_method.encode("utf-8"), C.byref(self.model),
                             C.byref(per_iter), _ptr(group_label), C.byref(n_labels),
                             None if grp is None else _ptr(grp), 0 if grp is None else len(grp))
        self.num_class = n_class.value
        self.tree_per_iter = per_iter.value
        self.group_label = group_label[: n_labels.value].tolist()
        if not self.model:
            raise RuntimeError("The model returned is empty!")
        return self

    def predict(self, X, groups=None):
        if not self.model:
            raise ValueError("Please train the model first or load model from file!")
        lib = _lib.load()
        dense = _dense(X)
        X = _csr(X) if dense is None else dense
        n = X.shape[0]
        n_out = n * self.num_class if self.objective == "multi:softprob" else n
        out = np.zeros(max(n_out, n * max(self.tree_per_iter, 1)), dtype=np.float32)
        labels = np.asarray(self._class_labels(), dtype=np.float32)
        grp = None if groups is None else np.ascontiguousarray(groups, dtype=np.int32)
        if dense is not None:
            lib.tgbm_predict_dense(n, X.shape[1], _ptr(X), int(X.dtype == np.float64), _ptr(out), C.byref(self.model),
                                   self.n_trees, self.tree_per_iter, self.objective.encode("utf-8"), self.num_class,
                                   self.learning_rate, _ptr(labels), None if grp is None else _ptr(grp),
                                   0 if grp is None else len(grp), self.verbose)
            return self._predictions(out, n, n_out)
        indptr = np.ascontiguousarray(X.indptr, dtype=np.int32)
        indices = np.ascontiguousarray(X.indices, dtype=np.int32)
        lib.sparse_predict_scikit(n, _ptr(X.data), _ptr(indptr), _ptr(indices), _ptr(out),
                                  C.cast(C.byref(self.model), C.c_void_p), self.n_trees, self.tree_per_iter,
                                  self.objective.encode("utf-8"), self.num_class, self.learning_rate, _ptr(labels),
                                  None if grp is None else _ptr(grp), 0 if grp is None else len(grp), self.verbose)
        return self._predictions(out, n, n_out)

    def _class_labels(self):
        """The labels a prediction maps to: the library reads num_class of them (a regressor's list has an entry per
        distinct target, none of which is read)."""
        return (self.group_label or [0.0])[: max(self.num_class, 2)]

    def _predictions(self, out, n, n_out):
        if self.objective == "multi:softprob":
            # the library returns class-major probabilities; the reference wrapper reshapes them as
            # [-1, num_class] without transposing (thundergbm.py:169-171) and so does this one
            self.predict_label = out[:n_out].reshape([-1, self.num_class])
        else:
            self.predict_label = out[:n].copy()
        return self.predict_label

    def predict_proba_class_major(self, X):
        """multi:softprob probabilities as [num_class, n_rows] (the layout the library produces)."""
        p = self.predict(X)
        return p.reshape(self.num_class, -1)

    def save_model(self, model_path):
        if not self.model:
            raise ValueError("Please train the model first or load model from file!")
        labels = np.asarray(self.group_label if self.group_label else [0.0], dtype=np.float32)
        _lib.load().save(model_path.encode("utf-8"), self.objective.encode("utf-8"), self.learning_rate,
                         self.num_class, self.n_trees, self.tree_per_iter, C.cast(C.byref(self.model), C.c_void_p),
                         _ptr(labels))

    def load_model(self, model_path):
        lib = _lib.load()
        self._release()
        self.model = C.c_void_p(None)
        lr = (C.c_float * 1)()
        n_class = (C.c_int * 1)()
        n_trees = (C.c_int * 1)()
        per_iter = (C.c_int * 1)()
        lib.load_model(model_path.encode("utf-8"), C.cast(lr, C.c_void_p), C.cast(n_class, C.c_void_p),
                       C.cast(n_trees, C.c_void_p), C.cast(per_iter, C.c_void_p),
                       C.cast(C.byref(self.model), C.c_void_p))
        if not self.model:
            raise ValueError("Model is None.")
        self.learning_rate = lr[0]
        self.num_class = n_class[0]
        self.n_trees = n_trees[0]
        self.tree_per_iter = per_iter[0]
        # load_config copies every label the file stores (scikit_tgbm.cpp:173-182) and has no capacity argument:
        # files written by the CLI for reg:* / rank:* objectives hold one label per training row, so the buffer is
        # sized from the file's own label count (header: i32 objective length, objective, f32 learning rate,
        # i32 num_class, i32 n_trees, f32 base_score, i32 label count; parser.cpp:146-157)
        n_stored = _stored_label_count(model_path)
        labels = (C.c_float * max(n_stored, self.num_class, 1))()
        lib.load_config(model_path.encode("utf-8"), C.cast(labels, C.c_void_p))
        self.group_label = [labels[i] for i in range(self.num_class)]

    def get_trees(self):
        """Every tree as parallel heap-ordered arrays (the dictionaries the reference hands to shap). The trees' arrays are disjoint parts
        of seven that all of them share: copy those of a tree that is kept without the others."""
        if not self.model:
            raise ValueError("Please train the model first or load model from file!")
        lib = _lib.load()
        total = self.n_trees * self.tree_per_iter
        n_nodes = np.zeros(total, dtype=np.int32)
        mp = C.cast(C.byref(self.model), C.c_void_p)
        lib.get_n_nodes(mp, _ptr(n_nodes), self.n_trees, self.tree_per_iter)
        ends = np.cumsum(n_nodes)
        n = int(ends[-1]) if total else 0
        names = ("children_left", "children_right", "children_default", "feature", "threshold", "value", "node_sample_weight")
        arrays = [np.empty(n, np.int32 if k < 4 else np.float32) for k in range(7)]
        lib.tgbm_get_trees(mp, total, *(_ptr(a) for a in arrays))  # (one call: seven arrays of each tree's own took 8 us a tree)
        arrays[5] = arrays[5].reshape(-1, 1)
        return [{name: a[e - k:e] for name, a in zip(names, arrays)} for k, e in zip(n_nodes.tolist(), ends.tolist())]

    def get_shap_trees(self):
        """The trees as shap.explainers.tree.Tree objects (python/thundergbm/thundergbm.py:284-348); like
        the reference only for models with one tree per iteration, and only when shap is installed."""
        if self.objective != "binary:logistic" and self.tree_per_iter != 1:
            raise RuntimeError("not supported yet!")
        import shap.explainers.tree as shap_tree
        return [shap_tree.Tree(t) for t in self.get_trees()[:: max(self.tree_per_iter, 1)]]

    def cv(self, X, y, folds=None, nfold=5, shuffle=True, seed=0):
        """k-fold cross-validation with the reference's fold construction and result keys
        (python/thundergbm/thundergbm.py:223-282): fold size int(n / nfold), folds cut from a seeded
        permutation, accuracy for classifiers and mean squared error (reported under the RMSE keys, as
        there) for regressors."""
        import statistics

        X = _csr(X)
        y = np.ascontiguousarray(y, dtype=np.float32)
        n = X.shape[0]
        if folds is not None:
            train_ids = [f[0] for f in folds]
            test_ids = [f[1] for f in folds]
            nfold = len(folds)
        else:
            order = np.random.RandomState(seed).permutation(n) if shuffle else np.arange(n)
            step = int(n / nfold)
            test_ids = [order[i:i + step] for i in range(0, n, step)]
            train_ids = [np.concatenate([test_ids[i] for i in range(nfold) if i != k]) for k in range(nfold)]
        classifier = getattr(self, "_impl", "") == "classifier"
        train_scores, test_scores = [], []
        for k in range(nfold):
            self.fit(X[train_ids[k], :], y[train_ids[k]])
            for ids, scores in ((train_ids[k], train_scores), (test_ids[k], test_scores)):
                pred = self.predict(X[ids, :])
                if classifier:
                    scores.append(float(np.mean(pred == y[ids])))
                else:
                    scores.append(float(np.mean((pred - y[ids]) ** 2)))
        name = "accuracy" if classifier else "RMSE"
        self.eval_res = {
            "train-%s-mean" % name: statistics.mean(train_scores), "train-%s-std" % name: statistics.stdev(train_scores),
            "test-%s-mean" % name: statistics.mean(test_scores), "test-%s-std" % name: statistics.stdev(test_scores)}
        return self.eval_res


class TGBMClassifier(TGBMModel, ClassifierMixin):
    _impl = "classifier"

    def __init__(self, depth=6, n_trees=40, n_gpus=1, min_child_weight=1.0, lambda_tgbm=1.0, gamma=1.0,
                 max_num_bin=255, verbose=1, column_sampling_rate=1.0, bagging=0, n_parallel_trees=1,
                 learning_rate=1.0, objective="multi:softmax", num_class=2, tree_method="auto"):
        super().__init__(depth, n_trees, n_gpus, min_child_weight, lambda_tgbm, gamma, max_num_bin, verbose,
                         column_sampling_rate, bagging, n_parallel_trees, learning_rate, objective, num_class,
                         tree_method)


class TGBMRegressor(TGBMModel, RegressorMixin):
    _impl = "regressor"

    def __init__(self, depth=6, n_trees=40, n_gpus=1, min_child_weight=1.0, lambda_tgbm=1.0, gamma=1.0,
                 max_num_bin=255, verbose=1, column_sampling_rate=1.0, bagging=0, n_parallel_trees=1,
                 learning_rate=1.0, objective="reg:linear", num_class=1, tree_method="auto"):
        super().__init__(depth, n_trees, n_gpus, min_child_weight, lambda_tgbm, gamma, max_num_bin, verbose,
                         column_sampling_rate, bagging, n_parallel_trees, learning_rate, objective, num_class,
                         tree_method)
