"""The work that users have this package do, as cases that can be timed: training and prediction through
thundersvm_amd.model, from a 150-row data set to hundreds of thousands of rows.

A case names a family of data (how rows and labels are distributed, dense or sparse), its sizes, the SVM type, kernel and
parameters, and what is called: `train`, `predict` or `cross_validation`.  `resident` says where the rows are before the
call: in HBM (a Dataset that the program has uploaded and keeps) or in host arrays that go through the whole call.
Feature values are exactly floats, as those of a LibSVM file are."""
import math

import numpy as np

from thundersvm_amd.data import CsrData
from thundersvm_amd.model import Dataset, Model, make_param

C_SVC, NU_SVC, ONE_CLASS, EPSILON_SVR, NU_SVR = range(5)
LINEAR, POLY, RBF, SIGMOID = range(4)

# Share of the training rows that end up as support vectors, about, by family: how many kernel rows a solution needs.
SV_SHARE = {"blobs": 0.7, "pixels": 0.9, "text": 0.5, "mixed": 0.33, "smooth": 0.8}


def _case(do, family, n, d, classes=2, svm=C_SVC, kernel=RBF, C=1.0, gamma=0.0, nu=0.5, p=0.1, spread=1.0, resident=False, rows=0, folds=0):
    return dict(do=do, family=family, n=n, d=d, classes=classes, svm=svm, kernel=kernel, C=C, gamma=gamma, nu=nu, p=p, spread=spread,
                resident=resident, rows=rows, folds=folds)


def listed():
    named = [
        # a first try on a textbook data set: three classes of flowers by four measurements
        ("train 3 classes 150x4", _case("train", "blobs", 150, 4, classes=3, C=10.0, gamma=0.5, spread=1.0)),
        # a small image or sensor problem with many classes: 45 one-vs-one problems of a few hundred rows
        ("train 10 classes 1797x64", _case("train", "blobs", 1797, 64, classes=10, C=10.0, gamma=0.0156, spread=0.6)),
        # the small binary benchmark configuration: 3,200 rows, two overlapping blobs
        ("train blobs 3200x32", _case("train", "blobs", 3200, 32, C=100.0, gamma=0.5, spread=0.5)),
        # nu-SVC, the other classification formulation, on an ordinary table
        ("train nu-svc 5001x23", _case("train", "blobs", 5001, 23, svm=NU_SVC, nu=0.4, gamma=0.05, spread=0.35)),
        # pixel-like images, 784 columns and four fifths zeros, uploaded once (a parameter search trains on them many times)
        ("train pixels 20000x784", _case("train", "pixels", 20000, 784, C=10.0, gamma=0.125, resident=True)),
        # sparse text with a linear kernel
        ("train text linear 18000", _case("train", "text", 18000, 20958, kernel=LINEAR, C=1.0)),
        # epsilon-SVR on ninety dense columns
        ("train svr 40000x90", _case("train", "smooth", 40000, 90, svm=EPSILON_SVR, C=10.0, gamma=0.05, p=0.1)),
        # the headline benchmark problem's data (ten continuous columns, two one-hot groups, seven skewed classes), at a size
        # that trains within two seconds whichever mixture a seed draws
        ("train 7 classes 300000x54", _case("train", "mixed", 300000, 54, classes=7, C=3.0, gamma=1.0, resident=True)),
        # five-fold cross-validation, what a grid search calls for each of its points
        ("cross-validation 1203x13", _case("cross_validation", "blobs", 1203, 13, C=2.0, gamma=0.08, spread=0.4, folds=5)),
        # serving: one request's rows against a trained model
        ("predict 3 rows", _case("predict", "blobs", 3200, 32, C=100.0, gamma=0.5, spread=0.5, rows=3)),
        # scoring a table that is already in HBM with a multi-class model
        ("predict 7 classes 50000x54", _case("predict", "mixed", 20000, 54, classes=7, C=3.0, gamma=1.0, resident=True, rows=50000)),
        # scoring sparse text from host arrays
        ("predict text 4099", _case("predict", "text", 12000, 20958, C=1.0, gamma=1.0, rows=4099)),
    ]
    return [dict(c, name=name) for name, c in named]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["few rows", "many classes", "blobs", "nu", "pixels", "text", "svr", "mixed", "folds", "serve", "score", "score text"])
    C = round(math.exp(rng.uniform(math.log(0.5), math.log(16.0))), 3)
    resident = rng.random() < 0.5
    if kind == "few rows":
        d = rng.randint(2, 40)
        return _case("train", "blobs", _log(rng, 60, 1000), d, classes=rng.randint(2, 4), kernel=rng.choice([LINEAR, POLY, RBF]), C=C,
                     gamma=round(1.0 / d, 4), spread=0.7, resident=resident)
    if kind == "many classes":
        d = rng.randint(8, 130)
        return _case("train", "blobs", _log(rng, 600, 8000), d, classes=rng.randint(5, 14), C=C, gamma=round(1.0 / d, 4), spread=0.6,
                     resident=resident)
    if kind == "blobs":
        return _case("train", "blobs", _log(rng, 1000, 30000), rng.randint(16, 64), C=round(C * 6, 3), gamma=0.5, spread=0.5, resident=resident)
    if kind == "nu":
        d = rng.randint(10, 60)
        svm = rng.choice([NU_SVC, ONE_CLASS, NU_SVR])
        return _case("train", "smooth" if svm == NU_SVR else "blobs", _log(rng, 500, 12000), d, svm=svm,
                     nu=round(rng.uniform(0.1, 0.5), 3), C=min(C, 4.0), gamma=round(1.0 / d, 4), spread=0.35, resident=resident)
    if kind == "pixels":
        return _case("train", "pixels", _log(rng, 2000, 40000), rng.randint(150, 900), C=C, gamma=round(98.0 / 784, 4), resident=resident)
    if kind == "text":
        return _case("train", "text", _log(rng, 2000, 60000), _log(rng, 5000, 60000), kernel=rng.choice([LINEAR, RBF]), C=min(C, 2.0), gamma=1.0,
                     resident=resident)
    if kind == "svr":
        return _case("train", "smooth", _log(rng, 2000, 120000), rng.randint(50, 120), svm=EPSILON_SVR, C=C, gamma=0.05, p=0.1, resident=resident)
    if kind == "mixed":
        return _case("train", "mixed", _log(rng, 3000, 240000), 54, classes=7, C=3.0, gamma=1.0, resident=resident)
    if kind == "folds":
        d = rng.randint(4, 60)
        return _case("cross_validation", "blobs", _log(rng, 150, 4000), d, classes=rng.randint(2, 4), C=C, gamma=round(1.0 / d, 4), spread=0.5,
                     folds=rng.choice([3, 5, 10]))
    if kind == "serve":
        d = rng.randint(8, 130)
        return _case("predict", "blobs", _log(rng, 500, 12000), d, classes=rng.randint(2, 6), C=C, gamma=round(1.0 / d, 4), spread=0.4,
                     rows=_log(rng, 1, 300), resident=False)
    if kind == "score":
        family = rng.choice(["mixed", "smooth", "pixels"])
        d = 54 if family == "mixed" else rng.randint(60, 500) if family == "pixels" else rng.randint(50, 120)
        return _case("predict", family, _log(rng, 3000, 20000), d, classes=7 if family == "mixed" else 2,
                     svm=EPSILON_SVR if family == "smooth" else C_SVC, C=3.0,
                     gamma={"mixed": 1.0, "smooth": 0.05, "pixels": 0.125}[family], rows=_log(rng, 1000, 60000), resident=resident)
    return _case("predict", "text", _log(rng, 2000, 16000), _log(rng, 5000, 60000), C=min(C, 2.0), gamma=1.0, kernel=rng.choice([LINEAR, RBF]),
                 rows=_log(rng, 30, 8000), resident=False)


# ------------------------------------------------------------------------------------------------
# Data.  `rng` draws everything, the distribution of a family's labels included, so another seed is another problem.
# ------------------------------------------------------------------------------------------------
def _dense_csr(x, y, keep_zeros=True):
    n, d = x.shape
    if keep_zeros:
        return CsrData(np.arange(n + 1, dtype=np.int64) * d, np.tile(np.arange(1, d + 1, dtype=np.int32), n), x.reshape(-1).astype(np.float64), y)
    stored = x != 0
    ptr = np.zeros(n + 1, dtype=np.int64)
    np.cumsum(stored.sum(axis=1), out=ptr[1:])
    return CsrData(ptr, np.nonzero(stored)[1].astype(np.int32) + 1, x[stored].astype(np.float64), y)


def _blobs(rng, case):
    """Gaussian blobs, one per class, their centres `spread` apart per column: an ordinary standardised table."""
    k, d = case["classes"], case["d"]
    sign = np.where(np.arange(2)[:, None] == 0, 1.0, -1.0) * np.ones(d)
    centres = (sign if k == 2 else rng.standard_normal((k, d))) * case["spread"]

    def make(n):
        c = rng.permutation(np.arange(n) % k)
        x = (centres[c] + rng.standard_normal((n, d))).astype(np.float32)
        return _dense_csr(x, (1.0 - 2.0 * c) if k == 2 else c + 1.0)
    return make


def _pixels(rng, case):
    """Pixels k/255, four fifths of them zero; the label says on which side of a random quadratic surface a row lies, 5 % flipped."""
    d = case["d"]
    w, u = rng.standard_normal(d), rng.standard_normal(d)

    def make(n):
        k = rng.integers(0, 256, size=(n, d), dtype=np.uint8)
        k[rng.integers(0, 256, size=(n, d), dtype=np.uint8) < 205] = 0
        x = k.astype(np.float32) / np.float32(255)
        score = x @ w.astype(np.float32) + (x * x) @ u.astype(np.float32)
        y = np.where(score > np.median(score), 1.0, -1.0)
        y[rng.random(n) < 0.05] *= -1
        return _dense_csr(x, y, keep_zeros=False)
    return make


def _text(rng, case):
    """Sparse rows of about fifty columns (Zipf 1.1), lognormal values, rows of length one; a sparse random hyperplane, 3 % flipped."""
    d = case["d"]
    cdf = np.cumsum(np.arange(1, d + 1, dtype=np.float64) ** -1.1)
    cdf /= cdf[-1]
    w = np.zeros(d + 1)
    w[np.searchsorted(cdf, rng.random(800)).clip(0, d - 1) + 1] = rng.standard_normal(800)

    def make(n):
        lens = np.maximum(rng.poisson(70, size=n), 1)
        row = np.repeat(np.arange(n, dtype=np.int64), lens)
        col = np.searchsorted(cdf, rng.random(len(row))).clip(0, d - 1) + 1
        key = np.unique(row * (d + 2) + col)
        row, col = key // (d + 2), (key % (d + 2)).astype(np.int32)
        ptr = np.zeros(n + 1, dtype=np.int64)
        np.cumsum(np.bincount(row, minlength=n), out=ptr[1:])
        v = rng.lognormal(0.0, 1.0, size=len(col))
        val = (v / np.sqrt(np.add.reduceat(v * v, ptr[:-1]))[row]).astype(np.float32).astype(np.float64)
        score = np.add.reduceat(val * w[col], ptr[:-1])
        y = np.where(score > np.median(score), 1.0, -1.0)
        y[rng.random(n) < 0.03] *= -1
        return CsrData(ptr, col, val, y)
    return make


def _mixed(rng, case):
    """Ten standardised columns from a seven-component mixture, then one-hot groups of 4 and 40: twelve stored values per row."""
    pri = np.array([0.36, 0.49, 0.06, 0.005, 0.016, 0.03, 0.035])
    pri /= pri.sum()
    means, scales = rng.standard_normal((7, 10)) * 1.5, 0.5 + rng.random((7, 10))
    c4 = np.cumsum(rng.dirichlet(np.ones(4) * 0.7, size=7), axis=1)
    c40 = np.cumsum(rng.dirichlet(np.ones(40) * 0.3, size=7), axis=1)
    mu, sd = pri @ means, np.sqrt(pri @ (scales ** 2 + means ** 2) - (pri @ means) ** 2)

    def make(n):
        cls = np.searchsorted(np.cumsum(pri), rng.random(n)).clip(0, 6)
        cls[:7] = np.arange(7)
        cont = ((means[cls] + scales[cls] * rng.standard_normal((n, 10)) - mu) / sd).astype(np.float32)
        u4, u40 = rng.random(n), rng.random(n)
        g4, g40 = np.zeros(n, dtype=np.int32), np.zeros(n, dtype=np.int32)
        for c in range(7):
            at = np.flatnonzero(cls == c)
            g4[at] = np.searchsorted(c4[c], u4[at]).clip(0, 3)
            g40[at] = np.searchsorted(c40[c], u40[at]).clip(0, 39)
        col = np.empty((n, 12), dtype=np.int32)
        col[:, :10], col[:, 10], col[:, 11] = np.arange(1, 11), 11 + g4, 15 + g40
        val = np.ones((n, 12))
        val[:, :10] = cont
        return CsrData(np.arange(n + 1, dtype=np.int64) * 12, col.reshape(-1), val.reshape(-1), cls + 1.0)
    return make


def _smooth(rng, case):
    """Standard normal columns, y = sin(w1.x) + 0.5 (w2.x)^2 + noise."""
    d = case["d"]
    w1, w2 = rng.standard_normal(d), rng.standard_normal(d)
    w1, w2 = w1 / np.linalg.norm(w1), w2 / np.linalg.norm(w2)

    def make(n):
        x = rng.standard_normal((n, d), dtype=np.float32)
        xd = x.astype(np.float64)
        y = np.sin(xd @ w1) + 0.5 * (xd @ w2) ** 2 + 0.1 * rng.standard_normal(n)
        return _dense_csr(x, y.astype(np.float32).astype(np.float64))
    return make


FAMILIES = {"blobs": _blobs, "pixels": _pixels, "text": _text, "mixed": _mixed, "smooth": _smooth}


def prepare(case, seed):
    """The rows (host arrays, or a Dataset uploaded to HBM), the parameters and, for prediction, the trained model."""
    make = FAMILIES[case["family"]](np.random.Generator(np.random.PCG64(seed)), case)
    param = make_param(svm_type=case["svm"], kernel_type=case["kernel"], C=case["C"], gamma=case["gamma"], nu=case["nu"], p=case["p"])
    data = make(case["n"])
    if case["svm"] == ONE_CLASS:
        data = CsrData(data.ptr, data.col, data.val, np.ones(data.n))
    state = dict(do=case["do"], svm=case["svm"], param=param, folds=case["folds"], n=case["n"])
    if case["do"] == "predict":
        state["model"] = Model(case["svm"]).train(data, param)
        data = make(case["rows"])
    if case["do"] == "cross_validation":
        data = Dataset(data)      # (this entry point takes no other form; its rows stay in host memory)
    elif case["resident"]:
        data = Dataset(data).to_device()
    state["data"] = data
    return state


def run(state):
    if state["do"] == "train":
        m = Model(state["svm"]).train(state["data"], state["param"])
        # one column of coefficients per training row: which rows are support vectors depends on the data
        coef = np.zeros((m.coef.size // max(m.total_sv, 1), state["n"]))
        coef[:, m.sv_indices] = m.coef.reshape(coef.shape[0], -1)
        return {"coef": coef, "rho": m.rho, "n_sv": m.n_sv, "label": m.label}
    if state["do"] == "cross_validation":
        return Model(state["svm"]).cross_validation(state["data"], state["param"], state["folds"])
    labels, dec = state["model"].predict(state["data"])
    return {"labels": labels, "dec": dec}


def _stored(case):
    """Stored values of a row, about."""
    return {"pixels": 0.2 * case["d"], "text": 50.0, "mixed": 12.0}.get(case["family"], float(case["d"]))


def work(case):
    """Training: the rows once, the kernel row of every support vector over the instances of its class pair, the coefficients.
    Prediction: both sets of rows once, one kernel value and one product per class pair side for every row and support vector."""
    n, k = case["n"], case["classes"] if case["svm"] in (C_SVC, NU_SVC) else 2
    per_value = 2.0 * _stored(case)
    share = SV_SHARE[case["family"]]
    row_bytes = 12.0 * _stored(case) + 8.0
    sv = share * n
    if case["do"] == "predict":
        return {"bytes": (case["rows"] + sv) * row_bytes + 8.0 * (k - 1) * sv + case["rows"] * 8.0 * (1 + k * (k - 1) / 2),
                "flops": case["rows"] * sv * (per_value + 2.0 * (k - 1))}
    if case["family"] == "mixed":
        pri = [0.36, 0.49, 0.06, 0.005, 0.016, 0.03, 0.035]
    else:
        pri = [1.0 / k] * k
    pairs = sum((pri[i] + pri[j]) ** 2 for i in range(k) for j in range(i)) if case["svm"] in (C_SVC, NU_SVC) else 1.0
    flops = share * float(n) * n * pairs * per_value
    if case["do"] == "cross_validation":
        f = case["folds"]
        return {"bytes": n * (row_bytes + 8.0), "flops": flops * ((f - 1.0) ** 2 / f + (f - 1.0) / f)}
    return {"bytes": n * row_bytes + 12.0 * (k - 1) * sv, "flops": flops}


def tolerance(case):
    """Kernel values are rounded to float, everything else is 64-bit; a solver that takes the same steps and sums in another order
    agrees to the last digits of a float (coefficients, rho and decision values: 1e-6)."""
    return {"rel": 1e-6}
