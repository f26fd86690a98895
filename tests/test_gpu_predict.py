"""Prediction in one pass (tsvm_predict_dec_values_dense behind SvmModel::predict_dec_values, replacing
svmmodel.cpp:74-117's get_rows + sum_kernel_values): decision values against the CPU oracle's serial sums at the
path's tolerance (1e-6 absolute), and against the two-call form on the device, for every shape the kernels
distinguish: one to eleven coefficient rows, few / many features, indicator columns, all four kernels, batch sizes
that do and do not fill a tile, rows already resident on the device."""
import numpy as np
import pytest
import torch

import gpu_util as G
import oracle_lib as O
from thundersvm_amd import capi
from thundersvm_amd import data as D
from thundersvm_amd.model import Dataset, Model, make_param

pytestmark = pytest.mark.gpu


def _oparam(prm):
    return O.make_param(svm_type=prm.svm_type, kernel_type=prm.kernel_type, degree=prm.degree, gamma=prm.gamma,
                        coef0=prm.coef0, C_=prm.C, nu=prm.nu, p=prm.p, epsilon=prm.epsilon, max_iter=prm.max_iter,
                        max_mem_size=prm.max_mem_size, expf_mode=1)


def _blobs(rng, k, per, d, one_hot=0, spread=0.8):
    """k Gaussian classes in d continuous features, optionally followed by a `one_hot`-way indicator block."""
    centres = 2.0 * rng.standard_normal((k, d))
    cls = rng.permutation(np.repeat(np.arange(k), per))
    x = (centres[cls] + spread * rng.standard_normal((k * per, d))).astype(np.float32)
    if one_hot:
        hot = np.zeros((k * per, one_hot), dtype=np.float32)
        hot[np.arange(k * per), (cls * 3 + rng.integers(0, 3, k * per)) % one_hot] = 1.0
        x = np.concatenate([x, hot], axis=1)
    return x, (cls + 1).astype(np.float64)


def _check(tr, te, prm, monkeypatch, batch=-1, tol=1e-6):
    gm = Model(prm.svm_type).train(tr, prm)
    om = O.Model(tr.ptr, tr.col, tr.val, tr.y, _oparam(prm))
    assert gm.total_sv == om.total_sv
    glab, gdec = gm.predict(te, batch)
    olab, odec = om.predict(te.ptr, te.col, te.val, 100)
    scale = max(1.0, float(np.abs(gm.coef).sum()) * 1e-6)      # (huge cancelling coefficients move with the order of the sums)
    assert np.abs(gdec - odec).max() < tol * scale
    clear = np.abs(odec).min(axis=1) > tol * scale
    if prm.svm_type in (0, 1):
        assert np.array_equal(glab[clear], olab[clear])
    # the same model through the two-call form (kernel rows written out, then sum_kernel_values)
    monkeypatch.setenv("TSVM_PREDICT_UNFUSED", "1")
    _, tdec = gm.predict(te, 100)
    monkeypatch.delenv("TSVM_PREDICT_UNFUSED")
    assert np.abs(gdec - tdec).max() < 1e-9 * max(1.0, float(np.abs(gm.coef).sum()))
    # rows resident on the device give what rows from the host give
    ds = Dataset(te).to_device()
    _, ddec = gm.predict(ds, batch)
    assert np.abs(ddec - gdec).max() < 1e-9 * max(1.0, float(np.abs(gm.coef).sum()))
    return gm, gdec


@pytest.mark.parametrize("k", [2, 3, 4, 5, 6, 7, 8, 9, 10, 12])
def test_class_counts_few_features(k, monkeypatch):
    rng = np.random.default_rng(100 + k)
    x, y = _blobs(rng, k, 60, 7)
    xt, _ = _blobs(np.random.default_rng(200 + k), k, 13, 7)
    _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=0, kernel_type=2, gamma=0.3, C=4.0),
           monkeypatch)


@pytest.mark.parametrize("k", [2, 3, 7, 9, 12])
def test_class_counts_indicator_columns(k, monkeypatch):
    rng = np.random.default_rng(300 + k)
    x, y = _blobs(rng, k, 80, 5, one_hot=40)
    xt, _ = _blobs(np.random.default_rng(400 + k), k, 21, 5, one_hot=40)
    gm, _ = _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))),
                   make_param(svm_type=0, kernel_type=2, gamma=0.2, C=4.0), monkeypatch)
    # a batch whose values in those columns are not all zeros and ones takes the plain columns
    xt2 = xt.copy()
    xt2[3, -2] = 0.5
    te2 = D.from_dense(xt2, np.zeros(len(xt2)))
    om = O.Model(D.from_dense(x, y).ptr, D.from_dense(x, y).col, D.from_dense(x, y).val, y, _oparam(make_param(svm_type=0, kernel_type=2, gamma=0.2, C=4.0)))
    _, gdec = gm.predict(te2)
    _, odec = om.predict(te2.ptr, te2.col, te2.val, 100)
    assert np.abs(gdec - odec).max() < 1e-6


@pytest.mark.parametrize("k", [2, 4, 12, 26])
def test_class_counts_many_features(k, monkeypatch):
    rng = np.random.default_rng(500 + k)
    x, y = _blobs(rng, k, 40, 200, spread=1.5)
    xt, _ = _blobs(np.random.default_rng(600 + k), k, 9, 200, spread=1.5)
    _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=0, kernel_type=2, gamma=0.004, C=4.0),
           monkeypatch)


@pytest.mark.parametrize("kt,extra", [(0, {}), (1, dict(gamma=0.1, degree=3, coef0=0.5)), (3, dict(gamma=0.05, coef0=0.1))])
@pytest.mark.parametrize("d", [12, 150])
def test_other_kernels(kt, extra, d, monkeypatch):
    rng = np.random.default_rng(700 + kt + d)
    x, y = _blobs(rng, 3, 70, d)
    xt, _ = _blobs(np.random.default_rng(800 + kt + d), 3, 17, d)
    if d > 100:
        x, xt = x * 0.2, xt * 0.2
    _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=0, kernel_type=kt, C=1.0, **extra),
           monkeypatch)


@pytest.mark.parametrize("svm_type,extra", [(3, dict(p=0.1, C=5.0)), (4, dict(nu=0.4, C=5.0)), (2, dict(nu=0.2)), (1, dict(nu=0.3))])
def test_other_models(svm_type, extra, monkeypatch):
    rng = np.random.default_rng(900 + svm_type)
    x = rng.standard_normal((500, 9)).astype(np.float32)
    y = np.sin(x[:, 0]) + 0.3 * x[:, 1] if svm_type in (3, 4) else np.where(x[:, 0] + x[:, 1] > 0, 1.0, -1.0)
    xt = rng.standard_normal((130, 9)).astype(np.float32)
    _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=svm_type, kernel_type=2, gamma=0.2, **extra),
           monkeypatch)


@pytest.mark.parametrize("batch", [1, 63, 64, 65, 1000, -1])
def test_batch_sizes(batch, monkeypatch):
    rng = np.random.default_rng(77)
    x, y = _blobs(rng, 4, 300, 20)
    xt, _ = _blobs(np.random.default_rng(78), 4, 50, 20)
    _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=0, kernel_type=2, gamma=0.1, C=2.0),
           monkeypatch, batch=batch)


def test_test_rows_with_other_feature_ranges(monkeypatch):
    """Features the support vectors do not have are dropped from the products but stay in the row's self dot product
    (kernelmatrix.cpp:290-295,392); rows with fewer features than the support vectors are padded."""
    rng = np.random.default_rng(5)
    x, y = _blobs(rng, 3, 100, 10)
    tr = D.from_dense(x, y)
    wide = np.concatenate([_blobs(np.random.default_rng(6), 3, 20, 10)[0], rng.standard_normal((60, 7)).astype(np.float32)], axis=1)
    narrow = _blobs(np.random.default_rng(7), 3, 20, 10)[0][:, :4]
    for xt in (wide, narrow):
        _check(tr, D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=0, kernel_type=2, gamma=0.3, C=4.0), monkeypatch)


def test_long_chunks_and_many_support_vectors(monkeypatch):
    """Enough support vectors and rows that workgroups walk chunks of many column tiles."""
    rng = np.random.default_rng(11)
    x = rng.standard_normal((20000, 16)).astype(np.float32)
    y = np.where(np.sin(3 * x[:, 0]) * x[:, 1] + 0.3 * rng.standard_normal(20000) > 0, 1.0, -1.0)
    xt = rng.standard_normal((9000, 16)).astype(np.float32)
    gm, _ = _check(D.from_dense(x, y), D.from_dense(xt, np.zeros(len(xt))), make_param(svm_type=0, kernel_type=2, gamma=0.5, C=1.0),
                   monkeypatch)
    assert gm.total_sv > 8000


@pytest.mark.parametrize("kt,long_row", [(2, False), (2, True), (0, False), (1, False)])
@pytest.mark.parametrize("m", [255, 256, 257, 300])
def test_sparse_rows_on_both_routes(kt, long_row, m):
    """Sparse support vectors: from 256 rows on a batch is multiplied with their sliced copy, smaller ones (and those with a
    row too long for it) are staged as a dense matrix.  The two agree in every bit and with the oracle; an empty row and
    columns that no support vector has are among the rows."""
    rng = np.random.default_rng(m + kt)
    n, d = 700, 2400

    def rows(count, width):
        lens = rng.integers(1, 20, count)
        lens[3] = 0
        if width > d and long_row:
            lens[5] = 1900
        ptr = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
        col = np.concatenate([np.sort(rng.choice(width, size=k, replace=False)) for k in lens]).astype(np.int32) + 1
        val = rng.standard_normal(len(col)).astype(np.float32).astype(np.float64)
        return D.CsrData(ptr, col, val, np.where(rng.random(count) < 0.5, 1.0, -1.0))
    tr, te = rows(n, d), rows(m, d + 50)
    prm = make_param(svm_type=0, kernel_type=kt, C=2.0, gamma=0.05, degree=2, coef0=0.5)
    gm = Model(0).train(tr, prm)
    om = O.Model(tr.ptr, tr.col, tr.val, tr.y, _oparam(prm))
    whole, parts = gm.predict(te)[1], gm.predict(te, 40)[1]
    assert np.array_equal(whole, parts)
    assert np.abs(whole - om.predict(te.ptr, te.col, te.val, 100)[1]).max() < 1e-6


def test_sparse_class_pair_whose_rows_are_all_empty():
    """A wide, sparse three-class problem in which two classes' rows hold no feature at all: their class pair is a CSR
    sub-problem without a single stored entry (every kernel value is kappa(0, 0)), so there is nothing to slice for the
    CSR kernels; training and prediction still agree with the oracle."""
    rng = np.random.default_rng(3)
    ptr, col, val, y = [0], [], [], []
    for i in range(12):
        cls = i % 3 + 1
        if cls == 3:
            c = np.sort(rng.choice(np.arange(1, 400), 3, replace=False))
            col += list(c)
            val += list(rng.standard_normal(3).astype(np.float32))
        ptr.append(len(col))
        y.append(float(cls))
    tr = D.CsrData(ptr, col, val, y)
    xt = rng.standard_normal((4, 399)).astype(np.float32) * (rng.random((4, 399)) < 0.01)
    te = D.from_dense(xt, np.zeros(4))
    prm = make_param(svm_type=0, kernel_type=2, gamma=0.01, C=1.0)
    gm = Model(0).train(tr, prm)
    om = O.Model(tr.ptr, tr.col, tr.val, tr.y, _oparam(prm))
    assert gm.total_sv == om.total_sv and np.array_equal(gm.coef, om.coef) and np.array_equal(gm.rho, om.rho)
    _, gdec = gm.predict(te)
    _, odec = om.predict(te.ptr, te.col, te.val, 100)
    assert np.abs(gdec - odec).max() < 1e-6


@pytest.mark.parametrize("last", [0.5, 0.1, float("inf")])
def test_what_is_known_of_sparse_values_goes_to_subsets(last):
    """The models of a sparse cross-validation take their support vectors out of the data set's device rows: finite values
    let them predict on the sliced copy, as a model of its own does."""
    import selftest_lib
    lib = selftest_lib.lib()
    assert lib.tsvm_selftest_subset_of_rows(last) == 0, lib.tsvm_selftest_last_error()


@pytest.mark.parametrize("last,first", [(1.0, 5), (0.0, 5), (2.0, -1)])
def test_indicator_columns_are_found_by_all_entries(last, first):
    """The host looks at the first entries only; what the last of 100,000 holds still decides."""
    import selftest_lib
    assert selftest_lib.lib().tsvm_selftest_indicator_run(last) == first


@pytest.mark.parametrize("m", [1, 255, 256, 300])
@pytest.mark.parametrize("kt", [0, 2])
def test_batch_without_any_entry(m, kt):
    """Rows without entries only, on sparse support vectors: every one is the zero vector."""
    rng = np.random.default_rng(kt)
    n, d = 700, 2400
    col = np.sort(rng.random((n, d)).argsort(1)[:, :12], 1).astype(np.int32).ravel() + 1
    tr = D.CsrData(np.arange(n + 1, dtype=np.int64) * 12, col, rng.standard_normal(12 * n).astype(np.float32).astype(np.float64),
                   np.where(rng.random(n) < 0.5, 1.0, -1.0))
    prm = make_param(kernel_type=kt, C=2.0, gamma=0.05)
    te = D.CsrData(np.zeros(m + 1, np.int64), np.zeros(0, np.int32), np.zeros(0), None)
    gm = Model(0).train(tr, prm)
    want = O.Model(tr.ptr, tr.col, tr.val, tr.y, _oparam(prm)).predict(te.ptr, te.col, te.val, 100)[1]
    for batch in (-1, 100):
        got = gm.predict(te, batch)[1]
        assert got.shape == want.shape and np.abs(got - want).max() < 1e-6 and (got == got[0]).all()
    assert np.array_equal(gm.predict(Dataset(te).to_device())[1], got)


@pytest.mark.parametrize("rows,entries", [(600, 4095), (600, 4096), (600, 4097), (9000, 37), (9000, 4096), (9000, 4097)])
def test_few_entries_are_read_in_place(rows, entries):
    """Dense support vectors: a batch of up to 4,096 entries is read by the kernel where it lies in host memory, however many rows
    they are spread over.  Either way the values are those of the same rows resident on the device, bit for bit, and the oracle's."""
    rng = np.random.default_rng(rows + entries)
    x, y = _blobs(rng, 3, 60, 9)
    tr = D.from_dense(x, y)
    prm = make_param(svm_type=0, kernel_type=2, gamma=0.3, C=2.0)
    at = np.sort(rng.choice(rows * 9, size=entries, replace=False))
    te = D.CsrData(np.searchsorted(at, np.arange(rows + 1, dtype=np.int64) * 9).astype(np.int64), (at % 9).astype(np.int32) + 1,
                   rng.standard_normal(entries).astype(np.float32).astype(np.float64), np.zeros(rows))
    gm = Model(0).train(tr, prm)
    got = gm.predict(te)[1]
    assert np.array_equal(got, gm.predict(Dataset(te).to_device())[1])
    assert np.array_equal(got, gm.predict(te)[1])
    om = O.Model(tr.ptr, tr.col, tr.val, tr.y, _oparam(prm))
    assert np.abs(got - om.predict(te.ptr, te.col, te.val, 100)[1]).max() < 1e-6


@pytest.mark.parametrize("groups", [1, 2, 3, 4, 5, 7])
def test_indicator_groups(groups, monkeypatch):
    """A row sets one column of each one-hot group: so many matches are added one by one, up to four without a loop."""
    rng = np.random.default_rng(300 + groups)
    x, y = _blobs(rng, 4, 60, 6)
    hot = np.zeros((len(y), groups * 9), dtype=np.float32)
    for g in range(groups):
        hot[np.arange(len(y)), g * 9 + (y.astype(int) * 2 + rng.integers(0, 3, len(y))) % 9] = 1.0
    x = np.concatenate([x, hot], axis=1)
    tr, te = D.CsrData(*_csr(x[:200]), y[:200]), D.CsrData(*_csr(x[200:]), y[200:])
    _check(tr, te, make_param(svm_type=0, kernel_type=2, gamma=0.1, C=2.0), monkeypatch)


def _csr(x):
    n, d = x.shape
    return np.arange(n + 1, dtype=np.int64) * d, np.tile(np.arange(1, d + 1, dtype=np.int32), n), x.reshape(-1).astype(np.float64)


def _votes(dec, k):
    m = dec.shape[0]
    votes = np.zeros((m, k), dtype=int)
    p = 0
    for i in range(k):
        for j in range(i + 1, k):
            pos = dec[:, p] > 0
            votes[:, i] += pos
            votes[:, j] += ~pos
            p += 1
    return votes.argmax(axis=1)   # (the first among equals)


@pytest.mark.parametrize("k", [2, 3, 7, 33, 64])
@pytest.mark.parametrize("m", [0, 1, 255, 256, 257, 1000])
def test_votes(k, m):
    """The vote kernel against the count in numpy: ties between classes, zeros (a vote for the second class), infinities and NaN."""
    import torch
    import gpu_util as G
    from thundersvm_amd import capi
    rng = np.random.default_rng(k * 1000 + m)
    dec = rng.choice([-1.5, -0.0, 0.0, 0.3, 2.0, np.inf, -np.inf, np.nan], size=(m, k * (k - 1) // 2))
    won = torch.full((m + 1,), -7, dtype=torch.int32, device="cuda")
    dec_d = G.dev(np.ascontiguousarray(dec if m else np.zeros((1, 1))))
    capi.call("tsvm_predict_votes", G.ptr(dec_d), m, k, G.ptr(won), G.stream())
    got = G.host(won)
    assert np.array_equal(got[:m], _votes(dec, k)) and got[m] == -7
    with pytest.raises(capi.TsvmError):
        capi.call("tsvm_predict_votes", G.ptr(dec_d), m, capi.kernel_lib().tsvm_predict_votes_max_classes() + 1, G.ptr(won), G.stream())


@pytest.mark.parametrize("k,rows", [(2, 20000), (5, 1638), (5, 1639), (70, 30)])
@pytest.mark.parametrize("dense", [True, False])
def test_labels_by_votes_on_the_device_and_on_the_host(k, rows, dense):
    """Labels are the vote over the decision values that come with them, whichever side takes it (16,384 pair votes on, up to 64
    classes: the device), in one batch or several, and a prediction leaves nothing to the next one."""
    rng = np.random.default_rng(k)
    x, y = _blobs(rng, k, 12 if k > 10 else 40, 6, spread=3.0)
    if not dense:
        x[rng.random(x.shape) < 0.3] = 0
        x = np.concatenate([x, np.zeros((len(y), 3000), dtype=np.float32)], axis=1)
        x[np.arange(len(y)), rng.integers(6, x.shape[1], len(y))] = 1.0
    def data(rows_of):
        if dense:
            return D.CsrData(*_csr(rows_of), y[:1].repeat(len(rows_of)))
        ptr = np.concatenate([[0], np.cumsum((rows_of != 0).sum(axis=1))]).astype(np.int64)
        r, c = np.nonzero(rows_of)
        return D.CsrData(ptr, c.astype(np.int32) + 1, rows_of[r, c].astype(np.float64), y[:1].repeat(len(rows_of)))
    tr = data(x)
    tr = D.CsrData(tr.ptr, tr.col, tr.val, y)
    prm = make_param(svm_type=0, kernel_type=2, gamma=0.1, C=1.0)
    m = Model(0).train(tr, prm)
    many, few = data(x[rng.integers(0, len(y), rows)]), data(x[:3])
    for d in (many, few, many):
        for batch in (-1, 700):
            labels, dec = m.predict(d, batch)
            assert np.array_equal(labels, m.label[_votes(dec, k)].astype(np.float64))


@pytest.mark.parametrize("svm_type,classes", [(capi.EPSILON_SVR, 2), (capi.NU_SVR, 2), (capi.C_SVC, 3), (capi.ONE_CLASS, 2)])
@pytest.mark.parametrize("n,d,kernel,folds", [(40, 3, capi.RBF, 5), (129, 16, capi.POLY, 2), (645, 17, capi.RBF, 10), (1003, 127, capi.LINEAR, 3),
                                              (1003, 128, capi.RBF, 3), (3300, 5, capi.RBF, 3)])
def test_folds_predicted_together(svm_type, classes, n, d, kernel, folds, monkeypatch):
    """A cross-validation whose folds are predicted by one launch gives what one call per fold gives: ragged blocks of rows, a fold
    of more than one batch (3,300 rows of three classes), one column too many for the kernel (128 features make 129 columns)."""
    rng = np.random.default_rng(n + d)
    x = rng.standard_normal((n, d)).astype(np.float32)
    c = rng.permutation(np.arange(n) % classes)
    # (folds are cut label by label, whatever the model: svmmodel.cpp:31-71)
    y = np.sign(x[:, 0]) if svm_type in (capi.EPSILON_SVR, capi.NU_SVR) else np.ones(n) if svm_type == capi.ONE_CLASS else c + 1.0
    if svm_type == capi.C_SVC:
        x[:, :2] += 1.5 * np.stack([c, c * c], axis=1)
    data = D.from_dense(x, y)
    prm = make_param(svm_type=svm_type, kernel_type=kernel, C=1.0, gamma=0.1 / d, nu=0.3, p=0.05, degree=2)
    together = Model(svm_type).cross_validation(Dataset(data), prm, folds)
    monkeypatch.setenv("TSVM_PREDICT_UNFUSED", "1")
    one_by_one = Model(svm_type).cross_validation(Dataset(data), prm, folds)
    if svm_type in (capi.EPSILON_SVR, capi.NU_SVR):
        # (the same kernel values and coefficients, their sums in another order: 1,000 terms of 2^-53 each, coefficients of at most 1)
        np.testing.assert_allclose(together, one_by_one, rtol=0, atol=1e-9 * (1 + np.abs(one_by_one).max()))
    else:
        assert np.mean(together != one_by_one) <= 0.002   # (a decision value of about zero may fall on either side)


@pytest.mark.parametrize("svm_type,classes", [(capi.EPSILON_SVR, 2), (capi.NU_SVR, 2), (capi.C_SVC, 3), (capi.ONE_CLASS, 1)])
@pytest.mark.parametrize("n,d,hot,kernel,folds", [(40, 3, 0, capi.RBF, 5), (129, 16, 0, capi.POLY, 2), (545, 17, 0, capi.RBF, 10), (603, 127, 0, capi.LINEAR, 3),
                                                  (603, 128, 0, capi.RBF, 3), (610, 6, 50, capi.LINEAR, 5), (610, 6, 50, capi.RBF, 5), (9000, 5, 0, capi.RBF, 3)])
def test_folds_are_predicted_as_one_by_one(svm_type, classes, n, d, hot, kernel, folds):
    """Every value of a cross-validation is, to the last bit, what a model that is trained on the fold's rows by themselves predicts in batches of
    1,000 rows.  Folds of small problems with up to 128 columns are predicted by one launch (128 features make 129)."""
    rng = np.random.default_rng(n + d + hot)
    x = rng.standard_normal((n, d + hot)).astype(np.float32)
    x[:, :d] *= (10.0 ** rng.uniform(-2, 0, d)).astype(np.float32)
    x[:, d:] = 0
    if hot:
        x[np.arange(n), d + rng.integers(0, hot - 2, n)] = 1
        x[np.arange(n), d + hot - 2 + rng.integers(0, 2, n)] = 1
    c = rng.permutation(np.arange(n) % classes)
    y = np.sign(x[:, 0]) if svm_type in (capi.EPSILON_SVR, capi.NU_SVR) else c + 1.0
    data = D.from_dense(x, y)
    prm = make_param(svm_type=svm_type, kernel_type=kernel, C=1.0, gamma=0.1 / d, nu=0.3, p=0.05, degree=2, max_iter=30)
    m = Model(svm_type)
    got = m.cross_validation(Dataset(data), prm, folds)
    # the folds (svmmodel.cpp:31-71): label by label in the order of the first instances, the last one takes what is left
    train, test = [[] for _ in range(folds)], [[] for _ in range(folds)]
    for label in y[np.sort(np.unique(y, return_index=True)[1])]:
        ids = np.flatnonzero(y == label)
        each = len(ids) // folds
        for k in range(folds):
            lo, hi = each * k, len(ids) if k == folds - 1 else each * (k + 1)
            test[k].append(ids[lo:hi])
            train[k].append(np.concatenate([ids[:lo], ids[hi:]]))
    want = np.zeros(n)
    for k in range(folds):
        tr, te = np.concatenate(train[k]), np.concatenate(test[k])
        want[te] = Model(svm_type).train(D.from_dense(x[tr], y[tr]), prm).predict(D.from_dense(x[te], y[te]), 1000)[0]
    assert np.array_equal(got, want)
    small = n < 9000 and d < 128
    assert m.folds_together() == (folds if small else 0)


@pytest.mark.parametrize("k,d,kernel", [(2, 3, capi.RBF), (2, 16, capi.SIGMOID), (3, 17, capi.POLY), (4, 40, capi.RBF), (7, 54, capi.RBF), (9, 128, capi.LINEAR)])
def test_groups_of_rows_in_one_launch(k, d, kernel):
    """tsvm_predict_groups_dense gives, to the last bit, what a call of tsvm_predict_dec_values_dense gives for every group: groups of 1, 63, 64, 65
    and 200 rows, classes of no support vectors, of one tile of 128 columns and of several, chunks of one tile and of two."""
    rng = np.random.default_rng(10 * k + d)
    n, ldx, nc, P = 500, (d + 7) // 8 * 8, k - 1, k * (k - 1) // 2
    x = np.zeros((n, ldx))
    x[:, :d] = rng.standard_normal((n, d))
    sd = (x * x).sum(axis=1)
    stride = capi.kernel_lib().tsvm_predict_nc_stride(k, d, 0)
    assert stride >= nc
    x_d, sd_d = G.dev(x), G.dev(sd)
    args = (kernel, 0.5 / d, 0.25, 2)
    col_map, coef, chunks, tasks, rows, row_group, starts, rhos, want = [], [], [], [], [], [], [], [], []
    most = 0
    for g, m in enumerate([1, 63, 64, 65, 200]):
        n_sv = [130 if c % 3 == 0 else 0 if (c + g) % 4 == 1 else 1 + 40 * c for c in range(k)]
        col0, row0, chunk0, per = sum(map(len, col_map)), len(rows), len(chunks), 1 + g % 2
        mine, start, tile = [], [0], 0
        for c in range(k):
            tiles = (n_sv[c] + 127) // 128
            ids, w = np.zeros(128 * tiles, dtype=np.int32), np.zeros((128 * tiles, stride))
            ids[:n_sv[c]] = rng.integers(0, n, n_sv[c])
            w[:n_sv[c], :nc] = rng.standard_normal((n_sv[c], nc))
            col_map.append(ids)
            coef.append(w)
            mine += [(t, min(t + per, tile + tiles)) for t in range(tile, tile + tiles, per)]
            tile += tiles
            start.append(len(mine))
        ids = rng.integers(0, n, m).astype(np.int32)
        rho = rng.standard_normal(P)
        group_cols, group_coef = np.concatenate(col_map[-k:]), np.concatenate(coef[-k:])
        part_d = torch.full((len(mine) * m * nc,), np.nan, dtype=torch.float64, device="cuda")
        dec_d = torch.full((m, P), np.nan, dtype=torch.float64, device="cuda")
        held = [G.dev(group_cols), G.dev(group_coef), G.dev(np.array(mine, dtype=np.int32)), G.dev(np.array(start, dtype=np.int32)), G.dev(rho), G.dev(x[ids]), G.dev(sd[ids])]
        capi.call("tsvm_predict_dec_values_dense", G.ptr(x_d), ldx, d, G.ptr(sd_d), None, G.ptr(held[0]), len(group_cols), G.ptr(held[1]), G.ptr(held[2]), len(mine),
                  G.ptr(held[3]), G.ptr(held[4]), k, G.ptr(held[5]), ldx, m, G.ptr(held[6]), None, 0, *args, G.ptr(part_d), G.ptr(dec_d), G.stream())
        want.append(G.host(dec_d))
        tasks += [(row0 + r, row0 + m, chunk0 + part, part) for part in range(len(mine)) for r in range(0, m, 64)]
        chunks += [(col0 // 128 + a, col0 // 128 + b) for a, b in mine]
        rows += list(ids)
        row_group += [g] * m
        starts += start
        rhos.append(rho)
        most = max(most, len(mine))
    want = np.concatenate(want)
    assert np.isfinite(want).all() and np.abs(want).max() > 0
    cols = np.concatenate(col_map)
    held = [G.dev(cols), G.dev(np.concatenate(coef)), G.dev(np.array(chunks, dtype=np.int32)), G.dev(np.array(tasks, dtype=np.int32)), G.dev(np.array(rows, dtype=np.int32)),
            G.dev(np.array(row_group, dtype=np.int32)), G.dev(np.array(starts, dtype=np.int32)), G.dev(np.concatenate(rhos))]
    part_d = torch.full((most * len(rows) * nc,), np.nan, dtype=torch.float64, device="cuda")
    dec_d = torch.full((len(rows), P), np.nan, dtype=torch.float64, device="cuda")
    capi.call("tsvm_predict_groups_dense", G.ptr(x_d), ldx, d, G.ptr(sd_d), G.ptr(held[0]), len(cols), G.ptr(held[1]), G.ptr(held[2]), G.ptr(held[3]), len(tasks),
              G.ptr(held[4]), len(rows), G.ptr(held[5]), G.ptr(held[6]), G.ptr(held[7]), k, *args, G.ptr(part_d), G.ptr(dec_d), G.stream())
    assert np.array_equal(G.host(dec_d), want)


@pytest.mark.parametrize("k,d,hot,kernel", [(2, 1, 0, capi.RBF), (2, 32, 0, capi.RBF), (3, 33, 0, capi.POLY), (4, 60, 0, capi.SIGMOID), (9, 127, 0, capi.LINEAR),
                                            (7, 5, 40, capi.RBF), (2, 12, 64, capi.LINEAR), (10, 4, 0, capi.RBF), (2, 150, 0, capi.RBF)])
def test_requests_of_a_few_rows(k, d, hot, kernel):
    """A few rows in one launch against the same rows as part of a batch on the device, which takes the kernels for many whatever its size: the
    same bits, whatever of the batch's rows a request asks for; ten classes and 150 columns take the other route."""
    rng = np.random.default_rng(1000 * k + d)
    x, y = _blobs(rng, k, 260 // k + 20, d, one_hot=hot)
    xt, _ = _blobs(np.random.default_rng(2000 * k + d), k, 100 // k, d, one_hot=hot)
    xt[3] = 0.0
    gm = Model(0).train(D.from_dense(x, y), make_param(svm_type=0, kernel_type=kernel, gamma=0.5 / d, coef0=0.1, degree=2, C=3.0))
    lab, dec = gm.predict(Dataset(D.from_dense(xt, np.zeros(len(xt)))).to_device())
    for first, m in [(0, 1), (3, 1), (0, 2), (5, 3), (1, 4), (2, 5), (0, 7), (1, 8), (0, 9), (7, 15), (4, 16), (0, 17)]:
        l, v = gm.predict(D.from_dense(xt[first:first + m], np.zeros(m)))
        assert np.array_equal(v, dec[first:first + m]) and np.array_equal(l, lab[first:first + m]), (first, m)


@pytest.mark.parametrize("kernel", [capi.RBF, capi.POLY, capi.SIGMOID, capi.LINEAR])
@pytest.mark.parametrize("k,d,hot", [(2, 1, 0), (2, 33, 0), (3, 16, 0), (4, 128, 0), (5, 100, 64), (7, 128, 64), (9, 60, 0), (8, 31, 33)])
def test_few_rows_kernel(k, d, hot, kernel):
    """tsvm_predict_few_rows' sums per 128 support vectors are those that tsvm_predict_dec_values_dense leaves, to the last bit: rows among
    the launch's arguments, in both sizes of these, and read from page-locked memory; up to 192 columns, the last `hot` of them indicators;
    classes of no support vectors, of one tile and of several."""
    rng = np.random.default_rng(100 * k + d + kernel)
    n, all_d, nc = 600, d + hot, k - 1
    ldx = (all_d + 7) // 8 * 8

    def rows_of(count):
        x = np.zeros((count, ldx))
        x[:, :d] = rng.standard_normal((count, d)).astype(np.float32)
        if hot:
            for _ in range(3):
                x[np.arange(count), d + rng.integers(0, hot, count)] = 1
        return x

    sv = rows_of(n)
    n_sv = [0 if k > 2 and c == 1 else 1 + (97 * c) % 250 for c in range(k)]
    stride = capi.kernel_lib().tsvm_predict_nc_stride(k, d, 1 if hot else 0)
    assert stride >= nc
    cols, coefs, tiles = [], [], 0
    chunks, starts = [], [0]
    for c in range(k):
        t = (n_sv[c] + 127) // 128
        ids, w = np.zeros(128 * t, dtype=np.int32), np.zeros((128 * t, stride))
        ids[:n_sv[c]] = rng.integers(0, n, n_sv[c])
        w[:n_sv[c], :nc] = rng.standard_normal((n_sv[c], nc))
        cols.append(ids)
        coefs.append(w)
        chunks += [(i, i + 1) for i in range(tiles, tiles + t)]
        tiles += t
        starts.append(tiles)
    sv_d, sd_d, map_d, coef_d = G.dev(sv), G.dev((sv * sv).sum(axis=1)), G.dev(np.concatenate(cols)), G.dev(np.concatenate(coefs))
    chunk_d, start_d, rho_d = G.dev(np.array(chunks, dtype=np.int32)), G.dev(np.array(starts, dtype=np.int32)), torch.zeros(k * nc // 2, dtype=torch.float64, device="cuda")

    def masks_of(x_d, count):
        masks, most = torch.zeros(count, dtype=torch.int64, device="cuda"), torch.zeros(1, dtype=torch.int32, device="cuda")
        capi.call("tsvm_indicator_masks", G.ptr(x_d), ldx, count, d, hot, G.ptr(masks), G.ptr(most), G.stream())
        return masks, int(G.host(most)[0])

    mask_sv, ones = masks_of(sv_d, n) if hot else (None, 0)
    args = (kernel, 0.5 / d, 0.1, 3)
    for m in (1, 2, 3, 4, 5, 9, 16, 61):
        a = rows_of(m)
        if m > 2: a[2] = 0.0
        if m > 4: a[4, :d] = (a[4, :d] * 1e-40).astype(np.float32)   # floats below the smallest normal one
        a_d, asd = G.dev(a), (a * a).sum(axis=1)
        asd_d = G.dev(asd)
        mask_a = masks_of(a_d, m)[0] if hot else None
        part = torch.full((tiles * m * nc,), np.nan, dtype=torch.float64, device="cuda")
        dec = torch.empty(m * k * nc // 2, dtype=torch.float64, device="cuda")
        capi.call("tsvm_predict_dec_values_dense", G.ptr(sv_d), ldx, d, G.ptr(sd_d), G.ptr(mask_sv), G.ptr(map_d), 128 * tiles, G.ptr(coef_d), G.ptr(chunk_d), tiles,
                  G.ptr(start_d), G.ptr(rho_d), k, G.ptr(a_d), ldx, m, G.ptr(asd_d), G.ptr(mask_a), ones, *args, G.ptr(part), G.ptr(dec), G.stream())
        size = capi.kernel_lib().tsvm_predict_few_rows_bytes(m, all_d)
        values = (m * all_d + 1) // 2 * 2
        assert size == 4 * values + 8 * m
        request = torch.zeros(size, dtype=torch.uint8).pin_memory()
        request.numpy()[:4 * m * all_d] = np.ascontiguousarray(a[:, :all_d].astype(np.float32)).view(np.uint8).ravel()
        request.numpy()[4 * values:] = asd.view(np.uint8)
        few = torch.full((tiles * m * nc,), -7.0, dtype=torch.float64, device="cuda")
        capi.call("tsvm_predict_few_rows", G.ptr(sv_d), ldx, all_d, G.ptr(sd_d), G.ptr(map_d), 128 * tiles, G.ptr(coef_d), stride, nc, request.data_ptr(),
                  request.data_ptr(), m, *args, G.ptr(few), G.stream())
        assert np.array_equal(G.host(few), G.host(part)), m
        assert np.isfinite(G.host(part)).all() and np.abs(G.host(part)).max() > 0


def test_requests_of_a_few_rows_that_are_not_plain_floats():
    """Values that are no floats, infinite ones, and columns that no support vector has: what the kernels for many rows give."""
    rng = np.random.default_rng(5)
    x, y = _blobs(rng, 2, 150, 6)
    gm = Model(0).train(D.from_dense(x, y), make_param(svm_type=0, kernel_type=2, gamma=0.1, C=3.0))
    rows = np.concatenate([x[:40].astype(np.float64), 3.0 * rng.standard_normal((40, 6))])
    rows[1, 2], rows[2, 0] = 0.1, np.inf
    xt = np.zeros((80, 9))
    xt[:, :6], xt[5, 8], xt[7, 7] = rows, 2.5, 1e-3
    ptr, col = np.arange(81, dtype=np.int64) * 9, np.tile(np.arange(1, 10, dtype=np.int32), 80)
    _, dec = gm.predict(D.CsrData(ptr, col, xt.reshape(-1), np.zeros(80)))   # (a value that is no float: the kernels for many rows)
    for first, m in [(0, 1), (1, 1), (2, 1), (0, 8), (3, 5), (41, 3), (70, 10)]:
        _, v = gm.predict(D.CsrData(ptr[:m + 1], col[:9 * m], xt[first:first + m].reshape(-1).copy(), np.zeros(m)))
        assert np.array_equal(v, dec[first:first + m], equal_nan=True), (first, m)
