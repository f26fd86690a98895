"""Whole solves of small problems in one kernel (csrc/smo_small.hip) against the CPU oracle, at the edges of its variants:
256, 512 and 1,024 slots (a class takes its instances rounded up to four), one instance, the first size that goes the other way,
repeated instances (ties decided by the working-set position), both element types, and several class pairs from one
kernel matrix.  Same trajectory, hence the tolerances of the model tests."""
import numpy as np
import pytest

from thundersvm_amd import data as D
from thundersvm_amd.model import Dataset, Model, make_param

import oracle_lib as O
import test_gpu_models as T

pytestmark = pytest.mark.gpu


def _rows(n, seed, ties):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, 6)).astype(np.float32)
    if ties:
        x[n // 2:] = x[:n - n // 2]
        x = np.round(x)
    return x, rng


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("svm_type,kernel_type", [(0, 2), (0, 0), (1, 2)])
@pytest.mark.parametrize("n_pos,n_neg", [(1, 1), (3, 5), (1, 252), (4, 252), (5, 249), (256, 256), (253, 257), (510, 511), (509, 512), (511, 513)])
def test_two_classes(n_pos, n_neg, svm_type, kernel_type, ties):
    n = n_pos + n_neg
    x, rng = _rows(n, n, ties)
    y = np.array([1.0] * n_pos + [0.0] * n_neg)
    order = rng.permutation(n)
    x[:, 0] += y - 0.5
    d = D.from_dense(x[order], y[order])
    nu = 0.5 * min(n_pos, n_neg) / n
    T._compare(d, d, make_param(svm_type=svm_type, kernel_type=kernel_type, gamma=0.2, C=3.0, nu=nu, max_iter=40), trace=0)


@pytest.mark.parametrize("ties", [False, True])
@pytest.mark.parametrize("svm_type,kernel_type", [(2, 2), (3, 2), (3, 0), (4, 2)])
@pytest.mark.parametrize("n", [1, 2, 63, 128, 129, 256, 257, 510, 512, 513])
def test_one_class_and_regression(n, svm_type, kernel_type, ties):
    x, rng = _rows(n, 1000 + n, ties)
    d = D.from_dense(x, np.sin(x[:, 0]))
    T._compare(d, d, make_param(svm_type=svm_type, kernel_type=kernel_type, gamma=0.2, C=3.0, nu=0.3, p=0.05, max_iter=40), trace=0)


@pytest.mark.parametrize("n", [257, 300, 512, 513, 900])
@pytest.mark.parametrize("what", ["almost repeated", "a few repeated", "a near zero", "all scores alike"])
def test_scores_that_a_float_cannot_tell_apart(n, what):
    """From 257 slots on the second index is chosen by scores rounded to float: where these are too close to one another, equal,
    or out of range, or where the first index is a tie, the working set's order and doubles decide as for the oracle."""
    x, rng = _rows(n, 2000 + n, False)
    gamma = 0.2
    if what == "almost repeated":
        x[n // 2:] = x[:n - n // 2] * (1 + 1e-6 * rng.standard_normal((n - n // 2, 1)))
    elif what == "a few repeated":
        twice = rng.permutation(n)[:n // 8 * 2]
        x[twice[::2]] = x[twice[1::2]]
    elif what == "a near zero":
        gamma = 1e-9
    else:
        x = (x > 0) * np.float32(1)      # 64 different instances
    y = (x[:, 0] + 0.5 * x[:, 1] * x[:, 2] > 0.1).astype(np.float64)
    flip = rng.permutation(n)[:n // 10]
    y[flip] = 1 - y[flip]
    d = D.from_dense(x, y)
    T._compare(d, d, make_param(svm_type=0, kernel_type=2, gamma=gamma, C=3.0, max_iter=40), trace=0)


@pytest.mark.parametrize("sizes", [(5, 40, 90), (300, 200, 700, 900), (8, 8, 1100)])
def test_class_pairs_from_one_matrix(sizes):
    """Small pairs side by side, in the second and third case next to pairs that are too large; the same pairs one at a time."""
    x, rng = _rows(sum(sizes), sum(sizes), False)
    y = np.repeat(np.arange(len(sizes)), sizes).astype(np.float64)
    x[:, 0] += y
    order = rng.permutation(len(y))
    d = D.from_dense(x[order], y[order])
    T._compare(d, d, make_param(gamma=0.2, C=3.0), trace=0)
    a = Model(0).train(d, make_param(gamma=0.2, C=3.0, kernel_type=0))
    b = Model(0).train(d, make_param(gamma=0.2, C=3.0, kernel_type=0, pair_lanes=1, cache_bytes=0))   # (asks for the other path)
    assert np.array_equal(a.coef, b.coef) and np.array_equal(a.rho, b.rho) and np.array_equal(a.sv_indices, b.sv_indices)


@pytest.mark.parametrize("svm_type,n,folds", [(0, 203, 5), (1, 120, 3), (2, 61, 4), (3, 90, 3), (4, 90, 3), (0, 1500, 3), (0, 12, 6)])
def test_folds_side_by_side(svm_type, n, folds):
    """Cross-validation with its folds solved together, and one fold after the other (a row budget asks for that path)."""
    x, rng = _rows(n, n + 7, False)
    # (folds are cut label by label, whatever the model: svmmodel.cpp:31-71)
    y = np.round(np.sin(x[:, 0])) if svm_type >= 3 else (x[:, 0] + 0.3 * rng.standard_normal(n) > 0).astype(np.float64) * (svm_type != 2)
    d = Dataset(D.from_dense(x, y))
    got = [Model(svm_type).cross_validation(d, make_param(svm_type=svm_type, gamma=0.2, C=3.0, nu=0.2, p=0.05, cache_bytes=c), folds)
           for c in (-1, 64 << 20)]
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("svm_type,n", [(0, 60), (0, 120), (0, 250), (0, 300), (0, 700), (3, 30), (3, 61), (3, 200), (3, 400)])
def test_infinite_C(svm_type, n):
    """A hard margin: no upper bound on alpha.  Classes that a plane parts with room to spare, and targets that the
    functions of the kernel take, so that the solution is finite; against the oracle and the path of the larger problems."""
    x, rng = _rows(n, 77 + n, False)
    y = (rng.random(n) < 0.4).astype(np.float64)
    x[:, 0] = x[:, 0] * 0.3 + np.where(y > 0, 2.0, -2.0)
    d = D.from_dense(x, y if svm_type == 0 else np.sin(x[:, 0]))
    prm = dict(svm_type=svm_type, gamma=0.05, C=np.inf, p=0.2, max_iter=40)
    gm, om, _, _ = T._compare(d, d, make_param(**prm), trace=0)
    assert np.isfinite(gm.coef).all() and gm.total_sv > 0
    alone = Model(svm_type).train(d, make_param(pair_lanes=1, cache_bytes=0, **prm))   # (asks for the other path)
    assert np.array_equal(gm.coef, alone.coef) and np.array_equal(gm.rho, alone.rho)


@pytest.mark.parametrize("weight", [0.0, -1.0])
@pytest.mark.parametrize("sizes,small", [((40, 300, 60), True), ((700, 600, 500), False), ((1500, 1100, 40), False)])
def test_class_without_room(sizes, small, weight):
    """A class weight of zero leaves a pair's working set without enough candidates: the small kernel gives such a pair back
    (beside pairs that it has solved), and the solve ends where it starts.  The third pair is not touched by it."""
    x, rng = _rows(sum(sizes), 3 * sum(sizes), False)
    y = np.repeat(np.arange(3), sizes).astype(np.float64)
    x[:, 0] += y
    d = D.from_dense(x, y)
    prm = dict(gamma=0.2, C=3.0)
    m = Model(0).train(d, make_param(weights={0: weight}, **prm), keep_binary=True)
    for k in (0, 1):
        alpha, f = m.binary(k)
        assert m.stats(k)["n_iter"] == 1 and m.stats(k)["local_iter"] == 0
        assert not alpha.any() and np.array_equal(f, np.where(np.arange(len(f)) < sizes[0], -1.0, 1.0))
    rest = Model(0).train(D.from_dense(x[sizes[0]:], y[sizes[0]:]), make_param(**prm), keep_binary=True)
    assert np.array_equal(m.binary(2)[0], rest.binary(0)[0]) and np.array_equal(m.binary(2)[1], rest.binary(0)[1])
    assert m.stats(2)["n_iter"] == rest.stats(0)["n_iter"] > 1 and m.rho[2] == rest.rho[0]
    if small:   # two classes alone: no other pair beside
        two = Model(0).train(D.from_dense(x[:sizes[0] + 20], y[:sizes[0] + 20]), make_param(weights={1: weight}, **prm), keep_binary=True)
        assert two.total_sv == 0 and not two.binary(0)[0].any()
    else:
        two = Model(0).train(D.from_dense(x[:sizes[0] + sizes[1]], y[:sizes[0] + sizes[1]]), make_param(weights={1: weight}, **prm))
        assert two.total_sv == 0


@pytest.mark.parametrize("svm_type,n,ws,C,gamma,max_iter,iters,steps", [
    (0, 300, 4, 3.0, 0.2, 600, 513, 0), (1, 300, 8, 1.0, 0.2, 600, 513, 0), (3, 150, 4, 3.0, 0.2, 600, 257, 0), (0, 900, 8, 3.0, 0.2, 300, 257, 0),
    (0, 200, 0, 1e6, 0.01, 7, 1, 600000), (3, 300, 0, 1e6, 0.02, 4, 1, 300000)])
def test_solves_of_several_launches(svm_type, n, ws, C, gamma, max_iter, iters, steps):
    """A launch ends after 256 outer iterations or 300,000 steps; the next one goes on from what it left: small working sets
    on overlapping classes, and boxes that are never reached."""
    x, rng = _rows(n, 900 + n, False)
    y = (rng.random(n) < 0.5).astype(np.float64)
    d = D.from_dense(x, y if svm_type < 2 else rng.standard_normal(n))
    gm, om, _, _ = T._compare(d, d, make_param(svm_type=svm_type, gamma=gamma, C=C, nu=0.3, p=0.05, max_iter=max_iter), ws=ws, trace=0)
    assert gm.stats(0)["n_iter"] >= iters and gm.stats(0)["local_iter"] >= steps
    assert np.array_equal(gm.binary(0)[0], om.binary(0)[0]) and np.array_equal(gm.binary(0)[1], om.binary(0)[1])


@pytest.mark.parametrize("n,seed,max_iter", [(60, 2, 6), (200, 1, 3), (200, 4, 6), (300, 4, 3), (128, 0, 3), (128, 3, 6)])
def test_alphas_that_run_away(n, seed, max_iter):
    """A sigmoid kernel that is not positive definite: steps with a negative a leave the box, alpha grows past 1e154 and the
    scores b^2/a overflow.  Still the oracle's steps, on this path and on the one of the larger problems."""
    rng = np.random.default_rng(seed)
    x = np.stack([rng.standard_normal(n), np.ones(n)], 1).astype(np.float32)
    d = D.from_dense(x, np.round(x[:, 0]))
    prm = dict(svm_type=2, kernel_type=3, gamma=0.5, coef0=0.0, nu=0.2, max_iter=max_iter)
    om = O.Model(d.ptr, d.col, d.val, d.y, T._oparam(make_param(**prm)))
    want_a, want_f = om.binary(0)
    assert 1e154 < np.abs(want_a).max() < np.inf
    for other in ({}, dict(pair_lanes=1, cache_bytes=0)):
        gm = Model(2).train(d, make_param(**prm, **other), keep_binary=True)
        a, f = gm.binary(0)
        assert gm.stats(0)["n_iter"] == om.n_iter[0] and gm.stats(0)["local_iter"] == om.local_iter[0]
        assert np.array_equal(a, want_a) and np.array_equal(f, want_f)
