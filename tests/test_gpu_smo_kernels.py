"""GPU parity: update_f, c_smo_solve, nu_smo_solve and the fused sort_f + select_working_set
through the C ABI vs the CPU oracle.  All bit-exact / index-exact."""
import numpy as np
import pytest
import torch

import gpu_util as G
import oracle_lib as O
from thundersvm_amd import capi
from thundersvm_amd.data import from_dense

pytestmark = pytest.mark.gpu


def _problem(n, d, seed, gamma=0.5):
    rng = np.random.default_rng(seed)
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    x = (rng.standard_normal((n, d)) + 0.4 * y[:, None]).astype(np.float32)
    data = from_dense(x)
    p = O.make_param(kernel_type=O.RBF, gamma=gamma, expf_mode=1)
    km = O.KernelMatrix(data.ptr, data.col, data.val, p)
    return rng, y, km


@pytest.mark.parametrize("n,ws,zero_frac", [(1, 1, 0.0), (1000, 1024, 0.5), (1537, 512, 0.0), (4099, 37, 0.9), (513, 2050, 0.3)])
@pytest.mark.parametrize("row_type", [capi.ROW_F64, capi.ROW_F32])
def test_update_f(n, ws, zero_frac, row_type):
    rng = np.random.default_rng(n + ws)
    ld = n + 3
    k = rng.random((ws + 5, ld))
    if row_type == capi.ROW_F32:
        k = k.astype(np.float32)
    k64 = k.astype(np.float64)
    ad = rng.standard_normal(ws)
    ad[rng.random(ws) < zero_frac] = 0
    f = rng.standard_normal(n)
    slots = rng.permutation(ws + 5)[:ws].astype(np.int32)
    want = O.update_f(f, ad, np.ascontiguousarray(k64[slots][:, :n]), n)
    f_d, ad_d, k_d, s_d = G.dev(f), G.dev(ad), G.dev(k), G.dev(slots)
    capi.call("tsvm_update_f", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d), row_type, G.ptr(s_d), ld, n, 1, G.stream())
    assert np.array_equal(G.host(f_d), want)
    # slots == NULL: identity
    want = O.update_f(f, ad, np.ascontiguousarray(k64[:ws, :n]), n)
    f_d = G.dev(f)
    capi.call("tsvm_update_f", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d), row_type, None, ld, n, 1, G.stream())
    assert np.array_equal(G.host(f_d), want)


@pytest.mark.parametrize("n,ld_pad,shift", [(63, 1, 0), (64, 0, 0), (16384, 0, 0), (16385, 3, 0), (16385, 2, 1), (32768, 0, 0), (32769, 3, 0),
                                            (32769, 3, 2), (65537, 7, 0), (100003, 0, 0), (262143, 1, 0)])
@pytest.mark.parametrize("ws,rows,repeat", [(1024, 1024, 1), (1024, 257, 2), (1030, 31, 5), (513, 16, 9), (64, 33, 1), (40, 0, 1)])
@pytest.mark.parametrize("row_type", [capi.ROW_F64, capi.ROW_F32])
def test_update_f_below_262144_columns(n, ld_pad, shift, ws, rows, repeat, row_type):
    """The kernel whose wavefronts take the rows in turn: one, two and four columns per thread (and one where a row's start is not
    aligned: `shift` elements off), a last group of rows that is full, short or missing, ragged columns, more copies than wavefronts."""
    if n > 40000 and (rows > 40 or repeat > 2):
        rows, ws, repeat = min(rows, 40), 64, min(repeat, 2)
    rng = np.random.default_rng(n + ws + rows)
    ld = n + ld_pad
    store = 70
    dt = np.float32 if row_type == capi.ROW_F32 else np.float64
    k_all = rng.random(shift + store * ld).astype(dt)
    k64 = k_all[shift:].reshape(store, ld)[:, :n].astype(np.float64)
    slots = rng.integers(0, store, size=ws).astype(np.int32)
    ad = np.zeros(ws)
    ad[rng.permutation(ws)[:rows]] = rng.standard_normal(rows)
    f = rng.standard_normal(n * repeat)
    # (the oracle's update on the distinct non-zero rows, in their order, copy by copy)
    at = np.flatnonzero(ad)
    want = np.concatenate([O.update_f(f[r * n:(r + 1) * n], ad[at], np.ascontiguousarray(k64[slots[at]]), n) if rows else f[r * n:(r + 1) * n]
                           for r in range(repeat)])
    f_d, ad_d, k_d, s_d = G.dev(f), G.dev(ad), G.dev(k_all), G.dev(slots)
    capi.call("tsvm_update_f", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d) + shift * k_all.itemsize, row_type, G.ptr(s_d), ld, n, repeat, G.stream())
    assert np.array_equal(G.host(f_d), want)


@pytest.mark.parametrize("n,rows", [(65, 255), (65, 256), (130, 257), (130, 1025), (200, 2111), (28672, 300), (28673, 300)])
@pytest.mark.parametrize("row_type", [capi.ROW_F64, capi.ROW_F32])
def test_update_f_wavefronts_in_turn(n, rows, row_type):
    """Every wavefront's second and later groups, a last group of one row, three chunks of the working set (one of them without a
    non-zero entry), and the line between one and two columns per thread."""
    rng = np.random.default_rng(n + rows)
    ws, ld, store = 3 * 1024, (n + 7) // 8 * 8, 50
    k = rng.random((store, ld)).astype(np.float32 if row_type == capi.ROW_F32 else np.float64)
    slots = rng.integers(0, store, size=ws).astype(np.int32)
    ad = np.zeros(ws)
    at = np.sort(np.concatenate([rng.permutation(1024)[:min(rows, 1024)], 2048 + rng.permutation(1024)[:max(min(rows, 2048) - 1024, 0)]]))
    ad[at] = rng.standard_normal(len(at))
    f = rng.standard_normal(n)
    want = O.update_f(f, ad[at], np.ascontiguousarray(k[slots[at], :n].astype(np.float64)), n)
    f_d, ad_d, k_d, s_d = G.dev(f), G.dev(ad), G.dev(k), G.dev(slots)
    capi.call("tsvm_update_f", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d), row_type, G.ptr(s_d), ld, n, 1, G.stream())
    assert np.array_equal(G.host(f_d), want)


@pytest.mark.parametrize("n,ws,ld_pad", [(300001, 64, 7), (262144, 33, 0), (270000, 40, 4)])
@pytest.mark.parametrize("row_type", [capi.ROW_F64, capi.ROW_F32])
def test_update_f_wide_and_repeated(n, ws, ld_pad, row_type):
    """Large n takes the 16-byte-load path (also with a ragged last vector); with repeat = 2 the kernel
    rows are n wide and f has 2n entries, which must equal the reference's update_f on [K K] rows."""
    rng = np.random.default_rng(n)
    ld = n + ld_pad
    k = rng.random((ws, ld))
    if row_type == capi.ROW_F32:
        k = k.astype(np.float32)
    k64 = k.astype(np.float64)[:, :n]
    ad = rng.standard_normal(ws)
    ad[::3] = 0
    f = rng.standard_normal(2 * n)
    want = O.update_f(f, ad, np.ascontiguousarray(np.concatenate([k64, k64], axis=1)), 2 * n)
    f_d, ad_d, k_d = G.dev(f), G.dev(ad), G.dev(k)
    capi.call("tsvm_update_f", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d), row_type, None, ld, n, 2, G.stream())
    assert np.array_equal(G.host(f_d), want)


@pytest.mark.parametrize("n,n_rows,batch,repeat", [(1, 1, 101, 1), (63, 31, 101, 2), (64, 32, 16, 1), (65, 33, 101, 1), (5001, 101, 101, 1),
                                                   (257, 102, 101, 2), (300, 640, 101, 1), (1000, 1010, 101, 2)])
@pytest.mark.parametrize("row_type", [capi.ROW_F64, capi.ROW_F32])
def test_update_f_in_batches(n, n_rows, batch, repeat, row_type):
    """One launch gives what one update_f per batch gives, bit for bit, on both sides of the rows it keeps on their way."""
    rng = np.random.default_rng(n + n_rows)
    ld = n + 3
    k = rng.standard_normal((n_rows, ld)).astype(np.float32 if row_type == capi.ROW_F32 else np.float64)
    coef, f = rng.standard_normal(n_rows), rng.standard_normal(n * repeat)
    want, rows = f, np.ascontiguousarray(np.tile(k[:, :n].astype(np.float64), (1, repeat)))
    for at in range(0, n_rows, batch):
        want = O.update_f(want, coef[at:at + batch], rows[at:at + batch], n * repeat)
    f_d, c_d, k_d = G.dev(f), G.dev(coef), G.dev(k)
    capi.call("tsvm_update_f_batches", G.ptr(f_d), G.ptr(c_d), n_rows, batch, G.ptr(k_d), row_type, ld, n, repeat, G.stream())
    assert np.array_equal(G.host(f_d), want)


def test_fold_ids():
    ids = np.array([0, 5, 9, 10, 19, 7], dtype=np.int32)
    out = torch.zeros(6, dtype=torch.int32, device="cuda")
    ids_d = G.dev(ids)
    capi.call("tsvm_fold_ids", G.ptr(ids_d), 6, 10, G.ptr(out), G.stream())
    assert np.array_equal(G.host(out), ids % 10)


def _solver_inputs(n, d, ws, seed, C, nu=False):
    rng, y, km = _problem(n, d, seed)
    alpha = np.zeros(n)
    # a mid-training state: some alphas at bounds, some free
    r = rng.random(n)
    alpha[r < 0.2] = C
    alpha[(r >= 0.2) & (r < 0.5)] = rng.random(int(((r >= 0.2) & (r < 0.5)).sum())) * C
    f = rng.standard_normal(n)
    ws_ids = rng.permutation(n)[:ws].astype(np.int32)
    k_rows = km.get_rows(ws_ids)
    diag = km.diag()
    return y, alpha, f, ws_ids, k_rows, diag


@pytest.mark.parametrize("n,ws,max_iter", [(300, 16, 100000), (2000, 1024, 100000), (1500, 512, 7), (700, 100, 100000), (64, 64, 0)])
def test_c_smo_solve(n, ws, max_iter):
    Cp, Cn, eps = 10.0, 4.0, 1e-3
    y, alpha, f, ws_ids, k_rows, diag = _solver_inputs(n, 12, ws, n + ws, Cn)
    a_want, ad_want, diff_want = O.c_smo_solve(y, f, alpha, ws_ids, Cp, Cn, k_rows, diag, n, eps, max_iter)
    slots = np.random.default_rng(1).permutation(ws).astype(np.int32)
    k_phys = np.empty_like(k_rows)
    k_phys[slots] = k_rows
    y_d, f_d, a_d, ws_d, k_d, s_d, dg_d = G.dev(y), G.dev(f), G.dev(alpha), G.dev(ws_ids), G.dev(k_phys), G.dev(slots), G.dev(diag)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_c_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cp, Cn, G.ptr(k_d),
              capi.ROW_F64, G.ptr(s_d), n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
    assert np.array_equal(G.host(diff_d), diff_want)
    assert np.array_equal(G.host(a_d), a_want)
    assert np.array_equal(G.host(ad_d), ad_want)
    # the same rows held as float (RBF values are float-exact): identical result
    a_d, k32_d = G.dev(alpha), G.dev(k_phys.astype(np.float32))
    assert np.array_equal(k_phys.astype(np.float32).astype(np.float64), k_phys)
    capi.call("tsvm_c_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cp, Cn, G.ptr(k32_d),
              capi.ROW_F32, G.ptr(s_d), n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
    assert np.array_equal(G.host(diff_d), diff_want)
    assert np.array_equal(G.host(a_d), a_want)
    assert np.array_equal(G.host(ad_d), ad_want)
    assert diff_want[1] > 0 or max_iter == 0 or diff_want[0] < eps


@pytest.mark.parametrize("n,ws", [(300, 16), (2000, 1024), (900, 200)])
def test_nu_smo_solve(n, ws):
    Cc, eps = 1.0, 1e-3
    y, alpha, f, ws_ids, k_rows, diag = _solver_inputs(n, 10, ws, 5 * n + ws, Cc)
    a_want, ad_want, diff_want = O.nu_smo_solve(y, f, alpha, ws_ids, Cc, k_rows, diag, n, eps, 100000)
    y_d, f_d, a_d, ws_d, k_d, dg_d = G.dev(y), G.dev(f), G.dev(alpha), G.dev(ws_ids), G.dev(k_rows), G.dev(diag)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_nu_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, G.ptr(k_d),
              capi.ROW_F64, None, n, G.ptr(dg_d), eps, G.ptr(diff_d), 100000, G.ptr(wsp), G.stream())
    assert G.host(diff_d)[0] == diff_want[0]
    assert np.array_equal(G.host(a_d), a_want)
    assert np.array_equal(G.host(ad_d), ad_want)
    # the same rows held as float: a float block inside, identical result
    a_d, k32_d = G.dev(alpha), G.dev(k_rows.astype(np.float32))
    capi.call("tsvm_nu_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, G.ptr(k32_d),
              capi.ROW_F32, None, n, G.ptr(dg_d), eps, G.ptr(diff_d), 100000, G.ptr(wsp), G.stream())
    assert G.host(diff_d)[0] == diff_want[0]
    assert np.array_equal(G.host(a_d), a_want)
    assert np.array_equal(G.host(ad_d), ad_want)


@pytest.mark.parametrize("ws", [16, 200, 300, 1024])
def test_nu_smo_solve_infinite_C(ws):
    """No upper bound on alpha: steps are bounded by alpha >= 0 and the quotient alone, for both labels."""
    n, eps = ws + 100, 1e-3
    y, alpha, f, ws_ids, k_rows, diag = _solver_inputs(n, 10, ws, 7 * n, 1.0)
    a_want, ad_want, diff_want = O.nu_smo_solve(y, f, alpha, ws_ids, np.inf, k_rows, diag, n, eps, 2000)
    assert np.isfinite(a_want).all() and (a_want >= 0).all() and a_want.max() > 1.0
    y_d, f_d, a_d, ws_d, k_d, dg_d = G.dev(y), G.dev(f), G.dev(alpha), G.dev(ws_ids), G.dev(k_rows), G.dev(diag)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_nu_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, np.inf, G.ptr(k_d),
              capi.ROW_F64, None, n, G.ptr(dg_d), eps, G.ptr(diff_d), 2000, G.ptr(wsp), G.stream())
    assert G.host(diff_d)[0] == diff_want[0]
    assert np.array_equal(G.host(a_d), a_want) and np.array_equal(G.host(ad_d), ad_want)


@pytest.mark.parametrize("ws", [2, 63, 64, 65, 128, 129, 256, 257, 512, 513, 1023, 1024])
@pytest.mark.parametrize("nu", [False, True])
@pytest.mark.parametrize("start", ["first iteration", "threshold zero"])
def test_local_solver_at_the_edges_of_its_variants(ws, nu, start):
    """Working-set sizes on both sides of every variant of the solver (one wavefront of one, two or four elements per
    thread, four wavefronts of two or four).  "first iteration": alpha = 0, f = -y and repeated instances, so that every
    extremum is a tie that the lowest index has to win, in both wavefront-wide and workgroup-wide reductions; "threshold
    zero": eps = 0 from a state without violators by more than that, where an element can violate without being a
    candidate for the second index.  Everything equals the oracle bit for bit."""
    n, Cc = ws + 37, 1.0
    y, alpha, f, ws_ids, _, _ = _solver_inputs(n, 6, ws, 3 * ws, Cc)
    rng = np.random.default_rng(ws)
    x = rng.standard_normal((n, 6)).astype(np.float32)
    x[n // 2:n // 2 + n // 4] = x[:n // 4]          # instances that occur twice: equal kernel rows, a = 0
    data = from_dense(x)
    km = O.KernelMatrix(data.ptr, data.col, data.val, O.make_param(kernel_type=O.RBF, gamma=0.5, expf_mode=1))
    k_rows, diag = km.get_rows(ws_ids), km.diag()
    eps, max_iter = 1e-3, 300
    if start == "first iteration":
        if not nu:
            alpha, f = np.zeros(n), -y.astype(np.float64)
        else:
            f = np.where(rng.random(n) < 0.5, 0.25, -0.5)
    else:
        eps, max_iter = 0.0, 40
        f = np.round(f)
    solve = O.nu_smo_solve if nu else O.c_smo_solve
    args = (Cc,) if nu else (Cc, Cc)
    a_want, ad_want, diff_want = solve(y, f, alpha, ws_ids, *args, k_rows, diag, n, eps, max_iter)
    y_d, f_d, ws_d, dg_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag)
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    for row_type, rows in ((capi.ROW_F64, k_rows), (capi.ROW_F32, k_rows.astype(np.float32))):
        a_d, k_d = G.dev(alpha), G.dev(rows)
        ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
        diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
        capi.call("tsvm_nu_smo_solve" if nu else "tsvm_c_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws,
                  *args, G.ptr(k_d), row_type, None, n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
        assert np.array_equal(G.host(diff_d), diff_want) if not nu else G.host(diff_d)[0] == diff_want[0]
        assert np.array_equal(G.host(a_d), a_want, equal_nan=True)
        assert np.array_equal(G.host(ad_d), ad_want, equal_nan=True)


@pytest.mark.parametrize("ws", [257, 512, 513, 1024])
@pytest.mark.parametrize("scores", ["apart by 1e-9", "apart by 1e-6", "pairs of equals", "negative a", "f times 1e-25", "f times 1e15", "some a are 0"])
def test_c_smo_solve_with_scores_that_a_float_cannot_tell_apart(ws, scores):
    """The four-wavefront solver ranks b^2/a in float and falls back to doubles where that does not decide: scores closer
    together than a float resolves, equal ones, none that is positive, out of a float's range, infinite.  The same steps as
    the oracle's, bit for bit."""
    rng = np.random.default_rng(ws + len(scores))
    n, Cc, eps, max_iter = ws + 5, 2.0, 1e-3, 60
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    b = rng.random((n, n))
    k = 0.2 * (b + b.T)
    f = -y + 0.01 * rng.standard_normal(n)
    alpha = np.zeros(n)
    if scores.startswith("apart by"):
        small = float(scores.split()[-1])
        k, f = small * k, -y * (1 + small * rng.random(n))
    elif scores == "pairs of equals":
        k[1::2][: n // 2] = k[0::2][: n // 2]
        k[:, 1::2][:, : n // 2] = k[:, 0::2][:, : n // 2]
        f[1::2], y[1::2] = f[0::2][: n // 2], y[0::2][: n // 2]
    elif scores == "negative a":
        k = 4.0 * k
    elif scores.startswith("f times"):
        f = f * float(scores.split()[-1])
        eps = 1e-30 if scores.endswith("-25") else eps
    else:
        same = rng.random((n, n)) < 0.05
        k[same | same.T] = 1.0
    np.fill_diagonal(k, 1.0)
    ws_ids = rng.permutation(n)[:ws].astype(np.int32)
    k_rows, diag = np.ascontiguousarray(k[ws_ids]), np.ones(n)
    a_want, ad_want, diff_want = O.c_smo_solve(y, f, alpha, ws_ids, Cc, Cc, k_rows, diag, n, eps, max_iter)
    y_d, f_d, ws_d, dg_d, a_d, k_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag), G.dev(alpha), G.dev(k_rows)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_c_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc, G.ptr(k_d), capi.ROW_F64, None,
              n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
    assert np.array_equal(G.host(diff_d), diff_want)
    assert np.array_equal(G.host(a_d), a_want, equal_nan=True)
    assert np.array_equal(G.host(ad_d), ad_want, equal_nan=True)


@pytest.mark.parametrize("ws", [257, 512, 513, 1024])
@pytest.mark.parametrize("scores", ["apart by 1e-9", "pairs of equals", "sides alike", "negative a", "f times 1e25", "f times 1e-25", "a full side",
                                    "a = 0 now and then", "row of the other side"])
def test_nu_smo_solve_with_scores_that_a_float_cannot_tell_apart(ws, scores):
    """As for the C variant, and over two sides: equal scores of both, a side that has no first index, and a score's a that is
    row ip's while the step's is row in's.  The same steps as the oracle's, bit for bit."""
    rng = np.random.default_rng(ws + len(scores))
    n, Cc, eps, max_iter = ws + 6, 2.0, 1e-3, 60
    y = np.where(np.arange(n) % 2 == 0, 1, -1).astype(np.int32)
    b = rng.random((n, n))
    k = 0.2 * (b + b.T)
    f = 0.3 * rng.standard_normal(n)
    alpha = np.where(rng.random(n) < 0.7, Cc * rng.random(n), 0.0)
    if scores.startswith("apart by"):
        small = float(scores.split()[-1])
        k, f = small * k, np.where(rng.random(n) < 0.5, 1.0, -1.0) * (1 + small * rng.random(n))
    elif scores in ("pairs of equals", "sides alike"):
        apart = 1 if scores == "sides alike" else 2     # (neighbours have different labels)
        first = np.flatnonzero(np.arange(n) % (2 * apart) < apart)[: n // (2 * apart)]
        first = first[first + apart < n]
        k[first + apart] = k[first]
        k[:, first + apart] = k[:, first]
        f[first + apart], alpha[first + apart] = f[first], alpha[first]
    elif scores == "negative a":
        k = 4.0 * k
    elif scores.startswith("f times"):
        f = f * float(scores.split()[-1])
        eps = 1e-30 if scores.endswith("-25") else eps
    elif scores == "a full side":
        alpha[y > 0] = Cc
    elif scores == "a = 0 now and then":
        same = rng.random((n, n)) < 0.05
        k[same | same.T] = 1.0
    np.fill_diagonal(k, 1.0)
    if scores == "row of the other side":
        k = k * np.where(y > 0, 1.0, 0.01)[:, None] * np.where(y > 0, 1.0, 0.01)[None, :]
    ws_ids = rng.permutation(n)[:ws].astype(np.int32)
    k_rows, diag = np.ascontiguousarray(k[ws_ids]), np.ascontiguousarray(np.diag(k))
    a_want, ad_want, diff_want = O.nu_smo_solve(y, f, alpha, ws_ids, Cc, k_rows, diag, n, eps, max_iter)
    y_d, f_d, ws_d, dg_d, a_d, k_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag), G.dev(alpha), G.dev(k_rows)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_nu_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, G.ptr(k_d), capi.ROW_F64, None,
              n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
    assert G.host(diff_d)[0] == diff_want[0]
    assert np.array_equal(G.host(a_d), a_want, equal_nan=True)
    assert np.array_equal(G.host(ad_d), ad_want, equal_nan=True)


@pytest.mark.parametrize("ws", [257, 512, 513, 1024])
@pytest.mark.parametrize("diagonal", ["2^126.5", "2^130", "2^-342", "0"])
def test_c_smo_solve_with_diagonals_out_of_float_range(ws, diagonal):
    """A few instances whose K_ii + K_tt - 2 K_it is no normal float, or has no normal float as its reciprocal, and whose f
    makes them the best second index all the same: the same steps as the oracle's, bit for bit."""
    rng = np.random.default_rng(ws + len(diagonal))
    n, Cc, eps, max_iter = ws + 5, 2.0, 1e-30, 60
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    b = rng.random((n, n))
    k = 0.2 * (b + b.T)
    f = -y + 0.01 * rng.standard_normal(n)
    np.fill_diagonal(k, 1.0)
    ws_ids = rng.permutation(n)[:ws].astype(np.int32)
    odd = ws_ids[rng.permutation(ws)[:4]]
    k[odd], k[:, odd] = 0.0, 0.0
    k[odd, odd] = 0.0 if diagonal == "0" else 2.0 ** float(diagonal[2:])
    if diagonal in ("2^126.5", "2^130"):           # scores of 8 and less by halves, the others' are below 4
        y[odd], f[odd] = -1, np.sqrt(np.array([8.0, 6.0, 5.0, 4.5]) * k[odd, odd])
    else:                                          # up is -1e-60: the odd instances' b is 1e-50, the others' 1e-3, eps 1e-30
        f = 1e-3 * (1.0 + rng.random(n))
        y[odd], f[odd] = [1, -1, -1, -1], [-1e-60, 1e-50, 2e-50, 3e-50]
    k_rows, diag = np.ascontiguousarray(k[ws_ids]), np.ascontiguousarray(np.diag(k))
    alpha = np.zeros(n)
    a_want, ad_want, diff_want = O.c_smo_solve(y, f, alpha, ws_ids, Cc, Cc, k_rows, diag, n, eps, max_iter)
    assert np.count_nonzero(a_want[odd]) >= 2 and diff_want[1] > 1
    y_d, f_d, ws_d, dg_d, a_d, k_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag), G.dev(alpha), G.dev(k_rows)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_c_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc, G.ptr(k_d), capi.ROW_F64, None,
              n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
    assert np.array_equal(G.host(diff_d), diff_want)
    assert np.array_equal(G.host(a_d), a_want, equal_nan=True)
    assert np.array_equal(G.host(ad_d), ad_want, equal_nan=True)


@pytest.mark.parametrize("nu", [False, True])
@pytest.mark.parametrize("ws", [2, 64, 100, 256, 257, 512, 1024])
@pytest.mark.parametrize("what", ["scores from 2^1023 on", "infinite scores", "some infinite scores", "NaN rows", "NaN f", "infinite f"])
def test_local_solvers_beyond_the_finite(ws, nu, what):
    """Scores that overflow (a kernel that is not positive definite, alphas that have run away) and values that are no
    numbers: a violating element without a finite score is no candidate, and the second index stays 0 without any, as for
    the oracle.  Bit for bit, wherever the alphas went."""
    if what == "infinite f" and ws == 2:
        pytest.skip("the only element of a side with an infinite f: the gap is inf - inf, which is nobody's threshold")
    rng = np.random.default_rng(ws + len(what))
    n, Cc, eps, max_iter = ws + 5, 2.0, 1e-3, 40
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    y[:2] = [1, -1]
    b = rng.random((n, n))
    k = 0.2 * (b + b.T)
    f = -y + 0.01 * rng.standard_normal(n)
    alpha = np.where(rng.random(n) < 0.3, rng.random(n), 0.0)
    if "scores" in what:
        if what.startswith("some"):
            k[: n // 2], k[:, : n // 2] = 4.0 * k[: n // 2], 4.0 * k[:, : n // 2]   # (positive a, too)
        else:
            k = k + 1.1                                                             # (negative a everywhere)
        f = f * 2.0 ** (510.8 if "2^1023" in what else 520)
    np.fill_diagonal(k, 1.0)
    odd = rng.permutation(n)[: max(1, n // 50)]
    if what == "NaN rows":
        k[odd], k[:, odd] = np.nan, np.nan
    elif what == "NaN f":
        f[odd] = np.nan
    elif what == "infinite f":
        f[odd], alpha[odd] = np.where(y[odd] > 0, -np.inf, np.inf), 0.0   # (on one side each: a gap of inf - inf is no number)
    ws_ids = rng.permutation(n)[:ws].astype(np.int32)
    k_rows, diag = np.ascontiguousarray(k[ws_ids]), np.ascontiguousarray(np.diag(k))
    solve, args = (O.nu_smo_solve, (Cc,)) if nu else (O.c_smo_solve, (Cc, Cc))
    a_want, ad_want, diff_want = solve(y, f, alpha, ws_ids, *args, k_rows, diag, n, eps, max_iter)
    y_d, f_d, ws_d, dg_d, a_d, k_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag), G.dev(alpha), G.dev(k_rows)
    ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
    diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_smo_solve_workspace(ws), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_nu_smo_solve" if nu else "tsvm_c_smo_solve", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, *args,
              G.ptr(k_d), capi.ROW_F64, None, n, G.ptr(dg_d), eps, G.ptr(diff_d), max_iter, G.ptr(wsp), G.stream())
    got = G.host(diff_d)
    assert np.array_equal(got if not nu else got[:1], diff_want if not nu else diff_want[:1], equal_nan=True)
    assert np.array_equal(G.host(a_d), a_want, equal_nan=True)
    assert np.array_equal(G.host(ad_d), ad_want, equal_nan=True)


@pytest.mark.parametrize("nu", [False, True])
@pytest.mark.parametrize("n,ws", [(300, 16), (2000, 1024), (900, 200)])
def test_smo_solve_block_on_a_chosen_xcd(n, ws, nu):
    """The block solvers launched as eight workgroups of which one is elected (tsvm_*_smo_solve_block_on_xcd): the same
    result as the one-workgroup launch, for every target XCD and launch after launch on one gate.  On an ordinary
    stream the eight workgroups land wherever there is room, so some targets have a workgroup on them and others
    do not: both ways of being elected (being on the target, being the last to arrive) are exercised, and exactly one
    workgroup solves either way (two would apply every step twice)."""
    Cc, eps = 1.0, 1e-3
    y, alpha, f, ws_ids, k_rows, diag = _solver_inputs(n, 10, ws, 7 * n + ws, Cc, nu)
    if nu:
        a_want, ad_want, diff_want = O.nu_smo_solve(y, f, alpha, ws_ids, Cc, k_rows, diag, n, eps, 100000)
    else:
        a_want, ad_want, diff_want = O.c_smo_solve(y, f, alpha, ws_ids, Cc, Cc, k_rows, diag, n, eps, 100000)
    ldk = capi.kernel_lib().tsvm_smo_solve_block_ld(ws)
    block = np.zeros((ws, ldk))
    block[:, :ws] = k_rows[:, ws_ids]
    y_d, f_d, ws_d, b_d, dg_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(block), G.dev(diag)
    assert np.array_equal(block.astype(np.float32).astype(np.float64), block)     # RBF values: a float block holds the same numbers
    b32_d = G.dev(block.astype(np.float32))
    gate = torch.zeros(4, dtype=torch.int32, device="cuda")
    seen = set()
    for epoch, xcd in enumerate([0, 3, 7, 5, 1, 2, 6, 4, 0, 0], start=1):
        a_d = G.dev(alpha)
        ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
        diff_d = torch.zeros(2, dtype=torch.float64, device="cuda")
        blk, bt = (b_d, capi.ROW_F64) if epoch % 2 else (b32_d, capi.ROW_F32)
        if nu:
            capi.call("tsvm_nu_smo_solve_block_on_xcd", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc,
                      G.ptr(blk), bt, G.ptr(dg_d), eps, G.ptr(diff_d), 100000, G.ptr(gate), epoch, xcd, G.stream())
        else:
            capi.call("tsvm_c_smo_solve_block_on_xcd", G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc,
                      G.ptr(blk), bt, G.ptr(dg_d), eps, G.ptr(diff_d), 100000, G.ptr(gate), epoch, xcd, G.stream())
        g = G.host(gate)
        assert g[0] == epoch and g[1] == 8 * epoch and 0 <= g[2] < 8
        seen.add(int(g[2]))
        assert G.host(diff_d)[0] == diff_want[0]
        assert np.array_equal(G.host(a_d), a_want)
        assert np.array_equal(G.host(ad_d), ad_want)
    # bad arguments are refused
    lib = capi.kernel_lib()
    assert lib.tsvm_c_smo_solve_block_on_xcd(G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc, G.ptr(b_d),
                                             capi.ROW_F64, G.ptr(dg_d), eps, G.ptr(diff_d), 10, G.ptr(gate), 0, 0, G.stream()) != 0
    assert lib.tsvm_c_smo_solve_block_on_xcd(G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc, G.ptr(b_d),
                                             capi.ROW_F64, G.ptr(dg_d), eps, G.ptr(diff_d), 10, G.ptr(gate), 1, 8, G.stream()) != 0
    assert lib.tsvm_c_smo_solve_block_on_xcd(G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc, G.ptr(b_d),
                                             7, G.ptr(dg_d), eps, G.ptr(diff_d), 10, G.ptr(gate), 1, 0, G.stream()) != 0


@pytest.mark.parametrize("nu", [False, True])
@pytest.mark.parametrize("n,ws", [(300, 16), (300, 130), (900, 200), (900, 300), (2000, 1024)])
def test_smo_solve_block_on_a_chosen_cu(n, ws, nu):
    """The block solvers launched on every CU of which one solves (tsvm_*_smo_solve_block_on_cu): the same result as ever for CUs
    that the launch visits and for one that does not exist, where the last workgroup to arrive solves; exactly one does."""
    Cc, eps = 1.0, 1e-3
    y, alpha, f, ws_ids, k_rows, diag = _solver_inputs(n, 10, ws, 9 * n + ws, Cc, nu)
    if nu:
        a_want, ad_want, diff_want = O.nu_smo_solve(y, f, alpha, ws_ids, Cc, k_rows, diag, n, eps, 100000)
    else:
        a_want, ad_want, diff_want = O.c_smo_solve(y, f, alpha, ws_ids, Cc, Cc, k_rows, diag, n, eps, 100000)
    block = np.zeros((ws, capi.kernel_lib().tsvm_smo_solve_block_ld(ws)))
    block[:, :ws] = k_rows[:, ws_ids]
    y_d, f_d, ws_d, dg_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag)
    blocks = [(G.dev(block), capi.ROW_F64), (G.dev(block.astype(np.float32)), capi.ROW_F32)]
    where_d = torch.zeros(256, dtype=torch.int32, device="cuda")
    capi.call("tsvm_where", G.ptr(where_d), 256, G.stream())
    where = G.host(where_d)
    assert set(where >> 16) == set(range(8))
    gate = torch.zeros(4, dtype=torch.int32, device="cuda")
    targets = [(int(where[b]) >> 16, int(where[b]) & 0xffff) for b in (0, 9, 130, 255)] + [(0, 0x7fff), (7, 0x7fff), (0, int(where[8]) & 0xffff)]
    for epoch, (xcd, cu) in enumerate(targets, start=1):
        a_d = G.dev(alpha)
        ad_d = torch.zeros(ws, dtype=torch.float64, device="cuda")
        diff_d = torch.zeros(3, dtype=torch.float64, device="cuda")
        blk, bt = blocks[epoch % 2]
        args = (G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws) + ((Cc,) if nu else (Cc, Cc))
        capi.call("tsvm_nu_smo_solve_block_on_cu" if nu else "tsvm_c_smo_solve_block_on_cu", *args, G.ptr(blk), bt, G.ptr(dg_d), eps, G.ptr(diff_d),
                  100000, G.ptr(gate), epoch, xcd, cu, G.stream())
        g = G.host(gate)
        assert g[0] == epoch and g[1] == 256 * epoch and 0 <= g[2] < 8
        assert G.host(diff_d)[0] == diff_want[0] and G.host(diff_d).view(np.int32)[4] == epoch
        assert np.array_equal(G.host(a_d), a_want)
        assert np.array_equal(G.host(ad_d), ad_want)
    with pytest.raises(capi.TsvmError):
        capi.call("tsvm_nu_smo_solve_block_on_cu" if nu else "tsvm_c_smo_solve_block_on_cu", *args, G.ptr(blk), bt, G.ptr(dg_d), eps, G.ptr(diff_d),
                  100000, G.ptr(gate), 1, 0, -1, G.stream())


@pytest.mark.parametrize("on", ["xcd", "cu"])
def test_arrivals_beyond_the_largest_int(on):
    """Somebody solves when the gate's count of workgroups has passed 2^31: here the last to arrive, as nobody is on the CU that is asked for
    (a die that is asked for has a workgroup: there only the count goes on)."""
    n, ws, Cc, eps = 300, 130, 1.0, 1e-3
    y, alpha, f, ws_ids, k_rows, diag = _solver_inputs(n, 10, ws, 7, Cc, False)
    a_want, ad_want, diff_want = O.c_smo_solve(y, f, alpha, ws_ids, Cc, Cc, k_rows, diag, n, eps, 100000)
    block = np.zeros((ws, capi.kernel_lib().tsvm_smo_solve_block_ld(ws)))
    block[:, :ws] = k_rows[:, ws_ids]
    y_d, f_d, ws_d, dg_d, blk_d = G.dev(y), G.dev(f), G.dev(ws_ids), G.dev(diag), G.dev(block)
    gate = G.dev(np.array([0, -2 ** 31, 0, 0], dtype=np.int32))
    for epoch in (1, 2):
        a_d = G.dev(alpha)
        ad_d, diff_d = torch.zeros(ws, dtype=torch.float64, device="cuda"), torch.zeros(3, dtype=torch.float64, device="cuda")
        where = (0,) if on == "xcd" else (0, 0x7fff)
        capi.call("tsvm_c_smo_solve_block_on_" + on, G.ptr(y_d), G.ptr(f_d), G.ptr(a_d), G.ptr(ad_d), G.ptr(ws_d), ws, Cc, Cc, G.ptr(blk_d), capi.ROW_F64,
                  G.ptr(dg_d), eps, G.ptr(diff_d), 100000, G.ptr(gate), epoch, *where, G.stream())
        assert G.host(gate)[0] == epoch and G.host(diff_d)[0] == diff_want[0]
        assert np.array_equal(G.host(a_d), a_want) and np.array_equal(G.host(ad_d), ad_want)


def _select_case(n, n_select, n_marked, seed, tie_mode, nu):
    rng = np.random.default_rng(seed)
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    C = 2.0
    alpha = np.zeros(n)
    r = rng.random(n)
    alpha[r < 0.25] = C
    free = (r >= 0.25) & (r < 0.5)
    alpha[free] = rng.random(int(free.sum())) * C
    if tie_mode == 0:
        f = rng.standard_normal(n)
    elif tie_mode == 1:
        f = -y.astype(np.float64)               # the initial state of C-SVC: massive ties
    else:
        f = np.round(rng.standard_normal(n), 1)  # few distinct values, signed zeros
        f[rng.random(n) < 0.1] = -0.0
    marked = rng.permutation(n)[:n_marked].astype(np.int32)
    return f, y, alpha, C, marked


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("tie_mode", [0, 1, 2])
@pytest.mark.parametrize("n,n_select,n_marked", [(2, 2, 0), (150, 128, 0), (150, 64, 64), (3200, 1024, 0), (3200, 512, 512),
                                                 (100000, 512, 512), (70001, 1024, 0), (1100, 1024, 0), (1030, 512, 512),
                                                 (1200000, 512, 512)])
def test_select_working_set(n, n_select, n_marked, tie_mode, nu):
    f, y, alpha, C, marked = _select_case(n, n_select, n_marked, n + n_select + tie_mode, tie_mode, nu)
    want = O.select_working_set(f, y, alpha, C, C, marked, n_select, nu=bool(nu))
    f_d, y_d, a_d, m_d = G.dev(f), G.dev(y), G.dev(alpha), G.dev(marked)
    out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_select_working_set", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, G.ptr(m_d) if n_marked else None,
              n_marked, G.ptr(out_d), n_select, nu, G.ptr(wsp), G.stream())
    got = G.host(out_d)
    assert np.array_equal(got, want), "first mismatch at %s" % np.flatnonzero(got != want)[:5]


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("tie_mode", [0, 2])
@pytest.mark.parametrize("state", ["all free", "few above 0", "few below C"])
@pytest.mark.parametrize("n", [9, 65, 129, 513, 1025, 4001])
def test_selection_whose_sides_meet_or_run_dry(n, state, tie_mode, nu):
    """Almost every candidate is wanted: the two ends of a pair of sides meet ("all free"), or one side has a few entries
    and the other goes on alone, with those that the first has not taken."""
    rng = np.random.default_rng(n + tie_mode)
    f, y, _, C, _ = _select_case(n, 1, 0, n, tie_mode, nu)
    few = rng.random(n) < 8.0 / n
    alpha = {"all free": 0.25 + rng.random(n), "few above 0": np.where(few, 0.5 + rng.random(n), 0.0),
             "few below C": np.where(few, 0.5 + rng.random(n), C)}[state]
    alpha = np.where(few & (rng.random(n) < 0.5), C - alpha, alpha)
    n_select = min(1024, n * 3 // 4 // 4 * 4)
    want = O.select_working_set(f, y, alpha, C, C, np.zeros(0, dtype=np.int32), n_select, nu=bool(nu))
    f_d, y_d, a_d = G.dev(f), G.dev(y), G.dev(alpha)
    out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_select_working_set", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, None, 0, G.ptr(out_d), n_select, nu, G.ptr(wsp),
              G.stream())
    got = G.host(out_d)
    assert np.array_equal(got, want), "first mismatch at %s" % np.flatnonzero(got != want)[:5]


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("tie_mode", [0, 1, 2])
def test_longer_selection_starts_with_the_shorter_one(tie_mode, nu):
    """Asking for more ids appends runners-up: the first n_select ids do not change."""
    n, n_marked = 50000, 512
    f, y, alpha, C, marked = _select_case(n, 512, n_marked, 99 + tie_mode, tie_mode, nu)
    f_d, y_d, a_d, m_d = G.dev(f), G.dev(y), G.dev(alpha), G.dev(marked)
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    outs = []
    for n_select in (512, 768):
        out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        capi.call("tsvm_select_working_set", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, G.ptr(m_d), n_marked, G.ptr(out_d),
                  n_select, nu, G.ptr(wsp), G.stream())
        outs.append(G.host(out_d))
    assert np.array_equal(outs[1][:512], outs[0])
    assert np.array_equal(outs[1], O.select_working_set(f, y, alpha, C, C, marked, 768, nu=bool(nu)))
    tail = outs[1][512:]
    assert (tail >= 0).all() and len(set(tail.tolist()) | set(outs[0].tolist()) | set(marked.tolist())) == 768 + n_marked


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("n", [700, 3200, 100000, 300001])
def test_selections_in_a_row_on_one_workspace(n, nu):
    """The solver's pattern (csmosolver.cpp:63-77): one full selection, then one per outer iteration that keeps
    half of the previous set, all on one workspace that each call leaves ready for the next.  The f values change
    from call to call between distinct values, massive ties (the remaining digits are then resolved by the final
    kernel's workgroup) and few distinct values."""
    ws = min(1024, 1 << (n.bit_length() - 1))
    q = ws // 2
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    wsp.random_(0, 256)   # whatever an earlier user of the memory left there
    prev = None
    for it, tie_mode in enumerate([0, 1, 0, 2, 1, 1, 0]):
        f, y, alpha, C, _ = _select_case(n, q, 0, 7 * n + it, tie_mode, nu)
        marked = np.zeros(0, dtype=np.int32) if it == 0 else np.ascontiguousarray(prev[q:])
        n_select = ws if it == 0 else q
        want = O.select_working_set(f, y, alpha, C, C, marked, n_select, nu=bool(nu))
        f_d, y_d, a_d, m_d = G.dev(f), G.dev(y), G.dev(alpha), G.dev(marked if it else np.zeros(1, dtype=np.int32))
        out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        capi.call("tsvm_select_working_set" if it == 0 else "tsvm_select_working_set_again", G.ptr(f_d), G.ptr(y_d),
                  G.ptr(a_d), n, C, C, G.ptr(m_d) if it else None, len(marked), G.ptr(out_d), n_select, nu, G.ptr(wsp),
                  G.stream())
        got = G.host(out_d)
        assert np.array_equal(got, want), "call %d: first mismatch at %s" % (it, np.flatnonzero(got != want)[:5])
        prev = got if it == 0 else np.concatenate([prev[q:], got])
        assert (prev >= 0).all()


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("group", [2, 63, 64, 255, 300])
@pytest.mark.parametrize("n,n_select", [(1030, 1000), (6000, 16), (6000, 64), (6000, 512)])
def test_selection_of_lists_with_equal_values(n, n_select, group, nu):
    """Every value of f belongs to `group` instances, all free: a list's order within a value, and the place of an instance in the
    paired side's list, are up to the index, in lists that end inside a group, inside sixteen entries and inside 64."""
    rng = np.random.default_rng(n + group)
    f = rng.permutation(np.repeat(rng.normal(size=n // group + 1), group)[:n])
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    alpha = np.full(n, 0.5)
    want = O.select_working_set(f, y, alpha, 1.0, 1.0, np.zeros(0, dtype=np.int32), n_select, nu=bool(nu))
    f_d, y_d, a_d = G.dev(f), G.dev(y), G.dev(alpha)
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    for entry in ("tsvm_select_working_set", "tsvm_select_working_set_again", "tsvm_select_working_set_again"):
        out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        capi.call(entry, G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, 1.0, 1.0, None, 0, G.ptr(out_d), n_select, nu, G.ptr(wsp), G.stream())
        got = G.host(out_d)
        assert np.array_equal(got, want), "first mismatch at %s" % np.flatnonzero(got != want)[:5]


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("n,tie_mode", [(150, 0), (5000, 2), (200000, 0), (200000, 1)])
def test_selection_with_folded_ids(n, tie_mode, nu):
    """The 2n-variable problem of SVR (svr.cpp:14-28): the selection also delivers each id modulo n / 2, the stored row
    behind the variable; same ids as the plain selection, on a fresh and on a re-used workspace."""
    half = n // 2
    ws = min(1024, 1 << (n.bit_length() - 1))
    q = ws // 2
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    prev = None
    for it in range(3):
        f, y, alpha, C, _ = _select_case(n, q, 0, 5 * n + it, tie_mode, nu)
        marked = np.zeros(0, dtype=np.int32) if it == 0 else np.ascontiguousarray(prev[q:])
        n_select = ws if it == 0 else q
        want = O.select_working_set(f, y, alpha, C, C, marked, n_select, nu=bool(nu))
        f_d, y_d, a_d, m_d = G.dev(f), G.dev(y), G.dev(alpha), G.dev(marked if it else np.zeros(1, dtype=np.int32))
        out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        fold_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        capi.call("tsvm_select_working_set_folded", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, G.ptr(m_d) if it else None,
                  len(marked), G.ptr(out_d), n_select, nu, G.ptr(wsp), int(it > 0), half, G.ptr(fold_d), G.stream())
        got = G.host(out_d)
        assert np.array_equal(got, want)
        assert np.array_equal(G.host(fold_d), np.where(want >= 0, want % half, -1))
        prev = got if it == 0 else np.concatenate([prev[q:], got])


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("row_type", [capi.ROW_F64, capi.ROW_F32])
@pytest.mark.parametrize("n_cols,repeat,ws,ld_pad,tie_mode", [(1, 1, 1, 0, 0), (700, 1, 512, 3, 0), (4099, 2, 64, 1, 2), (16385, 1, 300, 1, 0), (32771, 4, 100, 1, 2),
                                                             (300001, 1, 1024, 7, 0), (270000, 2, 200, 0, 0),
                                                             (262144, 1, 1024, 0, 1), (150000, 3, 16, 4, 2)])
def test_update_f_with_the_next_selection(n_cols, repeat, ws, ld_pad, tie_mode, row_type, nu):
    """One call that updates f and selects the next working set on the new values: f as the oracle's update_f leaves
    it, the ids as the oracle's selection on that f, with the half of the previous set that stays excluded.  Two such
    calls in a row on one workspace; with tie_mode 1 and 2 the update changes nothing (all alpha_diff zero), so that
    the selection meets massive ties and few distinct values."""
    n = n_cols * repeat
    rng = np.random.default_rng(n + ws + nu)
    ld = n_cols + ld_pad
    k = rng.random((ws, ld))
    if row_type == capi.ROW_F32:
        k = k.astype(np.float32)
    k64 = np.ascontiguousarray(np.concatenate([k.astype(np.float64)[:, :n_cols]] * repeat, axis=1))
    sel = min(1024, 1 << (n.bit_length() - 1))
    q = max(sel // 2, 1)
    f, y, alpha, C, _ = _select_case(n, q, 0, 3 * n + 1, tie_mode, nu)
    f_d, y_d, a_d, k_d = G.dev(f), G.dev(y), G.dev(alpha), G.dev(k)
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    wsp.random_(0, 256)
    out_d = torch.full((sel,), -7, dtype=torch.int32, device="cuda")
    capi.call("tsvm_select_working_set", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, None, 0, G.ptr(out_d), sel, nu, G.ptr(wsp),
              G.stream())
    prev = G.host(out_d)
    assert np.array_equal(prev, O.select_working_set(f, y, alpha, C, C, np.zeros(0, dtype=np.int32), sel, nu=bool(nu)))
    for call in range(2):
        marked = np.ascontiguousarray(prev[sel - q:]) if sel > 1 else np.zeros(0, dtype=np.int32)
        marked = marked[marked >= 0]
        ad = rng.standard_normal(ws)
        ad[rng.random(ws) < 0.4] = 0
        if tie_mode:
            ad[:] = 0
        f = O.update_f(f, ad, k64, n)
        want = O.select_working_set(f, y, alpha, C, C, marked, q, nu=bool(nu))
        ad_d, m_d = G.dev(ad), G.dev(marked if len(marked) else np.zeros(1, dtype=np.int32))
        new_d = torch.full((q,), -7, dtype=torch.int32, device="cuda")
        folded_d = torch.full((q,), -7, dtype=torch.int32, device="cuda")
        capi.call("tsvm_update_f_select", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d), row_type, None, ld, n_cols, repeat, G.ptr(y_d),
                  G.ptr(a_d), C, C, G.ptr(m_d) if len(marked) else None, len(marked), G.ptr(new_d), q, nu, G.ptr(wsp),
                  G.ptr(folded_d) if repeat > 1 else None, G.stream())
        assert np.array_equal(G.host(f_d), f)
        got = G.host(new_d)
        assert np.array_equal(got, want), "call %d: first mismatch at %s" % (call, np.flatnonzero(got != want)[:5])
        if repeat > 1:
            assert np.array_equal(G.host(folded_d), np.where(want >= 0, want % n_cols, -1))
        prev = np.concatenate([prev[q:], got]) if sel > 1 else got
        # the instances change their state between the calls, as the local solver would change them
        alpha = alpha.copy()
        alpha[rng.integers(0, n, size=min(n, 300))] = rng.choice([0.0, C, 0.5 * C], size=min(n, 300))
        a_d = G.dev(alpha)


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("n_cols,repeat,row_type", [(2, 1, capi.ROW_F32), (700, 1, capi.ROW_F64), (3200, 1, capi.ROW_F32), (30000, 2, capi.ROW_F32),
                                                    (70001, 1, capi.ROW_F64), (262144, 1, capi.ROW_F32), (1 << 20, 1, capi.ROW_F32)])
def test_guided_selections(n_cols, repeat, row_type, nu):
    """Selections that follow one another with the last one as a guide: f that moves a little, by far more than the guide reaches (either
    way, and in scale), ends in ties, has infinite values, and sides with fewer candidates than are asked for; and selections by
    digits in between, which find the workspace as they want it.  The ids are the oracle's whatever the guide was worth."""
    n = n_cols * repeat
    rng = np.random.default_rng(n + nu)
    sel = min(1024, 1 << (n.bit_length() - 1))
    q = max(sel // 2, 1)
    ld = n_cols
    k_d = G.dev(np.zeros((1, ld), dtype=np.float32 if row_type == capi.ROW_F32 else np.float64))
    ad_d = G.dev(np.zeros(1))
    y = np.where(rng.random(n) < 0.5, 1, -1).astype(np.int32)
    y[0] = 1
    C, f = 1.0, rng.standard_normal(n)
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    wsp.random_(0, 256)
    y_d = G.dev(y)
    prev = None
    missed_d = torch.zeros(1, dtype=torch.int32, device="cuda")
    near = rng.standard_normal(n)
    steps = [("digits", f), ("guided", f), ("guided", f + 0.01 * near), ("guided", f + 1e4), ("digits", f), ("guided", 1e-6 * f), ("guided", 1e6 * f),
             ("guided", np.round(f)), ("guided", f), ("guided", np.full(n, -1.0)), ("guided", f), ("guided", np.where(near > 1.5, np.inf, f)),
             ("guided", np.where(near > 1.5, -np.inf, f)), ("digits", np.zeros(n)), ("guided", f), ("few", f), ("guided", f - 0.02 * near)]
    for at, (how, fn) in enumerate(steps):
        alpha = rng.choice([0.0, 0.5 * C, C], size=n)
        if how == "few":   # (I_up has some seven instances)
            alpha = np.where(y > 0, C, 0.0)
            alpha[rng.integers(0, n, size=7)] = 0.5 * C
        fn = np.ascontiguousarray(fn, dtype=np.float64)
        marked = np.zeros(0, dtype=np.int32) if prev is None else np.ascontiguousarray(prev[prev >= 0][-q:])
        n_select = sel if prev is None else q
        want = O.select_working_set(fn, y, alpha, C, C, marked, n_select, nu=bool(nu))
        f_d, a_d, m_d = G.dev(fn), G.dev(alpha), G.dev(marked if len(marked) else np.zeros(1, dtype=np.int32))
        out_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        fold_d = torch.full((n_select,), -7, dtype=torch.int32, device="cuda")
        missed_d.zero_()
        m_ptr = G.ptr(m_d) if len(marked) else None
        args = (G.ptr(f_d), G.ptr(ad_d), 1, G.ptr(k_d), row_type, None, ld, n_cols, repeat, G.ptr(y_d), G.ptr(a_d), C, C, m_ptr, len(marked),
                G.ptr(out_d), n_select, nu, G.ptr(wsp), G.ptr(fold_d) if repeat > 1 else None)
        if prev is None:
            capi.call("tsvm_select_working_set", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, None, 0, G.ptr(out_d), n_select, nu, G.ptr(wsp), G.stream())
        elif how == "digits":
            capi.call("tsvm_update_f_select", *args, G.stream())
        else:
            capi.call("tsvm_update_f_select_guided", *args, None, 0, 0, G.ptr(missed_d), G.stream())
        got = G.host(out_d)
        assert np.array_equal(got, want), "step %d (%s): first mismatch at %s" % (at, how, np.flatnonzero(got != want)[:5])
        if repeat > 1 and prev is not None:
            assert np.array_equal(G.host(fold_d), np.where(want >= 0, want % n_cols, -1))
        if at == 2 or n <= 1024:
            assert G.host(missed_d)[0] == 0
        if at == 9 and n > 8192:   # (thousands of equal values)
            assert G.host(missed_d)[0] == 1
        prev = got


@pytest.mark.parametrize("row_type,line", [(capi.ROW_F64, 32768), (capi.ROW_F32, 65536)])
@pytest.mark.parametrize("beyond,ld_pad", [(0, 0), (0, 1), (1, 1), (1, 2)])
def test_update_f_at_the_line_between_its_kernels(row_type, line, beyond, ld_pad):
    """The last size of the kernel whose wavefronts take the rows in turn and the first of the one thread per column, rows aligned to two
    columns and not, with and without the selection's first pass."""
    n, ws = line + beyond, 48
    rng = np.random.default_rng(n + ld_pad)
    k = rng.random((ws, n + ld_pad)).astype(np.float32 if row_type == capi.ROW_F32 else np.float64)
    f, ad = rng.standard_normal(n), np.where(rng.random(ws) < 0.3, 0.0, rng.standard_normal(ws))
    f_d, ad_d, k_d = G.dev(f), G.dev(ad), G.dev(k)
    capi.call("tsvm_update_f", G.ptr(f_d), G.ptr(ad_d), ws, G.ptr(k_d), row_type, None, n + ld_pad, n, 1, G.stream())
    assert np.array_equal(G.host(f_d), O.update_f(f, ad, np.ascontiguousarray(k[:, :n].astype(np.float64)), n))
    test_update_f_with_the_next_selection(n, 2, ws, ld_pad, 0, row_type, 0)


def test_empty_inputs_are_no_ops():
    """Zero rows, zero columns, an empty working set, nothing to select: every entry point returns success and
    leaves its outputs untouched."""
    x = torch.zeros((4, 8), dtype=torch.float64, device="cuda")
    sd = torch.zeros(4, dtype=torch.float64, device="cuda")
    out = torch.full((4, 8), 7.0, dtype=torch.float64, device="cuda")
    for n, m in ((0, 4), (4, 0)):
        capi.call("tsvm_get_rows_dense", G.ptr(x), 8, None, n, 3, G.ptr(sd), G.ptr(x), 8, None, m, G.ptr(sd), 2, 0.5, 0.0, 3,
                  G.ptr(out), capi.ROW_F64, None, 8, G.stream())
    f = torch.full((5,), 3.0, dtype=torch.float64, device="cuda")
    ad = torch.ones(4, dtype=torch.float64, device="cuda")
    capi.call("tsvm_update_f", G.ptr(f), G.ptr(ad), 0, G.ptr(out), capi.ROW_F64, None, 8, 5, 1, G.stream())
    capi.call("tsvm_update_f", G.ptr(f), G.ptr(ad), 4, G.ptr(out), capi.ROW_F64, None, 8, 0, 1, G.stream())
    ids = torch.full((4,), -7, dtype=torch.int32, device="cuda")
    y = torch.ones(5, dtype=torch.int32, device="cuda")
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(5), dtype=torch.uint8, device="cuda")
    capi.call("tsvm_select_working_set", G.ptr(f), G.ptr(y), G.ptr(f), 5, 1.0, 1.0, None, 0, G.ptr(ids), 0, 0, G.ptr(wsp),
              G.stream())
    assert (G.host(out) == 7.0).all() and (G.host(f) == 3.0).all() and (G.host(ids) == -7).all()
    # an all-zero alpha_diff reads no row at all and leaves f as it is
    zeros = torch.zeros(4, dtype=torch.float64, device="cuda")
    capi.call("tsvm_update_f", G.ptr(f), G.ptr(zeros), 4, G.ptr(out), capi.ROW_F64, None, 8, 5, 1, G.stream())
    assert (G.host(f) == 3.0).all()


def test_report_ids_to_host_memory():
    """tsvm_report_ids: the ids land in host memory the device can write, folded when asked, and the word the host polls
    is there once the stream has run (a host-side row store reads its new ids this way instead of through a copy)."""
    rng = np.random.default_rng(4)
    ids = rng.integers(0, 50000, size=512).astype(np.int32)
    ids[7] = -1                                             # a side that ran dry leaves -1
    ids_d = G.dev(ids)
    host = torch.full((1024 + 16,), -7, dtype=torch.int32).pin_memory()
    for n_ids, fold, word in [(512, 0, 1), (512, 20000, 2), (100, 0, 3), (0, 0, 4)]:
        capi.call("tsvm_report_ids", G.ptr(ids_d), n_ids, fold, host.data_ptr(), 1024, word, G.stream())
        torch.cuda.synchronize()
        got = host.numpy()
        want = ids[:n_ids].copy()
        if fold:
            want[want >= 0] %= fold
        assert np.array_equal(got[:n_ids], want) and got[1024] == word
    with pytest.raises(capi.TsvmError):
        capi.call("tsvm_report_ids", G.ptr(ids_d), 600, 0, host.data_ptr(), 512, 1, G.stream())      # the word would lie inside the ids


@pytest.mark.parametrize("nu", [0, 1])
@pytest.mark.parametrize("n,tie_mode,fold", [(150, 0, 0), (5001, 2, 0), (5000, 0, 2500), (70000, 1, 35000)])
def test_selections_that_report_their_ids(n, tie_mode, fold, nu):
    """The selection whose last kernel tells the host: the same ids in device memory, folded and in host memory, and the word behind
    them, on the counting path, the one-workgroup path (ties) and where a side runs dry; alone and behind update_f."""
    ws = min(1024, 1 << (n.bit_length() - 1))
    q = ws // 2
    rng = np.random.default_rng(n)
    cols = fold if fold else n
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    host = torch.full((ws + 16,), -7, dtype=torch.int32).pin_memory()
    f, y, alpha, C, _ = _select_case(n, q, 0, 11 * n, tie_mode, nu)
    f_d, y_d, a_d = G.dev(f), G.dev(y), G.dev(alpha)
    out_d = torch.full((ws,), -7, dtype=torch.int32, device="cuda")
    fold_d = torch.full((ws,), -7, dtype=torch.int32, device="cuda")
    capi.call("tsvm_select_working_set_report", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, None, 0, G.ptr(out_d), ws, nu, G.ptr(wsp), 0, fold,
              G.ptr(fold_d) if fold else None, host.data_ptr(), ws, 41, G.stream())
    want = O.select_working_set(f, y, alpha, C, C, np.zeros(0, dtype=np.int32), ws, nu=bool(nu))
    torch.cuda.synchronize()
    assert np.array_equal(G.host(out_d), want) and np.array_equal(host.numpy()[:ws], want) and host.numpy()[ws] == 41
    if fold:
        assert np.array_equal(G.host(fold_d), np.where(want >= 0, want % fold, -1))
    marked = np.ascontiguousarray(want[q:][want[q:] >= 0])
    k = rng.random((32, cols)).astype(np.float32)
    ad = np.zeros(32) if tie_mode else rng.standard_normal(32)
    k64 = k.astype(np.float64)
    f = O.update_f(f, ad, np.ascontiguousarray(np.concatenate([k64, k64], axis=1) if fold else k64), n)
    want = O.select_working_set(f, y, alpha, C, C, marked, q, nu=bool(nu))
    ad_d, k_d, m_d = G.dev(ad), G.dev(k), G.dev(marked)
    capi.call("tsvm_update_f_select_report", G.ptr(f_d), G.ptr(ad_d), 32, G.ptr(k_d), capi.ROW_F32, None, cols, cols, n // cols, G.ptr(y_d), G.ptr(a_d),
              C, C, G.ptr(m_d), len(marked), G.ptr(out_d), q, nu, G.ptr(wsp), G.ptr(fold_d) if fold else None, host.data_ptr(), ws, 42, G.stream())
    torch.cuda.synchronize()
    assert np.array_equal(G.host(f_d), f)
    assert np.array_equal(G.host(out_d)[:q], want) and np.array_equal(host.numpy()[:q], want) and host.numpy()[ws] == 42
    with pytest.raises(capi.TsvmError):   # the word would lie inside the ids
        capi.call("tsvm_select_working_set_report", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, None, 0, G.ptr(out_d), ws, nu, G.ptr(wsp), 0, 0, None,
                  host.data_ptr(), ws - 1, 1, G.stream())


@pytest.mark.parametrize("nu", [0, 1])
def test_a_selection_of_no_ids_still_reports(nu):
    """n_select == 0: nothing is written but the word that the host polls."""
    n = 300
    f, y, alpha, C, _ = _select_case(n, 16, 0, 5, 0, nu)
    f_d, y_d, a_d = G.dev(f), G.dev(y), G.dev(alpha)
    wsp = torch.empty(capi.kernel_lib().tsvm_select_workspace(n), dtype=torch.uint8, device="cuda")
    out_d = torch.full((4,), -7, dtype=torch.int32, device="cuda")
    host = torch.full((4,), -7, dtype=torch.int32).pin_memory()
    capi.call("tsvm_select_working_set_report", G.ptr(f_d), G.ptr(y_d), G.ptr(a_d), n, C, C, None, 0, G.ptr(out_d), 0, nu, G.ptr(wsp), 0, 0, None,
              host.data_ptr(), 1, 43, G.stream())
    torch.cuda.synchronize()
    assert host.tolist() == [-7, 43, -7, -7] and out_d.tolist() == [-7] * 4
