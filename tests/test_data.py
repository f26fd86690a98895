"""Host-side data handling: LibSVM text round trip (float32 rounding on load) and the seeded workloads."""
import ctypes

import numpy as np
import pytest

import selftest_lib
from thundersvm_amd import data as D
from thundersvm_amd import model as M


def test_libsvm_round_trip(tmp_path):
    w = D.workload_c4(scale=0.002)
    path = str(tmp_path / "c4.txt")
    D.save_libsvm(path, w["train"])
    back = D.load_libsvm(path)
    assert np.array_equal(back.ptr, w["train"].ptr) and np.array_equal(back.col, w["train"].col)
    assert np.array_equal(back.val, w["train"].val) and np.array_equal(back.y, w["train"].y)


def test_values_are_float32_exact_and_seeded():
    for gen in (D.workload_c1, D.workload_c2, D.workload_c3, D.workload_c4, D.workload_c5):
        a, b = gen(0.01), gen(0.01)
        v = a["train"].val
        assert np.array_equal(v, v.astype(np.float32).astype(np.float64))
        assert np.array_equal(v, b["train"].val) and np.array_equal(a["train"].y, b["train"].y)


def test_workload_shapes():
    c4 = D.workload_c4(0.01)["train"]
    assert c4.n_features == 54 and set(np.unique(c4.y)) <= set(range(1, 8))
    assert np.all(np.diff(c4.ptr) == 12)                     # 10 continuous + 2 active one-hot columns
    c3 = D.workload_c3(0.01)["train"]
    assert c3.n_features <= 20958
    norms = np.sqrt(np.add.reduceat(c3.val ** 2, c3.ptr[:-1]))
    assert np.abs(norms - 1).max() < 1e-6
    c5 = D.workload_c5(0.01)
    assert c5["train"].n_features == 90 and np.all(np.diff(c5["train"].ptr) == 90)
    dense = c5["train"].to_dense()
    assert dense.shape[1] == 91 and np.all(dense[:, 0] == 0)


def _new_csr(n, ptr, col, val):
    L = M.host_lib()
    a = [None if v is None else np.ascontiguousarray(v, t) for v, t in ((ptr, np.int64), (col, np.int32), (val, np.float64))]
    types = [ctypes.POINTER(c) for c in (ctypes.c_int64, ctypes.c_int, ctypes.c_double)]
    h = L.tsvm_dataset_new_csr(n, *[None if v is None else v.ctypes.data_as(t) for v, t in zip(a, types)], None)
    if not h:
        return None
    rows = L.tsvm_dataset_rows(ctypes.c_void_p(h))
    L.tsvm_dataset_free(ctypes.c_void_p(h))
    return rows


def test_csr_rows_that_end_before_they_begin_are_refused():
    val, col = np.arange(1.0, 9.0), np.arange(8)
    assert _new_csr(3, [0, 2, 5, 8], col, val) == 3
    assert _new_csr(2, [2, 2, 8], col, val) == 2                 # an offset and an empty row are fine
    for n, ptr in ((3, [0, 5, 3, 8]), (2, [0, 3, 2]), (1, [4, 0]), (-1, [0, 1])):
        assert _new_csr(n, ptr, col, val) is None
        assert M.host_lib().tsvm_model_last_error()
    many = np.arange(100001, dtype=np.int64) // 20000
    assert _new_csr(100000, many, col, val) == 100000
    many[77777] = 0
    assert _new_csr(100000, many, col, val) is None
    assert _new_csr(0, None, None, None) == 0                    # no rows: nothing is read


@pytest.mark.parametrize("ptr,want", [([0, 2, 2, 6], [[0, 1], [], [2, 3, 4, 5]]), ([0, 5, 3, 6], [[0, 1, 2, 3, 4], [], [3, 4, 5]]),
                                      ([3, 6, 0, 2], [[3, 4, 5], [], [0, 1]]), ([0], [])])
def test_scikit_sparse_matrix(ptr, want):
    """Rows come out as the loop over [row_ptr[r], row_ptr[r + 1]) reads them: one that ends before it begins is empty."""
    L = selftest_lib.lib()
    val, col, p = np.arange(10, 16, dtype=np.float32), np.arange(6, dtype=np.int32), np.array(ptr, np.int32)
    out_ptr, out_col, out_val = np.zeros(len(ptr), np.int64), np.zeros(32, np.int32), np.zeros(32)
    n = L.tsvm_selftest_load_matrix(0, len(ptr) - 1, 0, val.ctypes.data, p.ctypes.data, col.ctypes.data, out_ptr.ctypes.data,
                                    out_col.ctypes.data, out_val.ctypes.data, 32)
    flat = [e for r in want for e in r]
    assert n == len(flat) and out_ptr.tolist() == np.concatenate([[0], np.cumsum([len(r) for r in want])]).astype(int).tolist()
    assert out_col[:n].tolist() == [e + 1 for e in flat] and out_val[:n].tolist() == [10.0 + e for e in flat]


@pytest.mark.parametrize("dense,rows,features", [(0, -1, 0), (1, -1, 0), (1, -1, 3), (1, 2, -1)])
def test_scikit_matrix_of_a_negative_size_is_refused(dense, rows, features):
    L = selftest_lib.lib()
    buf = np.zeros(64)
    at = buf.ctypes.data
    assert L.tsvm_selftest_load_matrix(dense, rows, features, at, at, at, at, at, at, 0) == -1


@pytest.mark.parametrize("entries", [3, 200000])
def test_feature_id_zero_in_csr_rows_is_noticed(entries):
    """One feature id 0 anywhere makes a data set zero-based (it moves every feature's place in the linear coefficients)."""
    rng = np.random.default_rng(entries)
    csr = D.CsrData(np.array([0, 2, entries], np.int64), rng.integers(1, 9, entries).astype(np.int32), np.ones(entries), np.array([1.0, 0.0]))
    csr.col[1] = 9
    assert M.Dataset(csr).csr()[1:] == (9, False)
    csr.col[entries - 1] = 0
    assert M.Dataset(csr).csr()[1:] == (9, True)
