"""Loads the test-only native library (tests/native/selftest.cpp, built by thundersvm_amd.build.build_selftests):
self-tests of host-layer pieces that no product entry point reaches."""
import ctypes
import os

from thundersvm_amd import model

_LIB = None


def lib():
    global _LIB
    if _LIB is None:
        model.host_lib()        # the product libraries it links against
        path = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native", "libtsvm_selftest.so")
        if not os.path.exists(path):
            raise RuntimeError("%s is missing: run `python -m thundersvm_amd.build`" % path)
        L = ctypes.CDLL(path)
        L.tsvm_selftest_last_error.restype = ctypes.c_char_p
        L.tsvm_selftest_row_cache.restype = ctypes.c_longlong
        L.tsvm_selftest_row_cache.argtypes = [ctypes.c_int] * 4
        L.tsvm_selftest_solver_wait.argtypes = [ctypes.c_int, ctypes.c_int]
        L.tsvm_selftest_subset_of_rows.argtypes = [ctypes.c_double]
        L.tsvm_selftest_indicator_run.argtypes = [ctypes.c_double]
        L.tsvm_selftest_load_matrix.restype = ctypes.c_longlong
        L.tsvm_selftest_load_matrix.argtypes = [ctypes.c_int] * 3 + [ctypes.c_void_p] * 6 + [ctypes.c_longlong]
        L.tsvm_selftest_chip_split.argtypes = [ctypes.c_int] * 2 + [ctypes.c_longlong] * 3
        L.tsvm_selftest_rows_ahead.argtypes = [ctypes.c_int] * 3 + [ctypes.c_longlong] * 2
        L.tsvm_selftest_thread_limit.argtypes = [ctypes.c_int] * 2
        L.tsvm_selftest_sliced_deal.argtypes = [ctypes.c_longlong] * 2 + [ctypes.c_int, ctypes.c_void_p]
        L.tsvm_selftest_guided.argtypes = [ctypes.c_longlong, ctypes.c_int, ctypes.c_int]
        L.tsvm_selftest_mark_support_vectors.restype = ctypes.c_double
        L.tsvm_selftest_mark_support_vectors.argtypes = [ctypes.c_int] * 2
        _LIB = L
    return _LIB
