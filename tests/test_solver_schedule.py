"""Which parts of an iteration run side by side in a solve that has the chip to itself (ChipSplit, host/solver.h).  Host only."""
import pytest

import selftest_lib

BESIDE, WARM = 1, 2


@pytest.mark.parametrize("features,n,before,now,want", [
    (784, 100000, 512, 512, BESIDE),          # rows for 1.2 ms: the block and the solver fit beside them
    (784, 20000, 512, 512, 0),                # 0.24 ms: they do not, and the rows outlast a second warming
    (90, 400000, 512, 512, BESIDE),
    (90, 40000, 512, 512, WARM),              # 0.06 ms
    (90, 40000, 0, 0, 0),                     # no rows that would push the block out
    (784, 100000, 512, 20, BESIDE),           # few misses after many: the block is on the solver's CUs, where it may not be there yet
    (784, 100000, 20, 512, 0),
])
def test_chip_split(features, n, before, now, want):
    assert selftest_lib.lib().tsvm_selftest_chip_split(features, 1024, n, before, now) == want


@pytest.mark.parametrize("dense,features,n,before,want", [
    (1, 784, 100000, 512, True),
    (1, 784, 20000, 512, False),
    (0, 20958, 18000, 512, False),
    (0, 20958, 60000, 512, False),            # sparse rows take microseconds where the dense price says milliseconds
    (0, 784, 100000, 512, False),
])
def test_rows_ahead(dense, features, n, before, want):
    assert selftest_lib.lib().tsvm_selftest_rows_ahead(dense, features, 1024, n, before) == want


@pytest.mark.parametrize("n", [2, 1000, 40000, 300000, 1 << 20])
def test_guides_that_fail_cost_little(n):
    """The first selection goes by digits and guides that decide are used ever after.  A guide that fails costs 3.6 ns an instance: however
    often they do, 10 us a selection at most, over 20,000 of them."""
    L = selftest_lib.lib()
    assert L.tsvm_selftest_guided(n, 1000, 0) == 999
    for every in (1, 2, 32, 33, 100):
        guided = L.tsvm_selftest_guided(n, 20000, every)
        assert guided // every * 3.6e-3 * n <= 10.0 * 20000
        assert guided > 0


def test_no_guides_for_many_instances():
    assert selftest_lib.lib().tsvm_selftest_guided((1 << 20) + 1, 1000, 0) == 0


@pytest.mark.parametrize("classes,each", [(1, 3), (2, 1), (3, 5), (7, 40), (150, 2)])
def test_marks_of_support_vectors(classes, each):
    assert selftest_lib.lib().tsvm_selftest_mark_support_vectors(classes, each) >= 0


def test_marks_take_time_with_the_pairs():
    """Two million pairs are gone through twice, once for each class (0.1 s), and not once for every class (3.6 s)."""
    assert 0 <= selftest_lib.lib().tsvm_selftest_mark_support_vectors(2000, 1) < 1e6
