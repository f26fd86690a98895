// Self-tests of host-layer pieces that have no other way in from a test: the device buffer type that stands in for
// the reference's SyncArray (the cases of src/test/test_syncmem.cpp and test_syncarray.cpp that apply), the kernel-row
// cache's bookkeeping, the host's bounded wait for the local solver, and the matrices of the scikit entry points.  Built into a library of its own, next to
// the tests; the product libraries do not contain it.
#include <omp.h>

#include <algorithm>
#include <chrono>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "../../thundersvm_amd/csrc/sliced_deal.h"
#include "../../thundersvm_amd/host/dataset.h"
#include "../../thundersvm_amd/host/device.h"
#include "../../thundersvm_amd/host/kernelmatrix.h"
#include "../../thundersvm_amd/host/models.h"
#include "../../thundersvm_amd/host/row_cache.h"
#include "../../thundersvm_amd/host/rows.h"
#include "../../thundersvm_amd/host/solver.h"

namespace {

thread_local std::string g_selftest_error;

#define SELFTEST_GUARD(...)                        \
    try {                                          \
        __VA_ARGS__;                               \
        return 0;                                  \
    } catch (const std::exception &e) {            \
        g_selftest_error = e.what();               \
        return -1;                                 \
    }

using tsvm::RowCache;

// Drives RowCache the way a solve does (first working set of ws rows, then q = ws / 2 new rows per iteration while the
// previous new half stays pinned) on a cyclic sequence of n_ids ids, and checks after every step that each row of the
// working set has a slot of its own and that the tables agree.  Returns the number of hits, or -1 with `what` set.
long long row_cache_selftest(int n_ids, int slots, int ws, int iterations, std::string &what) {
    if (n_ids < ws || slots < 2 * ws || ws < 2 || ws % 2) { what = "bad arguments"; return -1; }
    RowCache c;
    c.init(n_ids, slots);
    const int q = ws / 2;
    std::vector<int> ids(ws), slot(ws);
    long long hits = 0;
    int next_id = 0;
    for (int it = 0; it < iterations; ++it) {
        const int n_new = it == 0 ? ws : q, first_new = it == 0 ? 0 : q;
        if (it > 0) {
            for (int t = 0; t < q; ++t) c.release(slot[t]);
            for (int t = 0; t < q; ++t) { ids[t] = ids[t + q]; slot[t] = slot[t + q]; }
        }
        for (int t = 0; t < n_new; ++t) {
            const int id = next_id;
            next_id = (next_id + 1) % n_ids;
            int s = c.lookup(id);
            if (s >= 0) ++hits;
            else s = c.insert(id);
            if (s < 0) { what = "no slot left for a working-set row"; return -1; }
            ids[first_new + t] = id;
            slot[first_new + t] = s;
        }
        std::vector<char> taken(slots, 0);
        for (int t = 0; t < ws; ++t) {
            if (slot[t] < 0 || slot[t] >= slots || c.slot_of[ids[t]] != slot[t] || c.id_of[slot[t]] != ids[t]) {
                what = "a working-set row lost its slot";
                return -1;
            }
            if (taken[slot[t]] && n_ids >= 2 * ws) { what = "two working-set rows share a slot"; return -1; }
            taken[slot[t]] = 1;
            if (c.pins[slot[t]] < 1) { what = "a working-set row is not pinned"; return -1; }
        }
        int listed = 0;
        for (int s2 = c.head; s2 >= 0; s2 = c.next[s2]) {
            if (c.pins[s2] != 0) { what = "a pinned row is on the eviction list"; return -1; }
            if (++listed > slots) { what = "the eviction list has a cycle"; return -1; }
        }
        int pinned = 0;
        for (int s2 = 0; s2 < c.used; ++s2) pinned += c.pins[s2] > 0;
        if (listed + pinned != c.used) { what = "rows neither pinned nor listed"; return -1; }
    }
    return hits;
}

}  // namespace

extern "C" {

const char *tsvm_selftest_last_error(void) { return g_selftest_error.c_str(); }

// Needs a device.  0 on success, -1 with a message otherwise.
int tsvm_selftest_device_buffer(void) {
    SELFTEST_GUARD({
        using tsvm::DeviceBuffer;
        auto expect = [](bool ok, const char *what) { if (!ok) throw std::runtime_error(std::string("DeviceBuffer: ") + what); };
        const size_t base = tsvm::device_bytes_in_use();
        {
            DeviceBuffer<char> a(100);
            expect(a.data() != nullptr && a.size() == 100, "allocation");
            expect(tsvm::device_bytes_in_use() == base + 100, "one allocation counted");
            DeviceBuffer<char> b;                       // nothing allocated, nothing counted
            expect(b.data() == nullptr && tsvm::device_bytes_in_use() == base + 100, "empty buffer");
            b.resize(100);
            expect(tsvm::device_bytes_in_use() == base + 200, "second allocation counted");
            {
                DeviceBuffer<char> t(100);
                expect(tsvm::device_bytes_in_use() == base + 300, "third allocation counted");
                DeviceBuffer<char> moved(std::move(t));   // ownership moves, the bytes are counted once
                expect(t.data() == nullptr && t.size() == 0 && moved.size() == 100, "move");
                expect(tsvm::device_bytes_in_use() == base + 300, "move does not count twice");
            }
            expect(tsvm::device_bytes_in_use() == base + 200, "destruction releases");
            DeviceBuffer<int> d(100);
            expect(d.size() == 100 && tsvm::device_bytes_in_use() == base + 200 + 100 * sizeof(int), "typed size");
            d.resize(20);                               // a resize starts over, as SyncArray::resize does
            expect(d.size() == 20 && tsvm::device_bytes_in_use() == base + 200 + 20 * sizeof(int), "resize");
            std::vector<int> host(10);
            for (int i = 0; i < 10; ++i) host[i] = i;
            d.upload(host.data(), 10, 5);               // interior offsets are accepted
            for (int i = 0; i < 10; ++i) host[i] = -1;
            d.download(host.data(), 10, 5);
            for (int i = 0; i < 10; ++i) expect(host[i] == i, "round trip");
            d.zero();
            const std::vector<int> z = d.to_host();
            for (int v : z) expect(v == 0, "zero fill");
        }
        expect(tsvm::device_bytes_in_use() == base, "everything released");
    })
}

// No device needed.  Returns the number of hits, or -1 (tsvm_selftest_last_error says what broke).
long long tsvm_selftest_row_cache(int n_ids, int slots, int ws, int iterations) {
    std::string what;
    const long long hits = row_cache_selftest(n_ids, slots, ws, iterations, what);
    if (hits < 0) g_selftest_error = "row cache: " + what;
    return hits;
}

// No device needed: waits on a word that nobody writes, with a stream that reports "still running", and returns 0 when
// the wait gave up with its time-out error after timeout_ms (within a second of it), -1 otherwise.  never_written != 0
// makes the stream report "drained" instead: the wait must then fail with its "finished without reporting" error at once.
int tsvm_selftest_solver_wait(int timeout_ms, int never_written) {
    static volatile uint64_t word;
    word = 0x7ff8dead00000001ull;
    const auto t0 = std::chrono::steady_clock::now();
    try {
        if (never_written)
            tsvm::wait_while_pending(&word, word, timeout_ms, [](void *) { return hipSuccess; }, nullptr);
        else
            tsvm::wait_while_pending(&word, word, timeout_ms, [](void *) { return hipErrorNotReady; }, nullptr);
    } catch (const std::runtime_error &e) {
        const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        g_selftest_error = e.what();
        const bool timed_out = g_selftest_error.find("TSVM_SOLVER_TIMEOUT_MS") != std::string::npos;
        if (never_written) return !timed_out && ms < 1000.0 ? 0 : -1;
        return timed_out && ms >= timeout_ms && ms < timeout_ms + 1000.0 ? 0 : -1;
    }
    g_selftest_error = "the wait returned although the word never changed";
    return -1;
}

// No device needed: the same wait by asking, for something that is never done, is done at the third look, or fails.
// 0: as it should be.
int tsvm_selftest_wait_until_done(int timeout_ms) {
    static int looks;
    const auto t0 = std::chrono::steady_clock::now();
    try {
        tsvm::wait_until_done([](void *) { return hipErrorNotReady; }, nullptr, timeout_ms);
        return -1;
    } catch (const std::runtime_error &e) {
        g_selftest_error = e.what();
        const double ms = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
        if (g_selftest_error.find("TSVM_SOLVER_TIMEOUT_MS") == std::string::npos || ms < timeout_ms || ms >= timeout_ms + 1000.0) return -2;
    }
    looks = 0;
    try {
        tsvm::wait_until_done([](void *) { return ++looks < 3 ? hipErrorNotReady : hipSuccess; }, nullptr, 10000);
    } catch (const std::exception &) {
        return -3;
    }
    if (looks != 3) return -4;
    try {
        tsvm::wait_until_done([](void *) { return hipErrorInvalidHandle; }, nullptr, 10000);
        return -5;
    } catch (const std::runtime_error &) {
        return 0;
    }
}

// Needs a device.  What is known about the values of sparse rows and decides how a prediction reads them is known about a
// subset of them as well.  last: the last row's last value (infinite, or no float, or an ordinary one).
int tsvm_selftest_subset_of_rows(double last) {
    SELFTEST_GUARD({
        const int n = 300, per_row = 5;
        std::vector<int64_t> ptr(n + 1);
        std::vector<int> col(n * per_row);
        std::vector<double> val(n * per_row, 0.5);
        for (int r = 0; r <= n; ++r) ptr[r] = r * per_row;
        for (int e = 0; e < n * per_row; ++e) col[e] = 1 + e % per_row * 400 + e / per_row;
        val.back() = last;
        const RowStore rows(n, ptr.data(), col.data(), val.data());
        const std::shared_ptr<DeviceRows> all = DeviceRows::from_host(rows);
        std::vector<int> ids(100);
        for (int i = 0; i < 100; ++i) ids[i] = 299 - 2 * i;
        const std::shared_ptr<DeviceRows> some = DeviceRows::subset(*all, ids.data(), ids.size());
        auto expect = [](bool ok, const char *what) { if (!ok) throw std::runtime_error(std::string("DeviceRows::subset: ") + what); };
        expect(!all->dense && !some->dense && all->sliced_lds > 0 && some->sliced_lds > 0, "layout");
        expect(all->values_finite == (last - last == 0) && some->values_finite == all->values_finite, "finite values");
        expect(all->values_fit_float == ((double) (float) last == last) && some->values_fit_float == all->values_fit_float, "float values");
    })
}

// Needs a device.  The first of a run of indicator columns that ends with the last one: four ordinary columns and thirty
// that one entry a row is set in, 20,000 rows; `last` is the very last entry, in the last column (1: the run is there).
// Returns the first column of the run that get_rows leaves to its epilogue, -1 without one.
int tsvm_selftest_indicator_run(double last) {
    const int n = 20000, per_row = 5;
    std::vector<int64_t> ptr(n + 1);
    std::vector<int> col(n * per_row);
    std::vector<double> val(n * per_row, 0.25);
    for (int r = 0; r <= n; ++r) ptr[r] = r * per_row;
    for (int r = 0; r < n; ++r) {
        for (int c = 0; c < 4; ++c) col[r * per_row + c] = 1 + c;
        col[r * per_row + 4] = r == n - 1 ? 34 : 5 + r % 30;
        val[r * per_row + 4] = 1.0;
    }
    val.back() = last;
    try {
        return DeviceRows::from_host(RowStore(n, ptr.data(), col.data(), val.data()))->ind_first;
    } catch (const std::exception &e) {
        g_selftest_error = e.what();
        return -100;
    }
}

// No device needed.  DataSet::load_from_sparse (dense == 0) or load_from_dense (row_ptr and col_ptr unused) and the rows it
// holds afterwards: out_ptr [row_size + 1], out_col / out_val with room for `cap` entries.  Returns the entries, -1 when refused.
long long tsvm_selftest_load_matrix(int dense, int row_size, int features, float *val, int *row_ptr, int *col_ptr, long long *out_ptr,
                                    int *out_col, double *out_val, long long cap) {
    try {
        DataSet ds;
        if (dense) ds.load_from_dense(row_size, features, val, nullptr);
        else ds.load_from_sparse(row_size, val, row_ptr, col_ptr, nullptr);
        const RowStore &R = ds.rows();
        const long long nnz = (long long) R.nnz();
        for (size_t r = 0; r <= R.size(); ++r) out_ptr[r] = R.ptr()[r];
        for (long long e = 0; e < nnz && e < cap; ++e) { out_col[e] = R.col()[e]; out_val[e] = R.val()[e]; }
        return nnz;
    } catch (const std::exception &e) {
        g_selftest_error = e.what();
        return -1;
    }
}

// The schedule of a solve that has the chip to itself: bit 0 the block beside the rows, bit 1 a second warming behind them, when the
// previous iteration computed m_before rows of n values and this one m_now.
int tsvm_selftest_chip_split(int features, int ws, long long n, long long m_before, long long m_now) {
    using tsvm::ChipSplit;
    const bool beside = ChipSplit::block_beside_rows(features, ws, ChipSplit::rows_seconds(features, m_before, n));
    return (beside ? 1 : 0) | (ChipSplit::warm_behind_rows(beside, ChipSplit::rows_seconds(features, m_now, n)) ? 2 : 0);
}

// The marks of n_classes classes with `each` instances and c % 3 more in class c, whose instance l of pair (i, j) is a support vector where
// (l + 3 i + 7 j) % 11 is 0: the time that takes on one thread in us, or -1 if one is wrong.
double tsvm_selftest_mark_support_vectors(int n_classes, int each) {
    std::vector<int> count(n_classes), start(n_classes);
    int n = 0;
    for (int c = 0; c < n_classes; ++c) {
        start[c] = n;
        count[c] = each + c % 3;
        n += count[c];
    }
    std::vector<std::vector<double>> alpha;
    std::vector<unsigned char> want(n, 0);
    for (int i = 0; i < n_classes; ++i)
        for (int j = i + 1; j < n_classes; ++j) {
            alpha.emplace_back(count[i] + count[j], 0.0);
            for (int l = 0; l < count[i] + count[j]; ++l)
                if ((l + 3 * i + 7 * j) % 11 == 0) {
                    alpha.back()[l] = l % 2 ? 0.5 : -0.5;
                    want[l < count[i] ? start[i] + l : start[j] + l - count[i]] = 1;
                }
        }
    const auto t0 = std::chrono::steady_clock::now();
    const std::vector<unsigned char> got = tsvm::mark_support_vectors(count, start, alpha, 1);
    const double us = std::chrono::duration<double, std::micro>(std::chrono::steady_clock::now() - t0).count();
    return got == want ? us : -1;
}

// Whether an iteration's rows go ahead of the block and the solver, when the previous one computed m_before rows of n values.
int tsvm_selftest_rows_ahead(int dense, int features, int ws, long long n, long long m_before) {
    using tsvm::ChipSplit;
    return ChipSplit::rows_ahead(dense != 0, features, ws, ChipSplit::rows_seconds(features, m_before, n));
}

// Of `selections` selections of n instances in a row, how many are guided when every miss_every-th guided one fails (0: none does).
int tsvm_selftest_guided(long long n, int selections, int miss_every) {
    tsvm::GuideSchedule guides(n);
    int guided = 0;
    bool missed = false;
    for (int i = 0; i < selections; ++i) {
        const bool is = guides.next(missed);
        missed = is && miss_every > 0 && ++guided % miss_every == 0;
        if (is && miss_every == 0) ++guided;
    }
    return guided;
}

// The team of a parallel region when nobody has asked for a number of threads (how 0), n has been asked for as -o and n_jobs do (1), a
// program has set n for itself (2), or another of its threads has asked for n (3).
int tsvm_selftest_thread_limit(int how, int n) {
    if (how == 1) set_threads(n);
    if (how == 2) omp_set_num_threads(n);
    int limit = 0;
    if (how == 3) {
        set_threads(n);
        std::thread([&] { limit = thread_limit(); }).join();
    } else {
        limit = thread_limit();
    }
    set_threads(0);
    return limit;
}

// The sliced CSR kernel's work, n stored rows and n_blocks blocks of working rows: 0 if its workgroups take every slice of every block exactly
// once.  out: workgroups, the most slices that one takes, the most tiles that one builds.
int tsvm_selftest_sliced_deal(long long n, long long n_blocks, int places, long long *out) {
    const SlicedDeal deal = sliced_deal(n, n_blocks, (unsigned) places);
    const long long n_slices = (n + 63) / 64;
    std::vector<unsigned char> taken(n_slices * n_blocks, 0);
    out[0] = deal.workgroups;
    out[1] = out[2] = 0;
    for (unsigned w = 0; w < deal.workgroups; ++w) {
        SlicedWalk walk(deal, w);
        long long slices = 0, tiles = 0;
        for (unsigned block, slice0, slice1; walk.next(deal, block, slice0, slice1); ++tiles) {
            if (block >= n_blocks || slice1 <= slice0 || slice1 > n_slices) return -1;
            for (unsigned s = slice0; s < slice1; ++s)
                if (taken[block * n_slices + s]++) return -1;
            slices += slice1 - slice0;
        }
        out[1] = std::max(out[1], slices);
        out[2] = std::max(out[2], tiles);
    }
    return std::count(taken.begin(), taken.end(), 1) == (long long) taken.size() ? 0 : -1;
}

}  // extern "C"
