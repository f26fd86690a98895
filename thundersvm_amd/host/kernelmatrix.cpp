#include <memory>
#include "kernelmatrix.h"
#include <stdexcept>

#include <algorithm>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>

using tsvm::abi_check;

namespace tsvm {
static int current_device() {
    int dev = 0;
    TSVM_HIP_CHECK(hipGetDevice(&dev));
    return dev;
}

struct DevicePool::Impl {
    // A block beyond that is allocated and freed by every training call, and a free waits for all that the device has in flight, other class
    // pairs' kernels among it.  With 64 MB / 512 MB the staging matrices of 21,000 features (86 MB each) and the rows of the larger pairs of
    // 300,000 instances (115 MB) were: linear text, 18,000 rows, 31.8 -> 31.2 ms a call; seven classes of 300,000 rows 579.7 -> 572.8 and 664.8 ->
    // 656.6 on two cards, within what runs differ by on a third.
    static constexpr size_t MAX_BLOCK = (size_t) 256 << 20, MAX_TOTAL = (size_t) 2 << 30;
    std::mutex mu;
    // [device, block size] -> blocks; `waiting`: released since the device was last known to be idle
    std::map<std::pair<int, size_t>, std::vector<void *>> ready, waiting;
    size_t total = 0;
    // quarter powers of two from 256 bytes on
    static size_t block_size(size_t bytes) {
        size_t p = 256;
        while (p < bytes) p <<= 1;
        if (p == 256) return p;
        const size_t q = p / 8;   // between p/2 and p: p/2 + k * p/8
        return p / 2 + (bytes - p / 2 + q - 1) / q * q;
    }
    void flush_locked() {
        for (auto *m : {&ready, &waiting}) {
            for (auto &kv : *m)
                for (void *p : kv.second) (void) hipFree(p);
            m->clear();
        }
        total = 0;
    }
};

hipStream_t work_stream() {
    static std::mutex mu;
    static std::map<int, hipStream_t> streams;
    const int dev = current_device();
    std::lock_guard<std::mutex> lock(mu);
    auto it = streams.find(dev);
    if (it == streams.end()) {
        hipStream_t s = nullptr;
        TSVM_HIP_CHECK(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
        it = streams.emplace(dev, s).first;
        static bool registered = false;
        if (!registered) {
            registered = true;
            atexit([] {
                for (auto &kv : streams) (void) hipStreamDestroy(kv.second);
                streams.clear();
            });
        }
    }
    return it->second;
}

DevicePool &DevicePool::instance() {
    static DevicePool pool;
    return pool;
}

DevicePool::Impl &DevicePool::impl() {
    // (never destroyed; emptied by an atexit handler, which runs before the HIP runtime's tear-down)
    static Impl *i = [] {
        Impl *n = new Impl();
        atexit([] { DevicePool::instance().flush(); });
        return n;
    }();
    return *i;
}

void *DevicePool::take(size_t bytes, int *device) {
    Impl &I = impl();
    const int dev = *device = current_device();
    const size_t size = Impl::block_size(bytes);
    std::lock_guard<std::mutex> lock(I.mu);
    const auto key = std::make_pair(dev, size);
    auto it = I.ready.find(key);
    if (it == I.ready.end() || it->second.empty()) {
        auto w = I.waiting.find(key);
        if (w != I.waiting.end() && !w->second.empty()) {
            TSVM_HIP_CHECK(hipDeviceSynchronize());
            for (auto k = I.waiting.lower_bound(std::make_pair(dev, (size_t) 0)); k != I.waiting.end() && k->first.first == dev; ++k) {
                std::vector<void *> &to = I.ready[k->first];
                to.insert(to.end(), k->second.begin(), k->second.end());
                k->second.clear();
            }
            it = I.ready.find(key);
        }
    }
    if (it != I.ready.end() && !it->second.empty()) {
        void *p = it->second.back();
        it->second.pop_back();
        I.total -= size;
        return p;
    }
    void *p = nullptr;
    hipError_t e = hipMalloc(&p, size);
    if (e == hipErrorOutOfMemory && I.total > 0) {
        (void) hipGetLastError();
        I.flush_locked();
        e = hipMalloc(&p, size);
    }
    TSVM_HIP_CHECK(e);
    return p;
}

void DevicePool::give(void *p, size_t bytes, int device, bool idle) {
    Impl &I = impl();
    const size_t size = Impl::block_size(bytes);
    std::lock_guard<std::mutex> lock(I.mu);
    if (size > Impl::MAX_BLOCK || I.total + size > Impl::MAX_TOTAL) {
        (void) hipFree(p);
        return;
    }
    (idle || Idle::depth() > 0 ? I.ready : I.waiting)[std::make_pair(device, size)].push_back(p);
    I.total += size;
}

void DevicePool::flush() {
    Impl &I = impl();
    std::lock_guard<std::mutex> lock(I.mu);
    I.flush_locked();
}

namespace {
// (as the pool above: never destroyed, emptied before the HIP runtime's tear-down)
struct HostPool {
    std::mutex mu;
    std::vector<PinnedBlock> pinned;
    std::map<int, std::vector<hipEvent_t>> events;   // by device
};
HostPool &host_pool() {
    static HostPool *h = [] {
        HostPool *n = new HostPool();
        atexit([] {
            HostPool &p = host_pool();
            std::lock_guard<std::mutex> lock(p.mu);
            for (const PinnedBlock &b : p.pinned) (void) hipHostFree(b.host);
            for (auto &kv : p.events)
                for (hipEvent_t e : kv.second) (void) hipEventDestroy(e);
            p.pinned.clear();
            p.events.clear();
        });
        return n;
    }();
    return *h;
}
constexpr size_t HOST_POOL_MAX = 64;   // blocks, and events per device, kept at most
}  // namespace

PinnedBlock take_pinned_block() {
    HostPool &h = host_pool();
    {
        std::lock_guard<std::mutex> lock(h.mu);
        if (!h.pinned.empty()) {
            const PinnedBlock b = h.pinned.back();
            h.pinned.pop_back();
            return b;
        }
    }
    PinnedBlock b;
    TSVM_HIP_CHECK(hipHostMalloc((void **) &b.host, PINNED_BLOCK, hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable));
    TSVM_HIP_CHECK(hipHostGetDevicePointer((void **) &b.dev, b.host, 0));
    return b;
}

void give_pinned_block(const PinnedBlock &b) {
    HostPool &h = host_pool();
    std::lock_guard<std::mutex> lock(h.mu);
    if (h.pinned.size() < HOST_POOL_MAX) h.pinned.push_back(b);
    else (void) hipHostFree(b.host);
}

const double *ResultBlock::wait_for(size_t count) {
    const volatile uint64_t *const word = (const volatile uint64_t *) block_.host;
    const auto start = std::chrono::steady_clock::now();
    size_t at = 0;
    for (unsigned spins = 1; at < count; ++spins) {
        if (word[at] != NOT_YET) {
            ++at;
        } else if (spins % 256 == 0 && std::chrono::steady_clock::now() - start > std::chrono::milliseconds(2)) {
            wait();   // (behind other work, or the kernels have failed)
            for (; at < count; ++at)
                if (word[at] == NOT_YET) throw std::runtime_error("ResultBlock: the kernels finished without a result");
        }
    }
    __atomic_thread_fence(__ATOMIC_ACQUIRE);
    arrived_ = true;
    return (const double *) block_.host;
}

DeviceEvent take_event() {
    HostPool &h = host_pool();
    DeviceEvent e;
    e.device = current_device();
    {
        std::lock_guard<std::mutex> lock(h.mu);
        std::vector<hipEvent_t> &v = h.events[e.device];
        if (!v.empty()) {
            e.event = v.back();
            v.pop_back();
            return e;
        }
    }
    TSVM_HIP_CHECK(hipEventCreateWithFlags(&e.event, hipEventDisableTiming));
    return e;
}

void give_event(const DeviceEvent &e) {
    HostPool &h = host_pool();
    {
        std::lock_guard<std::mutex> lock(h.mu);
        std::vector<hipEvent_t> &v = h.events[e.device];
        if (v.size() < HOST_POOL_MAX) {
            v.push_back(e.event);
            return;
        }
    }
    (void) hipEventDestroy(e.event);
}

void parallel_memcpy(void *to, const void *from, size_t bytes) {
    const size_t piece = (size_t) 256 << 10;
    if (bytes < 4 * piece) {
        memcpy(to, from, bytes);
        return;
    }
    const long n = (long) ((bytes + piece - 1) / piece);
    // (the whole team, also for fewer pieces: a team of another size than the last one's ends and starts threads)
#pragma omp parallel for schedule(static) num_threads(thread_limit())
    for (long i = 0; i < n; ++i) memcpy((char *) to + i * piece, (const char *) from + i * piece, std::min(piece, bytes - i * piece));
}

void wait_until_done(hipError_t (*state_of)(void *), void *thing, long long timeout_ms) {
    const auto start = std::chrono::steady_clock::now();
    for (;;) {
        const hipError_t e = state_of(thing);
        if (e == hipSuccess) return;
        if (e != hipErrorNotReady) TSVM_HIP_CHECK(e);
        if (std::chrono::steady_clock::now() - start > std::chrono::milliseconds(timeout_ms))
            throw std::runtime_error("no result from the device after " + std::to_string(timeout_ms) +
                                     " ms (TSVM_SOLVER_TIMEOUT_MS); the device may be hung");
    }
}

struct HostStaging::Impl {
    static constexpr int CHUNKS = 4;
    std::mutex mu;
    struct Chunk {
        char *host = nullptr;
        DeviceEvent pending;   // (no event: nothing is on its way)
    } chunk[CHUNKS];
    int next = 0;
    Chunk &take(long long timeout_ms = 0) {
        Chunk &c = chunk[next];
        next = (next + 1) % CHUNKS;
        if (!c.host) TSVM_HIP_CHECK(hipHostMalloc((void **) &c.host, CHUNK, hipHostMallocPortable));
        wait(c, timeout_ms);
        return c;
    }
    void wait(Chunk &c, long long timeout_ms) {   // (0: as long as it takes)
        if (!c.pending.event) return;
        if (timeout_ms > 0) wait_until_done([](void *e) { return hipEventQuery((hipEvent_t) e); }, c.pending.event, timeout_ms);
        else TSVM_HIP_CHECK(hipEventSynchronize(c.pending.event));
        give_event(c.pending);
        c.pending = DeviceEvent();
    }
    void record(Chunk &c, hipStream_t stream) {
        c.pending = take_event();
        TSVM_HIP_CHECK(hipEventRecord(c.pending.event, stream));
    }
};

HostStaging &HostStaging::instance() {
    static HostStaging s;
    return s;
}

HostStaging::Impl &HostStaging::impl() {
    static Impl *i = [] {   // (never destroyed; its memory goes back before the HIP runtime's tear-down)
        Impl *n = new Impl();
        atexit([] {
            Impl &I = HostStaging::instance().impl();
            std::lock_guard<std::mutex> lock(I.mu);
            for (Impl::Chunk &c : I.chunk) {
                if (c.host) (void) hipHostFree(c.host);
                c = Impl::Chunk();
            }
        });
        return n;
    }();
    return *i;
}

void HostStaging::upload(void *dst, size_t bytes, const std::function<void(char *, size_t, size_t)> &fill, hipStream_t stream) {
    Impl &I = impl();
    std::lock_guard<std::mutex> lock(I.mu);
    for (size_t off = 0; off < bytes; off += CHUNK) {
        const size_t len = std::min(CHUNK, bytes - off);
        Impl::Chunk &c = I.take();
        fill(c.host, off, len);
        TSVM_HIP_CHECK(hipMemcpyAsync((char *) dst + off, c.host, len, hipMemcpyHostToDevice, stream));
        I.record(c, stream);
    }
}

void HostStaging::upload(void *dst, const std::vector<Part> &parts, hipStream_t stream) {
    if (parts.empty()) return;
    upload(dst, parts.back().at + parts.back().bytes, [&](char *to, size_t off, size_t len) {
        for (const Part &p : parts) {
            const size_t lo = std::max(off, p.at), hi = std::min(off + len, p.at + p.bytes);
            if (lo < hi) parallel_memcpy(to + (lo - off), (const char *) p.from + (lo - p.at), hi - lo);
        }
    }, stream);
}

void HostStaging::download(const void *src, size_t bytes, const std::function<void(const char *, size_t, size_t)> &take, hipStream_t stream,
                           long long timeout_ms) {
    Impl &I = impl();
    std::lock_guard<std::mutex> lock(I.mu);
    struct Flying { Impl::Chunk *c; size_t off, len; };
    std::vector<Flying> queue;
    size_t head = 0, off = 0;
    while (head < queue.size() || off < bytes) {
        while (off < bytes && queue.size() - head < Impl::CHUNKS - 1) {
            const size_t len = std::min(CHUNK, bytes - off);
            Impl::Chunk &c = I.take(timeout_ms);
            TSVM_HIP_CHECK(hipMemcpyAsync(c.host, (const char *) src + off, len, hipMemcpyDeviceToHost, stream));
            I.record(c, stream);
            queue.push_back({&c, off, len});
            off += len;
        }
        const Flying f = queue[head++];
        I.wait(*f.c, timeout_ms);
        take(f.c->host, f.off, f.len);
    }
}

size_t &device_bytes_in_use() {
    static size_t bytes = 0;
    return bytes;
}

std::recursive_mutex &device_work_mutex() {
    static std::recursive_mutex m;
    return m;
}

RowArena &RowArena::instance() {
    static RowArena arena;
    return arena;
}

size_t RowArena::auto_budget() {
    if (full_budget_) return cap_;   // the arena already is the budget: never chase small changes in free memory
    size_t free_b = 0, total_b = 0;
    TSVM_HIP_CHECK(hipMemGetInfo(&free_b, &total_b));
    // Nine tenths of what is free or already held, unless TSVM_ARENA_PERCENT (10..95) says otherwise: kernel rows
    // are what the memory is for (hits grow in proportion to the slots; the set-up of a class pair or a prediction
    // takes a few GB at most, and partial sums of predictions come out of the arena itself).  On the seven-class and
    // the regression benchmark: half 1.80 s / 1.77 s, three quarters 1.71 / 1.63, 85 % 1.68 / 1.59 with the kernels
    // of that time; with the present ones three quarters 1.576 / 1.586 (hits 46.8 % / 37.7 %), nine tenths
    // 1.530 / 1.550 (50.9 % / 43.7 %).
    const char *e = getenv("TSVM_ARENA_PERCENT");
    const int asked = e ? atoi(e) : 90;
    const size_t pct = (size_t) (asked < 10 ? 10 : asked > 95 ? 95 : asked);
    return (free_b + cap_) / 100 * pct;
}

// The arena only ever grows.  Small requests (tests, small problems) get twice what they ask for, so
// that little is held and little has to be scrubbed by the driver when the process ends (giving back
// ~140 GB was measured to stall the next process on the device for 2-3 s).  A request above a quarter
// of the automatic budget takes the whole budget at once: a multi-class run then allocates a single
// time instead of releasing and re-allocating tens of gigabytes between its sub-problems, each release
// costing up to a second.
void *RowArena::acquire(size_t bytes, bool auto_sized) {
    if (bytes <= cap_) return ptr_;
    size_t want = bytes;
    bool take_all = false;
    if (auto_sized) {
        const size_t budget = auto_budget();
        take_all = bytes > budget / 4;
        want = take_all ? std::max(bytes, budget) : std::max(bytes * 2, cap_ + cap_ / 2);
    }
    release();
    hipError_t e = hipMalloc(&ptr_, want);
    if (e == hipErrorOutOfMemory) {   // (what other buffers have left in the pool may be what is missing)
        (void) hipGetLastError();
        DevicePool::instance().flush();
        e = hipMalloc(&ptr_, want);
    }
    TSVM_HIP_CHECK(e);
    cap_ = want;
    full_budget_ = take_all;
    static bool registered = false;
    if (!registered) {
        registered = true;
        atexit([] { RowArena::instance().release(); });
    }
    return ptr_;
}

void RowArena::release() {
    if (ptr_) (void) hipFree(ptr_);
    ptr_ = nullptr;
    cap_ = 0;
    full_budget_ = false;
}
}  // namespace tsvm

// Dense rows cost d_pad MFMA k-steps per output, CSR rows cost one L2 gather per stored non-zero;
// the matrix cores run roughly 30 k-steps in the time of one gather, so dense wins unless rows
// are very sparse.  Dense storage is also capped at 64 GiB.
bool KernelMatrix::choose_dense(size_t n, size_t n_features, size_t nnz) {
    if (n == 0) return true;
    const size_t ld = (n_features + 7) / 8 * 8;
    const double avg = (double) nnz / (double) n;
    if ((double) ld * (double) n * 8.0 > 64.0 * 1024 * 1024 * 1024) return false;
    return (double) ld <= 32.0 * std::max(avg, 1.0);
}

// The reference's CSR arrays (kernelmatrix.cpp:183-207): n_features = largest feature id + 1, ids kept as given; self dot
// products from the CSR values in stored order; then the layout is chosen.
std::shared_ptr<DeviceRows> DeviceRows::from_host(const RowStore &rows) {
    auto out = std::make_shared<DeviceRows>();
    DeviceRows &r = *out;
    r.n = rows.size();
    r.nnz = rows.nnz();
    const int64_t first = rows.ptr()[0];
    const int *const col = rows.col() + first;
    const kernel_type *const val = rows.val() + first;
    int max_index = 0, all_float = 1, all_finite = 1;
#pragma omp parallel for schedule(static) reduction(max : max_index) reduction(min : all_float, all_finite) num_threads(threads_for(r.nnz))
    for (size_t e = 0; e < r.nnz; ++e) {
        max_index = std::max(max_index, col[e]);
        all_float = (double) (float) val[e] != (double) val[e] ? 0 : all_float;
        all_finite = val[e] - val[e] == 0 ? all_finite : 0;
    }
    r.n_features = (size_t) max_index + 1;
    r.values_fit_float = all_float != 0;
    r.values_finite = all_finite != 0;
    r.dense = KernelMatrix::choose_dense(r.n, r.n_features, r.nnz);
    if (!r.dense) {
        // (an entry whose column is not larger than the one's before may only be one where a row begins)
        const int64_t *const at = rows.ptr();
        int64_t descents = 0, at_starts = 0;
#pragma omp parallel num_threads(threads_for(r.nnz))
        {
#pragma omp for schedule(static) reduction(+ : descents) nowait
            for (size_t e = 1; e < r.nnz; ++e) descents += col[e] <= col[e - 1];
#pragma omp for schedule(static) reduction(+ : at_starts)
            for (size_t i = 0; i < r.n; ++i) {
                const int64_t e = at[i] - first;
                at_starts += e > 0 && at[i + 1] > at[i] && col[e] <= col[e - 1];
            }
        }
        r.columns_ascend = descents == at_starts;
    }
    tsvm::HostStaging &staging = tsvm::HostStaging::instance();
    std::vector<int64_t> ptr;
    const int64_t *host_ptr = rows.ptr();
    if (first != 0 || !r.dense) {
        ptr.assign(rows.ptr(), rows.ptr() + r.n + 1);
        for (int64_t &p : ptr) p -= first;
        host_ptr = ptr.data();
    }
    r.self_dot.resize(r.n);
    if (r.dense) {
        // one upload of the three arrays, which are not needed any more once they are a matrix
        const size_t val_bytes = r.nnz * sizeof(kernel_type), ptr_bytes = (r.n + 1) * sizeof(int64_t), col_bytes = r.nnz * sizeof(int);
        tsvm::DeviceBuffer<char> csr(ptr_bytes + val_bytes + col_bytes);
        std::vector<tsvm::HostStaging::Part> parts{{host_ptr, ptr_bytes, 0}};
        if (r.nnz) {
            parts.push_back({val, val_bytes, ptr_bytes});
            parts.push_back({col, col_bytes, ptr_bytes + val_bytes});
        }
        staging.upload(csr.data(), parts, tsvm::work_stream());
        r.ld = (int64_t) ((r.n_features + 7) / 8 * 8);
        r.x.resize(r.n * (size_t) r.ld);
        abi_check(tsvm_csr_rows_to_dense((const kernel_type *) (csr.data() + ptr_bytes), (const int *) (csr.data() + ptr_bytes + val_bytes),
                                         (const int64_t *) csr.data(), (int64_t) r.n, r.x.data(), r.ld, r.self_dot.data(), tsvm::work_stream()));
        csr.release();
        // indicator columns are a run that ends with the last column: one other value there, in most data sets the
        // first, and there are none (a few of the entries are looked at here, all of them by the device's count)
        bool last_is_indicator = true;
        for (size_t e = 0; e < std::min<size_t>(r.nnz, 16384) && last_is_indicator; ++e)
            if (col[e] == max_index && val[e] != 0.0 && val[e] != 1.0) last_is_indicator = false;
        if (last_is_indicator) r.find_indicator_columns();
    } else {
        r.val.resize(r.nnz);
        r.col.resize(r.nnz);
        r.row_ptr.resize(r.n + 1);
        if (r.nnz) {
            staging.upload(r.val.data(), {{val, r.nnz * sizeof(kernel_type), 0}}, tsvm::work_stream());
            staging.upload(r.col.data(), {{col, r.nnz * sizeof(int), 0}}, tsvm::work_stream());
        }
        staging.upload(r.row_ptr.data(), {{host_ptr, (r.n + 1) * sizeof(int64_t), 0}}, tsvm::work_stream());
        abi_check(tsvm_csr_self_dot(r.val.data(), r.row_ptr.data(), (int64_t) r.n, r.self_dot.data(), tsvm::work_stream()));
        r.host_row_ptr = std::move(ptr);
        r.build_sliced();
    }
    return out;
}

// The sliced copy of CSR rows (row offsets are known on the host).
void DeviceRows::build_sliced() {
    sliced_lds = 0;
    max_row_nnz = 0;
    if (dense || n == 0 || getenv("TSVM_NO_SLICED")) return;
    for (size_t i = 0; i < n; ++i) max_row_nnz = std::max(max_row_nnz, (int) (host_row_ptr[i + 1] - host_row_ptr[i]));
    const int vt = values_fit_float ? TSVM_ROW_F32 : TSVM_ROW_F64;
    const size_t need = tsvm_get_rows_csr_sliced_lds((int) n_features, max_row_nnz, vt);
    if (need == 0) return;
    const size_t n_slices = (n + 63) / 64;
    std::vector<int64_t> sp(n_slices + 1, 0);
    for (size_t s = 0; s < n_slices; ++s) {
        int64_t w = 0;
        for (size_t i = s * 64; i < std::min(n, s * 64 + 64); ++i) w = std::max(w, host_row_ptr[i + 1] - host_row_ptr[i]);
        sp[s + 1] = sp[s] + 64 * w;
    }
    // (a few very long rows would blow the padded copy up: then the plain CSR kernel stays in charge)
    if ((size_t) sp[n_slices] > 4 * nnz + 64 * n_slices) return;
    if (sp[n_slices] == 0) return;   // every row is empty: nothing to slice, the plain kernel writes kappa(0, 0)
    slice_ptr.upload(sp);
    ell_col.resize((size_t) sp[n_slices]);
    ell_val.resize((size_t) sp[n_slices] * (values_fit_float ? sizeof(float) : sizeof(double)));
    abi_check(tsvm_csr_to_sliced(val.data(), col.data(), row_ptr.data(), (int64_t) n, slice_ptr.data(), (int) n_features, ell_col.data(),
                                 ell_val.data(), vt, tsvm::work_stream()));
    sliced_lds = need;
}

std::shared_ptr<DeviceRows> DeviceRows::subset(const DeviceRows &base, const int *rows, size_t n_rows, const SvmParam *param, kernel_type *diag) {
    auto out = std::make_shared<DeviceRows>();
    DeviceRows &r = *out;
    r.n = n_rows;
    r.n_features = base.n_features;
    r.dense = base.dense;
    r.values_fit_float = base.values_fit_float;
    r.values_finite = base.values_finite;
    r.columns_ascend = base.columns_ascend;
    r.ld = base.ld;
    const bool by_value = base.dense && n_rows <= (size_t) tsvm_subset_rows_dense_max_ids((int64_t) base.n);
    tsvm::DeviceBuffer<int> d_rows(by_value ? 0 : n_rows);
    d_rows.upload(rows, d_rows.size());
    r.self_dot.resize(n_rows);
    if (base.dense) {
        r.x.resize(n_rows * (size_t) r.ld);
        r.nnz = n_rows ? base.nnz / std::max<size_t>(base.n, 1) * n_rows : 0;   // estimate, informational only
        if (base.ind_first >= 0) {   // indicator columns of all rows are indicator columns of a subset (masks move as 8-byte words)
            r.ind_first = base.ind_first;
            r.ind_max_ones = base.ind_max_ones;
            r.ind_mask.resize(n_rows);
        }
        const SvmParam kernel = param ? *param : SvmParam();
        abi_check(tsvm_subset_rows_dense(base.x.data(), base.ld, by_value ? rows : d_rows.data(), (int64_t) n_rows, base.self_dot.data(),
                                         r.ind_first >= 0 ? base.ind_mask.data() : nullptr, r.x.data(), r.self_dot.data(), r.ind_mask.data(),
                                         (int) kernel.kernel_type, kernel.gamma, kernel.coef0, kernel.degree, diag, by_value, tsvm::work_stream()));
    } else {
        abi_check(tsvm_gather_f64(base.self_dot.data(), d_rows.data(), (int) n_rows, r.self_dot.data(), tsvm::work_stream()));
        if (diag)
            abi_check(tsvm_kernel_diag(r.self_dot.data(), (int64_t) n_rows, (int) param->kernel_type, param->gamma, param->coef0,
                                       param->degree, diag, tsvm::work_stream()));
        r.host_row_ptr.assign(n_rows + 1, 0);
        for (size_t i = 0; i < n_rows; ++i)
            r.host_row_ptr[i + 1] = r.host_row_ptr[i] + base.host_row_ptr[rows[i] + 1] - base.host_row_ptr[rows[i]];
        r.nnz = (size_t) r.host_row_ptr[n_rows];
        r.row_ptr.upload(r.host_row_ptr);
        r.val.resize(r.nnz);
        r.col.resize(r.nnz);
        abi_check(tsvm_csr_gather_rows(base.val.data(), base.col.data(), base.row_ptr.data(), d_rows.data(), (int64_t) n_rows,
                                       r.row_ptr.data(), r.val.data(), r.col.data(), tsvm::work_stream()));
        r.build_sliced();
    }
    return out;
}

const std::vector<int> &DeviceRows::column_stats() const {
    if (column_stats_.size() != 2 * n_features) {
        tsvm::DeviceBuffer<int> d_counts(2 * n_features);
        if (dense) abi_check(tsvm_column_stats_dense(x.data(), ld, (int64_t) n, (int) n_features, d_counts.data(), tsvm::work_stream()));
        else abi_check(tsvm_column_stats_csr(val.data(), col.data(), (int64_t) nnz, (int) n_features, d_counts.data(), tsvm::work_stream()));
        column_stats_ = d_counts.to_host();
    }
    return column_stats_;
}

// The trailing run of columns whose values are all 0 or 1 (at most 64 of them): its first column, n_features when
// the last column is not such a column.  stats: the 2 * n_features counts of column_stats().
int DeviceRows::indicator_run_start(const int *stats, int n_features) {
    int first = n_features;
    while (first > 0 && n_features - first < 64 && stats[n_features + first - 1] == 0) --first;
    return first;
}

// Leaving the run to the kernel's epilogue pays when it saves more than the additions cost there: one 4-column step
// of the matrix cores per value is worth about one epilogue instruction, an indicator column that may match about three.
bool DeviceRows::indicator_run_pays(int n_features, int first, int max_ones) {
    const int steps_saved = (n_features + 3) / 4 - (first + 3) / 4;
    return steps_saved >= 2 + 3 * max_ones;
}

void DeviceRows::find_indicator_columns() {
    ind_first = -1;
    if (!dense || n == 0 || n_features == 0 || getenv("TSVM_NO_INDICATOR")) return;
    const std::vector<int> &stats = column_stats();
    const int first = indicator_run_start(stats.data(), (int) n_features);
    if (first == (int) n_features) return;
    tsvm::DeviceBuffer<uint64_t> masks(n);
    tsvm::DeviceBuffer<int> d_max(1);
    abi_check(tsvm_indicator_masks(x.data(), ld, (int64_t) n, first, (int) n_features - first, masks.data(), d_max.data(), tsvm::work_stream()));
    const int max_ones = d_max.to_host()[0];
    if (!indicator_run_pays((int) n_features, first, max_ones)) return;
    ind_first = first;
    ind_max_ones = max_ones;
    ind_mask = std::move(masks);
}

std::shared_ptr<DeviceRows> DeviceRows::of(const DataSet &dataset) {
    std::shared_ptr<void> &slot = dataset.device_cache();
    if (!slot) slot = from_host(dataset.rows());
    return std::static_pointer_cast<DeviceRows>(slot);
}

KernelMatrix::KernelMatrix(const RowStore &rows, SvmParam param) : param(param) {
    rows_ = DeviceRows::from_host(rows);
    finish(1);
}

KernelMatrix::KernelMatrix(const DataSet &dataset, const int *rows, size_t n_rows, SvmParam param, int repeat)
    : param(param) {
    std::shared_ptr<DeviceRows> all = DeviceRows::of(dataset);
    if (rows) diag_.resize(n_rows * repeat);
    rows_ = rows ? DeviceRows::subset(*all, rows, n_rows, &this->param, diag_.data()) : all;
    finish(repeat, rows != nullptr);
}

// diag from the self dot products (kernelmatrix.cpp:225-247).  With repeat > 1 the reference stacks the
// same rows several times (the 2n-row problem of SVR, svr.cpp:14-15); here the rows are stored once and
// only the diagonal, which the solver kernels index by instance id, is replicated.
void KernelMatrix::finish(int repeat, bool have_diag) {
    n_unique_ = rows_->n;
    repeat_ = repeat;
    if (!have_diag) {
        diag_.resize(n_unique_ * repeat_);
        abi_check(tsvm_kernel_diag(rows_->self_dot.data(), (int64_t) n_unique_, (int) param.kernel_type, param.gamma, param.coef0,
                                   param.degree, diag_.data(), tsvm::work_stream()));
    }
    for (int rep = 1; rep < repeat_; ++rep)
        TSVM_HIP_CHECK(hipMemcpyAsync(diag_.data() + rep * n_unique_, diag_.data(), n_unique_ * sizeof(kernel_type),
                                      hipMemcpyDeviceToDevice, tsvm::work_stream()));
}

size_t KernelMatrix::reference_syncmem_bytes() const {
    const DeviceRows &R = *rows_;
    const std::vector<int> &stats = R.column_stats();
    const long long nf = (long long) R.n_features, m = (long long) n_instances();
    std::vector<long long> cnt(nf);
    long long entries = 0;
    for (long long c = 0; c < nf; ++c) {
        cnt[c] = (long long) stats[c] * repeat_;
        entries += cnt[c];
    }
    // columns by entry count ascending, ties by index (kernelmatrix.cpp:32-41); leading columns go to the sparse part
    // while the part stays under 5 % full, the column under 50 % full, and four times its entries do not exceed
    // the cells left to the dense part (kernelmatrix.cpp:58-74)
    std::vector<int> order(nf);
    for (long long c = 0; c < nf; ++c) order[c] = (int) c;
    std::sort(order.begin(), order.end(), [&](int a, int b) { return cnt[a] != cnt[b] ? cnt[a] < cnt[b] : a < b; });
    long long total_csr = 0, total_dense = m * nf, row_sum = 0, dense_cols = nf, nnz_sparse = 0;
    for (long long i = 0; i < nf; ++i) {
        const long long c = cnt[order[i]];
        total_csr += c;
        total_dense -= m;
        row_sum += m;
        if ((long double) total_csr / row_sum > 0.05 || (long double) c / m > 0.5 || total_csr * 4 > total_dense) break;
        --dense_cols;
        nnz_sparse += c;
    }
    size_t bytes = (size_t) entries * (sizeof(kernel_type) + sizeof(int)) + (size_t) (m + 1) * sizeof(int) +
                   2 * (size_t) m * sizeof(kernel_type);
    if (dense_cols > 0) bytes += (size_t) m * dense_cols * sizeof(kernel_type);                      // dense.val, kernelmatrix.cpp:79-83
    if (dense_cols < nf && nnz_sparse != 0)   // some entry lies outside the dense part (kernelmatrix.cpp:151-176)
        bytes += (size_t) nnz_sparse * (sizeof(kernel_type) + sizeof(int)) + (size_t) (m + 1) * sizeof(int);
    return bytes;
}

size_t KernelMatrix::reference_syncmem_bytes_at_most(size_t m, size_t n_features, size_t entries) {
    // every stored entry counted twice (in the CSR arrays and in the sparse part), every column in the dense part
    return 2 * entries * (sizeof(kernel_type) + sizeof(int)) + 2 * (m + 1) * sizeof(int) + 2 * m * sizeof(kernel_type) +
           m * n_features * sizeof(kernel_type);
}

size_t KernelMatrix::entries_at_most() const {   // (a gathered dense subset's entry count is an estimate: every cell then)
    return rows_->dense ? n_instances() * n_features() : rows_->nnz * repeat_;
}

// A staging buffer that is all-zero whenever it is not in use: grown (and cleared) only when a call needs more.
static void grow_zeroed(tsvm::DeviceBuffer<unsigned char> &b, size_t bytes, hipStream_t stream) {
    if (b.size() >= bytes) return;
    b.resize(bytes);
    TSVM_HIP_CHECK(hipMemsetAsync(b.data(), 0, bytes, stream));
}

void KernelMatrix::get_rows(const int *d_idx, int m, void *d_out, int64_t ld, const int *d_out_slots,
                            hipStream_t stream) const {
    const DeviceRows &R = *rows_;
    const int n = (int) n_unique_;
    if (R.dense && R.ind_first >= 0) {
        abi_check(tsvm_get_rows_dense_indicator(R.x.data(), R.ld, nullptr, n, R.ind_first, R.self_dot.data(), R.ind_mask.data(),
                                                R.x.data(), R.ld, d_idx, m, nullptr, R.self_dot.data(), R.ind_mask.data(),
                                                R.ind_max_ones, (int) param.kernel_type, param.gamma, param.coef0, param.degree,
                                                d_out, row_type(), d_out_slots, ld, stream));
        return;
    }
    if (R.dense) {
        abi_check(tsvm_get_rows_dense(R.x.data(), R.ld, nullptr, n, (int) R.n_features, R.self_dot.data(), R.x.data(), R.ld, d_idx,
                                      m, R.self_dot.data(), (int) param.kernel_type, param.gamma, param.coef0, param.degree,
                                      d_out, row_type(), d_out_slots, ld, stream));
        return;
    }
    const int wt = R.values_fit_float ? TSVM_ROW_F32 : TSVM_ROW_F64;
    if (R.sliced_lds) {   // the stored rows streamed once per sixteen working rows, the working rows in LDS
        abi_check(tsvm_get_rows_csr_sliced(R.ell_col.data(), R.ell_val.data(), wt, R.slice_ptr.data(), n, R.self_dot.data(),
                                           R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, R.self_dot.data(),
                                           (int) R.n_features, R.max_row_nnz, (int) param.kernel_type, param.gamma, param.coef0,
                                           param.degree, d_out, row_type(), d_out_slots, ld, stream));
        return;
    }
    // The staging matrix [n_features][m] is kept all-zero between uses: the working rows' non-zeros are written
    // into it and taken out again afterwards (nnz entries each way instead of a fill of n_features x m).
    grow_zeroed(stage_w_, (size_t) m * R.n_features * (R.values_fit_float ? sizeof(float) : sizeof(double)), stream);
    if (stage_sd_.size() < (size_t) m) stage_sd_.resize(m);
    abi_check(tsvm_csr_scatter_rows(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, (int) R.n_features,
                                    stage_w_.data(), wt, 0, stream));
    abi_check(tsvm_gather_f64(R.self_dot.data(), d_idx, m, stage_sd_.data(), stream));
    abi_check(tsvm_get_rows_csr_staged(R.val.data(), R.col.data(), R.row_ptr.data(), nullptr, n, R.self_dot.data(),
                                       stage_w_.data(), wt, m, stage_sd_.data(), (int) param.kernel_type, param.gamma,
                                       param.coef0, param.degree, d_out, row_type(), d_out_slots, ld, stream));
    abi_check(tsvm_csr_scatter_rows(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, (int) R.n_features,
                                    stage_w_.data(), wt, 1, stream));
}

void KernelMatrix::get_rows_counted(const int *d_idx, int m_max, const int *d_m, void *d_out, int64_t ld,
                                    const int *d_out_slots, hipStream_t stream) const {
    const DeviceRows &R = *rows_;
    if (!R.dense) throw std::logic_error("KernelMatrix::get_rows_counted: dense layout only");
    if (R.ind_first >= 0) {
        abi_check(tsvm_get_rows_dense_indicator(R.x.data(), R.ld, nullptr, (int) n_unique_, R.ind_first, R.self_dot.data(),
                                                R.ind_mask.data(), R.x.data(), R.ld, d_idx, m_max, d_m, R.self_dot.data(),
                                                R.ind_mask.data(), R.ind_max_ones, (int) param.kernel_type, param.gamma,
                                                param.coef0, param.degree, d_out, row_type(), d_out_slots, ld, stream));
        return;
    }
    abi_check(tsvm_get_rows_dense_counted(R.x.data(), R.ld, nullptr, (int) n_unique_, (int) R.n_features, R.self_dot.data(),
                                          R.x.data(), R.ld, d_idx, m_max, d_m, R.self_dot.data(), (int) param.kernel_type,
                                          param.gamma, param.coef0, param.degree, d_out, row_type(), d_out_slots, ld, stream));
}

// Staging matrices of up to this size come in pairs, so that one's rows are taken out by the launch that puts the next block's into the
// other.  It is a launch of 1 to 3 us that this saves, and nothing once the matrix is larger than the caches, where the two cost
// more than the launch: the block of 1,024 rows of 3,000 features (floats, 12 MB) 26.4 us with two, 27.7 with one, of 21,000 (86 MB)
// 32.2 / 33.4, doubles (172 MB) 49.1 / 48.0, of 200,000 (819 MB) 38.5 / 35.3.  A row cache takes nine tenths of what memory is free before
// the first block is asked for: of 3.2 million features one matrix is 13 GB, and a second need not fit.
constexpr size_t STAGE_TURNS_MAX = (size_t) 128 << 20;

// K(x_idx[r], x_idx[t]) for r, t < m: the same kernels with the column set restricted to the m rows,
// so every value is bit-identical to the corresponding entry of a full kernel row.  Elements are row_type() wide.
void KernelMatrix::get_block(const int *d_idx, int m, void *d_out, int64_t ld, hipStream_t stream) const {
    const DeviceRows &R = *rows_;
    if (R.dense) {
        abi_check(tsvm_get_rows_dense(R.x.data(), R.ld, d_idx, m, (int) R.n_features, R.self_dot.data(), R.x.data(), R.ld, d_idx, m,
                                      R.self_dot.data(), (int) param.kernel_type, param.gamma, param.coef0, param.degree,
                                      d_out, row_type(), nullptr, ld, stream));
        return;
    }
    const int wt = R.values_fit_float ? TSVM_ROW_F32 : TSVM_ROW_F64;
    const size_t bytes = (size_t) m * R.n_features * (R.values_fit_float ? sizeof(float) : sizeof(double));
    // K(r, t) is K(t, r) to the last bit unless a value times an absent (zero) one is not zero, or the two rows' common features come in two orders
    if (R.values_finite && R.columns_ascend && R.nnz > 0) {
        if (turn_[turn_now_].m != 0) throw std::logic_error("KernelMatrix::get_block: rows in the staging matrix");
        bool turns = std::max(bytes, turn_[turn_now_].w.size()) <= STAGE_TURNS_MAX && !one_stage_;
        try {
            grow_zeroed(turn_[turn_now_].w, bytes, stream);
        } catch (const std::bad_alloc &) {
            BlockStage &first = turn_[turn_now_ ^ 1];
            if (first.w.size() < bytes) throw;
            (void) hipGetLastError();   // no room for a second one: the first has to do from now on
            if (first.m) abi_check(tsvm_csr_scatter_rows(R.val.data(), R.col.data(), R.row_ptr.data(), first.ids.data(), first.m, (int) R.n_features,
                                                         first.w.data(), wt, 1, stream));
            first.m = 0;
            turn_now_ ^= 1;
            one_stage_ = true;
            turns = false;
        }
        BlockStage &now = turn_[turn_now_], &last = turn_[turn_now_ ^ 1];
        if (now.ids.size() < (size_t) m) now.ids.resize(m);
        abi_check(tsvm_csr_block(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, R.self_dot.data(), now.w.data(), now.ids.data(), last.w.data(),
                                 last.ids.data(), last.m, wt, (int) param.kernel_type, param.gamma, param.coef0, param.degree, d_out, row_type(), ld, stream));
        last.m = 0;
        if (turns) {
            now.m = m;
            turn_now_ ^= 1;
        } else {
            abi_check(tsvm_csr_scatter_rows(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, (int) R.n_features, now.w.data(), wt, 1, stream));
        }
        return;
    }
    // kept all-zero between uses, as in get_rows
    grow_zeroed(stage_blk_, bytes, stream);
    if (stage_blk_sd_.size() < (size_t) m) stage_blk_sd_.resize(m);
    abi_check(tsvm_csr_scatter_rows(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, (int) R.n_features,
                                    stage_blk_.data(), wt, 0, stream));
    abi_check(tsvm_gather_f64(R.self_dot.data(), d_idx, m, stage_blk_sd_.data(), stream));
    abi_check(tsvm_get_rows_csr_staged(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, R.self_dot.data(),
                                       stage_blk_.data(), wt, m, stage_blk_sd_.data(), (int) param.kernel_type, param.gamma,
                                       param.coef0, param.degree, d_out, row_type(), nullptr, ld, stream));
    abi_check(tsvm_csr_scatter_rows(R.val.data(), R.col.data(), R.row_ptr.data(), d_idx, m, (int) R.n_features,
                                    stage_blk_.data(), wt, 1, stream));
}

constexpr size_t READ_FROM_HOST = 4096;   // entries

// The batch goes to the device as CSR (flattened by all cores into pinned memory, copied asynchronously) together
// with its rows' self dot products; with dense stored rows it is also laid out as a dense matrix of the stored rows'
// width (columns >= n_features are dropped from the products, kernelmatrix.cpp:392, but stay in the self dot).
KernelMatrix::StagedBatch KernelMatrix::stage_batch(const RowStore &batch, size_t first, size_t n_rows) const {
    const DeviceRows &R = *rows_;
    const int m = (int) n_rows;
    TSVM_HIP_CHECK(hipStreamSynchronize(tsvm::work_stream()));   // a previous batch's copies have left the staging memory
    h_ptr_.reserve((size_t) m + 1);
    int64_t *ptr = h_ptr_.data();
    const int64_t e0 = batch.ptr()[first];
    for (int r = 0; r <= m; ++r) ptr[r] = batch.ptr()[first + r] - e0;
    const size_t total = (size_t) ptr[m];
    h_val_.reserve(total);
    h_col_.reserve(total);
    kernel_type *val = h_val_.data();
    int *col = h_col_.data();
    const kernel_type *const from_val = batch.val() + e0;
    const int *const from_col = batch.col() + e0;
    // (indicator columns of the stored rows: the batch can use them when its own values there are zeros and ones)
    const int ind_lo = R.ind_first >= 0 ? R.ind_first : 0x7fffffff, ind_hi = (int) R.n_features;
    int not_indicator = 0;
#pragma omp parallel for schedule(static) reduction(max : not_indicator) num_threads(threads_for(total))
    for (size_t e = 0; e < total; ++e) {
        val[e] = from_val[e];
        col[e] = from_col[e];
        if (col[e] >= ind_lo && col[e] < ind_hi && val[e] != 0.0 && val[e] != 1.0) not_indicator = 1;
    }
    if (stage_sd_.size() < (size_t) m) stage_sd_.resize(m);
    StagedBatch out;
    out.sd = stage_sd_.data();
    out.indicator_values = R.ind_first >= 0 && !not_indicator;
    // A request of a few rows is read by the kernel where it is, in page-locked host memory: three copies of a microsecond's work
    // cost 5 us each.  However many rows the entries are spread over: 4,000 rows of one entry 82 us (as copies 100), 3,900
    // entries over 16,000 rows 235 (276), over 65,536 rows 283 (296); rows without any entry 203 (196) and 269 (229).
    const kernel_type *d_val = val;
    const int *d_col = col;
    const int64_t *d_ptr = ptr;
    if (!R.dense || total > READ_FROM_HOST) {
        if (b_val_.size() < total) { b_val_.resize(total); b_col_.resize(total); }
        if (b_ptr_.size() < (size_t) m + 1) b_ptr_.resize(m + 1);
        if (total) {
            TSVM_HIP_CHECK(hipMemcpyAsync(b_val_.data(), val, total * sizeof(kernel_type), hipMemcpyHostToDevice, tsvm::work_stream()));
            TSVM_HIP_CHECK(hipMemcpyAsync(b_col_.data(), col, total * sizeof(int), hipMemcpyHostToDevice, tsvm::work_stream()));
        }
        TSVM_HIP_CHECK(hipMemcpyAsync(b_ptr_.data(), ptr, ((size_t) m + 1) * sizeof(int64_t), hipMemcpyHostToDevice, tsvm::work_stream()));
        d_val = b_val_.data();
        d_col = b_col_.data();
        d_ptr = b_ptr_.data();
    }
    if (R.dense) {
        if (stage_.size() < (size_t) m * R.ld) stage_.resize((size_t) m * R.ld);
        abi_check(tsvm_csr_rows_to_dense(d_val, d_col, d_ptr, m, stage_.data(), R.ld, stage_sd_.data(), tsvm::work_stream()));
        out.a = stage_.data();
        out.lda = R.ld;
    } else {
        abi_check(tsvm_csr_self_dot(d_val, d_ptr, m, stage_sd_.data(), tsvm::work_stream()));
    }
    return out;
}

// External batch (kernelmatrix.cpp:281-312, 385-406).
void KernelMatrix::get_rows(const RowStore &batch, size_t first, size_t n_rows, void *d_out, int64_t ld) const {
    const DeviceRows &R = *rows_;
    const int m = (int) n_rows;
    if (m == 0) return;
    const StagedBatch b = stage_batch(batch, first, n_rows);
    const int n = (int) n_unique_;
    if (R.dense) {
        abi_check(tsvm_get_rows_dense(R.x.data(), R.ld, nullptr, n, (int) R.n_features, R.self_dot.data(), b.a, b.lda, nullptr, m,
                                      b.sd, (int) param.kernel_type, param.gamma, param.coef0, param.degree,
                                      d_out, row_type(), nullptr, ld, tsvm::work_stream()));
        return;
    }
    // The batch's rows wait in LDS, sixteen at a time, and the support vectors' sliced copy streams by, as in training; a batch
    // with a row too long for that or without any entry is staged as a dense matrix, and so is any batch when a support vector holds an infinity
    // or NaN, whose product with an absent (zero) feature is not zero.  Kernel values of text rows, staged / sliced, us: 6,000
    // support vectors 71 / 25 for one row, 98 / 32 for 64, 228 / 73 for 1,000, 1,159 / 221 for 4,099; 800 support vectors 25 / 25,
    // 28 / 31, 68 / 33, 322 / 64; 3,000 33 / 25, 40 / 34, 137 / 44, 680 / 146: few of them fill few workgroups, so few rows go
    // the staged way there.
    const int wt = R.values_fit_float ? TSVM_ROW_F32 : TSVM_ROW_F64;
    int longest = 0;
    for (int r = 0; r < m; ++r) longest = std::max(longest, (int) (h_ptr_.data()[r + 1] - h_ptr_.data()[r]));
    if (longest > 0 && R.sliced_lds && R.values_finite && (n >= 3072 || m >= 256) && tsvm_get_rows_csr_sliced_lds((int) R.n_features, longest, wt) > 0) {
        abi_check(tsvm_get_rows_csr_sliced(R.ell_col.data(), R.ell_val.data(), wt, R.slice_ptr.data(), n, R.self_dot.data(),
                                           b_val_.data(), b_col_.data(), b_ptr_.data(), nullptr, m, b.sd, (int) R.n_features, longest,
                                           (int) param.kernel_type, param.gamma, param.coef0, param.degree, d_out, row_type(), nullptr, ld,
                                           tsvm::work_stream()));
        return;
    }
    if (stage_.size() < (size_t) m * R.n_features) stage_.resize((size_t) m * R.n_features);
    abi_check(tsvm_csr_stage_rows(b_val_.data(), b_col_.data(), b_ptr_.data(), nullptr, m, (int) R.n_features,
                                  stage_.data(), tsvm::work_stream()));
    abi_check(tsvm_get_rows_csr(R.val.data(), R.col.data(), R.row_ptr.data(), nullptr, n, R.self_dot.data(), stage_.data(), m,
                                b.sd, (int) param.kernel_type, param.gamma, param.coef0, param.degree,
                                d_out, row_type(), nullptr, ld, tsvm::work_stream()));
}
