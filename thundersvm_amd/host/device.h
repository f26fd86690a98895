// Device memory and error plumbing of the host layer.  DeviceBuffer<T> is the native replacement
// for the reference's SyncArray<T> on this path: it owns device memory only, and every transfer is
// an explicit call (the reference's implicit host_data()/device_data() mirroring,
// src/thundersvm/syncmem.cpp:58-108, is what forces a device-host round trip per solver iteration).
#pragma once
#include <functional>
#include <mutex>
#include <hip/hip_runtime.h>

#include <new>
#include <stdexcept>
#include <string>
#include <vector>

#include "../../include/thundersvm_amd.h"

namespace tsvm {

inline void hip_check(hipError_t e, const char *what) {
    if (e == hipSuccess) return;
    if (e == hipErrorOutOfMemory) throw std::bad_alloc();   // include/thundersvm/util/common.h:33-39
    throw std::runtime_error(std::string(what) + ": " + hipGetErrorString(e));
}
#define TSVM_HIP_CHECK(expr) ::tsvm::hip_check((expr), #expr)

// Status of a C-ABI kernel call -> exception (2 == hipErrorOutOfMemory).
inline void abi_check(int rc) {
    if (rc == 0) return;
    if (rc == 2) throw std::bad_alloc();
    throw std::runtime_error(std::string("thundersvm_amd kernel call failed: ") + tsvm_last_error());
}

// The stream that everything outside a solve's own streams is enqueued on: uploads, row layouts, prediction.  One per
// device and process, independent of the default stream (whose work would wait for, and hold up, every class pair that
// is being solved).
hipStream_t work_stream();

// Device blocks that buffers have released, kept for the next buffer of about the same size: hipMalloc and hipFree cost
// microseconds to milliseconds each (hipFree waits for the device), and a small training run makes some forty of them.
// Blocks are rounded up to quarter powers of two; blocks above 256 MiB and whatever would take the pool over 2 GiB go
// back to the driver, everything does when the device runs out of memory, on tsvm_release_device_cache() and when the
// process ends.  A block is handed out again only after the device has been idle since its release (as hipFree would
// have waited for), unless whoever released it knows that nothing uses it any more (`idle`).  One list per device, a
// block's own, whichever is current when it is released; any number of threads.
class DevicePool {
public:
    static DevicePool &instance();
    void *take(size_t bytes, int *device);   // *device: the current device, whose memory it is
    void give(void *p, size_t bytes, int device, bool idle);
    void flush();
    // While one exists on a thread, what the thread releases counts as idle.
    struct Idle {
        Idle() { ++depth(); }
        ~Idle() { --depth(); }
        static int &depth() { static thread_local int d = 0; return d; }
    };

private:
    struct Impl;
    Impl &impl();
};

// Small page-locked, device-mapped host blocks (PINNED_BLOCK bytes each; any device's) and events without timing, kept
// likewise.  An event belongs to the device that was current when it was taken.
constexpr size_t PINNED_BLOCK = 32768;
struct PinnedBlock {
    char *host = nullptr, *dev = nullptr;
};
PinnedBlock take_pinned_block();
void give_pinned_block(const PinnedBlock &b);
// Such a block for a result that kernels on `stream` write into it.  Left by an exception before anybody has waited for the
// stream, it goes back to the pool only behind the kernels, and not at all if the stream cannot be waited for: whoever takes
// it next may be a solve that reads the solver's words from it.
class ResultBlock {
public:
    explicit ResultBlock(hipStream_t stream) : block_(take_pinned_block()), stream_(stream) {}
    ResultBlock(const ResultBlock &) = delete;
    ResultBlock &operator=(const ResultBlock &) = delete;
    ~ResultBlock() { if (arrived_ || hipStreamSynchronize(stream_) == hipSuccess) give_pinned_block(block_); }
    char *dev() const { return block_.dev; }
    char *host() const { return block_.host; }
    void unused() { arrived_ = true; }   // nothing that is enqueued uses it (any more)
    const char *wait() {   // the result, on the host
        TSVM_HIP_CHECK(hipStreamSynchronize(stream_));
        arrived_ = true;
        return block_.host;
    }
    // The same for `count` numbers that the kernels write one by one, each once, by looking at them: the runtime's own wait is some
    // microseconds behind the last write.  expect() comes before the kernels; nothing that they compute is NOT_YET, a signalling NaN.
    static constexpr uint64_t NOT_YET = 0x7ff4a5c3961e87d2ull;
    void expect(size_t count) {
        for (size_t i = 0; i < count; ++i) ((volatile uint64_t *) block_.host)[i] = NOT_YET;
    }
    const double *wait_for(size_t count);

private:
    PinnedBlock block_;
    hipStream_t stream_;
    bool arrived_ = false;
};
struct DeviceEvent {
    hipEvent_t event = nullptr;
    int device = -1;
};
DeviceEvent take_event();
void give_event(const DeviceEvent &e);

// Copies between pageable host memory and the device through a ring of page-locked chunks: the host fills (or empties)
// one chunk while the others are on their way.  Asynchronous on `stream` as far as the device side goes; when upload()
// returns the source has been read, when download() returns the destination holds the data.  One ring per process,
// one user at a time.
class HostStaging {
public:
    static HostStaging &instance();
    // fill(to, offset, length): writes bytes [offset, offset + length) of what is to be uploaded
    void upload(void *dst, size_t bytes, const std::function<void(char *, size_t, size_t)> &fill, hipStream_t stream);
    // what lies at `parts`, one after another
    struct Part {
        const void *from;
        size_t bytes, at;   // at: byte offset in the destination, ascending
    };
    void upload(void *dst, const std::vector<Part> &parts, hipStream_t stream);
    // take(from, offset, length): bytes [offset, offset + length) have arrived.  timeout_ms > 0: gives up (std::runtime_error)
    // when nothing has arrived for that long, for a stream whose kernels may hang; whoever sets it leaves the stream's
    // memory alone afterwards.
    void download(const void *src, size_t bytes, const std::function<void(const char *, size_t, size_t)> &take, hipStream_t stream,
                  long long timeout_ms = 0);

    static constexpr size_t CHUNK = (size_t) 4 << 20;

private:
    struct Impl;
    Impl &impl();
};
// Asks state_of(thing) until it says hipSuccess; throws any error but hipErrorNotReady, and std::runtime_error after
// timeout_ms.
void wait_until_done(hipError_t (*state_of)(void *), void *thing, long long timeout_ms);
// memcpy on as many threads as pay for a block of this size
void parallel_memcpy(void *to, const void *from, size_t bytes);

size_t &device_bytes_in_use();   // running total of DeviceBuffer allocations (the SyncMem byte counter's role)

// One grow-only device allocation that outlives individual solves and holds the kernel rows (working-set
// rows plus the row cache).  Releasing a multi-gigabyte allocation costs up to seconds on this platform,
// so the 21 one-vs-one solves of a 7-class problem must not each allocate and free their own pool.
// Not counted in device_bytes_in_use().
// One training or prediction call at a time per process: the row arena, the pooled CU-masked streams and the staging
// buffers are shared by all of them (the reference is not re-entrant either: one cuSPARSE handle, one SyncMem
// counter).  The model-level entry points hold this lock for their duration, so calls from several host threads
// take turns instead of sharing those buffers.
std::recursive_mutex &device_work_mutex();

class RowArena {
public:
    static RowArena &instance();
    // bytes a solve may use when the caller gave no explicit budget: nine tenths of what is free or already held
    size_t auto_budget();
    void *acquire(size_t bytes, bool auto_sized);
    void release();
    size_t capacity() const { return cap_; }

private:
    void *ptr_ = nullptr;
    size_t cap_ = 0;
    bool full_budget_ = false;
};

template <typename T>
class DeviceBuffer {
public:
    DeviceBuffer() = default;
    explicit DeviceBuffer(size_t count) { resize(count); }
    DeviceBuffer(const DeviceBuffer &) = delete;
    DeviceBuffer &operator=(const DeviceBuffer &) = delete;
    DeviceBuffer(DeviceBuffer &&o) noexcept : ptr_(o.ptr_), count_(o.count_), device_(o.device_) { o.ptr_ = nullptr; o.count_ = 0; }
    DeviceBuffer &operator=(DeviceBuffer &&o) noexcept {
        if (this != &o) { release(); ptr_ = o.ptr_; count_ = o.count_; device_ = o.device_; o.ptr_ = nullptr; o.count_ = 0; }
        return *this;
    }
    ~DeviceBuffer() { release(); }

    void resize(size_t count) {
        if (count == count_) return;
        release();
        if (count) {
            ptr_ = (T *) DevicePool::instance().take(count * sizeof(T), &device_);
            device_bytes_in_use() += count * sizeof(T);
        }
        count_ = count;
    }
    // idle: nothing enqueued on the device uses the buffer any more (otherwise it is handed out again only after the
    // device has been idle)
    void release(bool idle = false) {
        if (ptr_) {
            DevicePool::instance().give(ptr_, count_ * sizeof(T), device_, idle);
            device_bytes_in_use() -= count_ * sizeof(T);
        }
        ptr_ = nullptr;
        count_ = 0;
    }
    T *data() { return ptr_; }
    const T *data() const { return ptr_; }
    size_t size() const { return count_; }
    // Gives the memory up without freeing it: for a device that has stopped answering, where hipFree would not return.
    void abandon() { ptr_ = nullptr; count_ = 0; }

    // (on work_stream(), as everything here; when upload returns the source has been read)
    void upload(const T *host, size_t count, size_t offset = 0) {
        if (count) HostStaging::instance().upload(ptr_ + offset, {{host, count * sizeof(T), 0}}, work_stream());
    }
    void upload(const std::vector<T> &v) { resize(v.size()); upload(v.data(), v.size()); }
    void download(T *host, size_t count, size_t offset = 0) const {
        if (count)
            HostStaging::instance().download(ptr_ + offset, count * sizeof(T), [host](const char *from, size_t off, size_t len) {
                parallel_memcpy((char *) host + off, from, len);
            }, work_stream());
    }
    std::vector<T> to_host() const { std::vector<T> v(count_); download(v.data(), count_); return v; }
    void zero() { if (count_) TSVM_HIP_CHECK(hipMemsetAsync(ptr_, 0, count_ * sizeof(T), work_stream())); }

private:
    T *ptr_ = nullptr;
    size_t count_ = 0;
    int device_ = -1;   // whose memory it is
};

// Page-locked host staging memory that only grows (hipHostMalloc; copies from it are asynchronous and run at
// the link's rate).  Kernels read it in place too: mapped and coherent whatever the environment's default is, on any device.
template <typename T>
class PinnedBuffer {
public:
    PinnedBuffer() = default;
    PinnedBuffer(const PinnedBuffer &) = delete;
    PinnedBuffer &operator=(const PinnedBuffer &) = delete;
    ~PinnedBuffer() { if (ptr_) (void) hipHostFree(ptr_); }
    void reserve(size_t count) {
        if (count <= count_) return;
        if (ptr_) (void) hipHostFree(ptr_);
        ptr_ = nullptr;
        count_ = 0;
        TSVM_HIP_CHECK(hipHostMalloc((void **) &ptr_, count * sizeof(T), hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable));
        count_ = count;
    }
    T *data() { return ptr_; }
    size_t size() const { return count_; }

private:
    T *ptr_ = nullptr;
    size_t count_ = 0;
};

}  // namespace tsvm
