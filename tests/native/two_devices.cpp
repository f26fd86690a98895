// The pools of the host layer with two devices, which a single-GPU machine does not have, and the wait of a download for a
// device that does not answer: a program of its own whose
// definitions of the HIP calls stand in for the runtime's (the host library's calls resolve to them), hand out host memory and
// remember which device every block, stream and event belongs to.  Exits with 0, or prints what went wrong.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "../../thundersvm_amd/host/device.h"

static int g_current = 0, g_failures = 0;
static bool g_hung = false;                   // events are never reached
static hipError_t g_stream_state = hipSuccess;   // what waiting for a stream says
static int g_stream_waits = 0;
static unsigned g_host_flags = 0;              // of the last page-locked allocation
static std::map<const void *, int> g_owner;   // device of every live block, stream and event

static void expect(bool ok, const char *what) {
    if (ok) return;
    ++g_failures;
    fprintf(stderr, "two devices: %s\n", what);
}
template <typename T>
static hipError_t make(T *out, size_t bytes) {
    *out = (T) malloc(bytes);
    g_owner[*out] = g_current;
    return hipSuccess;
}
static hipError_t drop(void *p) {
    expect(!p || g_owner.erase(p) == 1, "something is given back twice");
    free(p);
    return hipSuccess;
}

extern "C" {
hipError_t hipGetDevice(int *d) { *d = g_current; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_current = d; return hipSuccess; }
hipError_t hipMalloc(void **p, size_t bytes) { return make(p, bytes); }
hipError_t hipFree(void *p) { return drop(p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned flags) { g_host_flags = flags; return make(p, bytes); }
hipError_t hipHostFree(void *p) { return drop(p); }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { ++g_stream_waits; return g_stream_state; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { return make(s, 1); }
hipError_t hipStreamDestroy(hipStream_t s) { return drop(s); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return make(e, 1); }
hipError_t hipEventDestroy(hipEvent_t e) { return drop(e); }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return g_hung ? hipErrorNotReady : hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {   // (the runtime refuses this too)
    expect(g_owner.at(e) == g_owner.at(s), "an event is recorded on a stream of the other device");
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t) {
    memcpy(to, from, bytes);
    return hipSuccess;
}
}

static void blocks(bool idle) {
    g_current = 0;
    tsvm::DeviceBuffer<char> a(5000);
    const void *const block = a.data();
    g_current = 1;
    a.release(idle);                              // freed while the other device is the current one
    tsvm::DeviceBuffer<char> b(5000);
    expect(g_owner.at(b.data()) == 1, "a buffer of device 1 got device 0's memory");
    g_current = 0;
    tsvm::DeviceBuffer<char> c(5000);
    expect(c.data() == block, "device 0 did not get its block back");
    tsvm::DeviceBuffer<char> moved(std::move(b)), assigned;
    assigned = std::move(moved);
    assigned.release(idle);
    tsvm::DeviceBuffer<char> d(5000);
    expect(g_owner.at(d.data()) == 0, "a buffer of device 0 got device 1's memory after a move");
}

// A block that kernels write a result into: waited for, left by an exception, and left on a stream that reports an error.
static void result_blocks() {
    const void *first = nullptr;
    for (int step = 0; step < 4; ++step) {
        g_stream_waits = 0;
        g_stream_state = step == 2 ? hipErrorLaunchFailure : hipSuccess;
        try {
            tsvm::ResultBlock b(nullptr);
            if (step == 0) first = b.dev();
            expect((b.dev() == first) == (step < 3), "a result's block is not the one that is free");
            if (step == 0) expect(b.wait() == first, "a result on the host");
            else throw std::runtime_error("a launch that was refused");
        } catch (const std::runtime_error &) {
        }
        expect(step == 3 || g_stream_waits == 1, "a block went back without anybody having waited for its stream");
    }
}

int main() {
    result_blocks();
    g_stream_state = hipSuccess;
    tsvm::PinnedBuffer<double> staging;
    staging.reserve(100);
    expect(g_host_flags == (hipHostMallocMapped | hipHostMallocCoherent | hipHostMallocPortable), "staging memory that kernels read in place");
    blocks(true);
    tsvm::DevicePool::instance().flush();
    blocks(false);
    g_current = 0;
    const tsvm::DeviceEvent e = tsvm::take_event();
    g_current = 1;
    tsvm::give_event(e);
    expect(g_owner.at(tsvm::take_event().event) == 1, "device 1 got device 0's event");
    std::vector<int> data(1000, 7);
    for (int round = 0; round < 6; ++round) {     // (more uploads than the ring has chunks: each waits for an older one's event)
        g_current = round & 1;
        tsvm::DeviceBuffer<int> x(data.size());
        for (int i = 0; i < 5; ++i) x.upload(data.data(), data.size());
        expect(g_owner.at(x.data()) == g_current, "an upload's buffer is on the other device");
    }
    // a download that is given a limit gives up on a device that has stopped answering, and the next one is whole
    tsvm::DeviceBuffer<int> x(data.size());
    x.upload(data.data(), data.size());
    std::vector<int> back(data.size(), 0);
    const auto take = [&](const char *from, size_t off, size_t len) { memcpy((char *) back.data() + off, from, len); };
    for (int attempt = 0; attempt < 2; ++attempt) {
        g_hung = attempt == 0;
        bool gave_up = false;
        try {
            tsvm::HostStaging::instance().download(x.data(), data.size() * sizeof(int), take, tsvm::work_stream(), 20);
        } catch (const std::runtime_error &) {
            gave_up = true;
        }
        expect(gave_up == g_hung && back[0] == (g_hung ? 0 : 7), "a download with a limit");
    }
    if (g_failures == 0) puts("ok");
    return g_failures != 0;
}
