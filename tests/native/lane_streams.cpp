// The pool of CU-masked streams when the calls that make them fail, one after another: a program of its own whose definitions of the
// HIP calls and of tsvm_where stand in for the libraries'.  Exits with 0, or prints what went wrong.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <set>

#include "../../include/thundersvm_amd.h"
#include "../../thundersvm_amd/host/lane_streams.h"

static int g_device = 0, g_failures = 0, g_calls = 0, g_fail_at = -1, g_made = 0;
static bool g_no_die = false;                 // no workgroup reports XCD 0
static std::set<const void *> g_live;

static void expect(bool ok, const char *what) {
    if (ok) return;
    ++g_failures;
    fprintf(stderr, "lane streams: %s (device %d, call %d fails)\n", what, g_device, g_fail_at);
}
static bool fails() { return g_calls++ == g_fail_at; }

extern "C" {
hipError_t hipGetDevice(int *d) { *d = g_device; return hipSuccess; }
hipError_t hipSetDevice(int d) { g_device = d; return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipMalloc(void **p, size_t bytes) { *p = malloc(bytes); return hipSuccess; }
hipError_t hipFree(void *p) { free(p); return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipExtStreamCreateWithCUMask(hipStream_t *s, uint32_t, const uint32_t *) {
    if (fails()) return hipErrorOutOfMemory;
    ++g_made;
    *s = (hipStream_t) malloc(1);
    g_live.insert(*s);
    return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t s) {
    expect(g_live.erase(s) == 1, "a stream is destroyed twice");
    free(s);
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t) {
    if (fails()) return hipErrorUnknown;
    memcpy(to, from, bytes);
    return hipSuccess;
}
int tsvm_where(int *out, int n, tsvm_stream) {
    if (fails()) return 1;
    for (int b = 0; b < n; ++b) out[b] = (b + (g_no_die ? 1 : 0)) << 16 | (100 + b);
    return 0;
}
const char *tsvm_last_error(void) { return "a launch that was refused"; }
}

// A device of its own for every attempt: calls number `fail_at` fails while its streams of n_lanes lanes are made.
static void attempt(int n_lanes, int fail_at) {
    ++g_device;
    g_calls = 0;
    g_fail_at = fail_at;
    const size_t before = g_live.size();
    tsvm::LaneLease lease;
    if (fail_at >= 0) {
        expect(!tsvm::take_lane_streams(0, n_lanes, lease), "streams although a call has failed");
        expect(g_live.size() == before, "a failure leaves streams behind");
        const int made = g_made;
        g_fail_at = -1;
        expect(!tsvm::take_lane_streams(0, n_lanes, lease) && g_made == made, "a device that has refused is asked again");
        return;
    }
    expect(tsvm::take_lane_streams(0, n_lanes, lease), "no streams");
    expect(g_live.size() == before + 2 * n_lanes, "two streams a lane");
    expect(n_lanes == 1 ? lease.chain && !lease.solver && lease.solver_cu == 100 : lease.solver && !lease.chain, "a lane's streams");
    tsvm::LaneLease second, again;
    expect(tsvm::take_lane_streams(0, n_lanes, second) && second.chip != lease.chip, "streams that are in use");
    expect(g_live.size() == before + 4 * n_lanes && second.solver_cu == lease.solver_cu, "two streams a lane of a second group");
    tsvm::give_lane_streams(lease);
    expect(tsvm::take_lane_streams(0, n_lanes, again) && again.chip == lease.chip && g_live.size() == before + 4 * n_lanes, "streams that were given back");
}

int main() {
    for (int n_lanes : {1, 2, 8}) attempt(n_lanes, -1);
    for (int call = 0; call < 5; ++call) attempt(1, call);   // three streams, the launch, the copy
    for (int call = 0; call < 4; ++call) attempt(2, call);
    g_no_die = true;
    attempt(1, 1000);
    if (g_failures == 0) puts("ok");
    return g_failures != 0;
}
