#include "lane_streams.h"

#include <cstdint>
#include <cstdlib>
#include <exception>
#include <map>
#include <mutex>
#include <set>
#include <utility>
#include <vector>

#include "device.h"

namespace {

// CU-masked streams are kept for the life of the process and handed from one solve to the next: creating one
// makes a hardware queue, which costs far more than a solve's other set-up (and every few creations the runtime
// spends tens of milliseconds on queue housekeeping).  Keyed by device and lane count (which fix the masks).
struct LaneStreams {
    hipStream_t chip = nullptr, solver = nullptr;
    bool in_use = false;
};
// the streams of all lanes of one lane count on one device: made together, because the chip-wide mask leaves out
// exactly the CUs on which the lanes' solvers land
struct LaneGroup {
    std::vector<LaneStreams> lanes;
    hipStream_t chain = nullptr;   // of one lane, in place of the solver's
};
std::mutex g_mutex;
std::map<long long, std::vector<LaneGroup>> g_groups;
std::map<int, int> g_solver_cu;    // by device
std::set<long long> g_unavailable;

hipStream_t masked_stream(const uint32_t (&mask)[8]) {
    hipStream_t s = nullptr;
    TSVM_HIP_CHECK(hipExtStreamCreateWithCUMask(&s, 8, mask));
    return s;
}

void destroy(hipStream_t &s) {
    if (s) (void) hipStreamDestroy(s);
    s = nullptr;
}
void destroy(LaneGroup &g) {
    for (LaneStreams &m : g.lanes) {
        destroy(m.solver);
        destroy(m.chip);
    }
    destroy(g.chain);
}

// The pooled streams are destroyed by an atexit handler, registered when the first one is made and therefore run
// before the HIP runtime's own tear-down (which, under a profiler, crashed on queues still alive at that point).
void destroy_groups() {
    std::lock_guard<std::mutex> lock(g_mutex);
    for (auto &kv : g_groups)
        for (LaneGroup &g : kv.second) destroy(g);
    g_groups.clear();
}

// tsvm_where's number of XCD 0's only CU in the mask of `stream`, which has one of every XCD.
int find_solver_cu(hipStream_t stream) {
    tsvm::DeviceBuffer<int> d_where(8);
    int where[8];
    tsvm::abi_check(tsvm_where(d_where.data(), 8, stream));
    TSVM_HIP_CHECK(hipMemcpyAsync(where, d_where.data(), sizeof(where), hipMemcpyDeviceToHost, stream));
    TSVM_HIP_CHECK(hipStreamSynchronize(stream));
    for (int w : where)
        if (w >> 16 == 0) return w & 0xffff;
    throw std::runtime_error("no workgroup on XCD 0");
}

// Makes the streams of a group, two a lane.  Bit i of a CU mask names CU i/8 of XCD i%8 on the 8-XCD, 256-CU part (a
// mask has to leave every XCD at least one CU: workgroups are dealt to the XCDs in turn).  Every solver stream gets
// CU 0 of every XCD, and lane l's solver is launched so that it runs on XCD l (tsvm_c_smo_solve_block_on_xcd: eight
// workgroups, one per XCD, the one on XCD l solves, the others leave at once).  The lanes thus share the eight CUs
// without sharing a CU, each solver behind another L2.  The chip-wide streams get every CU but those the solvers
// really run on, CU 0 of XCDs 0 .. n_lanes-1: 255 CUs for one lane, 248 for eight.  (On the CUs the two masks share,
// a solver launch's seven idle workgroups wait for room like any workgroup; the solver's result is behind them only in
// stream order, and they are gone long before it is done.)  A lane that is the only one has a stream with every CU instead, on which
// its solver finds that CU by itself; a solver stream only shows, the first time, which one it is, and is given back: a
// process that also has the streams of other lane counts has more queues than the hardware runs at a time, and each costs (after
// solves in one, three and six lanes a nu-SVC of 21 pairs takes 250 ms, 360 with that queue kept, 88 in a process of its own).
void make_lane_group(int device, int n_lanes, LaneGroup &g) {
    const uint32_t small[8] = {0xffu, 0, 0, 0, 0, 0, 0, 0}, all[8] = {~0u, ~0u, ~0u, ~0u, ~0u, ~0u, ~0u, ~0u};
    const uint32_t big[8] = {~((1u << n_lanes) - 1u), ~0u, ~0u, ~0u, ~0u, ~0u, ~0u, ~0u};   // all but CU 0 of XCDs 0 .. n_lanes-1
    g.lanes.assign(n_lanes, LaneStreams());
    for (LaneStreams &m : g.lanes) {
        if (n_lanes > 1 || !g_solver_cu.count(device)) m.solver = masked_stream(small);
        m.chip = masked_stream(big);
    }
    if (n_lanes > 1) return;
    g.chain = masked_stream(all);
    if (!g_solver_cu.count(device)) g_solver_cu[device] = find_solver_cu(g.lanes[0].solver);
    destroy(g.lanes[0].solver);
}

}  // namespace

namespace tsvm {

bool take_lane_streams(int lane, int n_lanes, LaneLease &lease) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess) return false;
    const long long key = (long long) dev * 16 + n_lanes;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (g_unavailable.count(key)) return false;
    std::vector<LaneGroup> &groups = g_groups[key];
    LaneGroup *group = nullptr;
    for (LaneGroup &g : groups)
        if (!g.lanes[lane].in_use) { group = &g; break; }
    if (!group) {
        LaneGroup g;
        try {
            make_lane_group(dev, n_lanes, g);
        } catch (const std::exception &) {
            (void) hipGetLastError();
            destroy(g);
            g_unavailable.insert(key);
            return false;
        }
        static bool registered = false;
        if (!registered) {
            registered = true;
            atexit(destroy_groups);
        }
        groups.push_back(std::move(g));
        group = &groups.back();
    }
    LaneStreams &mine = group->lanes[lane];
    mine.in_use = true;
    lease.chip = mine.chip;
    lease.solver = mine.solver;
    lease.chain = group->chain;
    lease.solver_cu = group->chain ? g_solver_cu.at(dev) : -1;
    lease.key = key;
    lease.lane = lane;
    return true;
}

void give_lane_streams(const LaneLease &lease) {
    std::lock_guard<std::mutex> lock(g_mutex);
    for (LaneGroup &g : g_groups[lease.key])
        if (g.lanes[lease.lane].chip == lease.chip) g.lanes[lease.lane].in_use = false;
}

}  // namespace tsvm
