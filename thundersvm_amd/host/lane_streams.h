// The streams of the solves that are in flight, by which the local solvers have compute units of their own.
#pragma once
#include <hip/hip_runtime_api.h>

namespace tsvm {

// What a task has of the pool until it gives it back.
struct LaneLease {
    hipStream_t chip = nullptr;     // every CU but those on which the lanes' solvers land
    hipStream_t solver = nullptr;   // tasks beside others: CU 0 of every XCD
    // A task that runs alone: a stream with every CU, and the CU that its chip-wide stream leaves out (tsvm_where's number).
    hipStream_t chain = nullptr;
    int solver_cu = -1;
    long long key = 0;
    int lane = 0;
};

// The streams of lane `lane` of n_lanes (1 .. 8) on the current device; false when they cannot be had.  A device on which they could
// not be made once is not asked again.
bool take_lane_streams(int lane, int n_lanes, LaneLease &lease);
void give_lane_streams(const LaneLease &lease);   // (by a task that has nothing left on them)

}  // namespace tsvm
