// The local SMO solvers: c_smo_solve / nu_smo_solve (src/thundersvm/kernel/smo_kernel.cpp:12-287,
// USE_CUDA=OFF semantics) as one LDS-resident workgroup on gfx950.
//
// Shape of the kernels.  One workgroup of one or four wavefronts (one per SIMD of the CU) holds the whole working set:
// element t = tid*E + e lives in register slot e of thread tid (a thread's elements are neighbours, so its share of a
// block row is one load) with its f and diagonal; alpha lives in LDS (only two entries change per iteration) and the
// I_up / I_low membership of a thread's elements is a bit field in a register.  One inner iteration is
//   1. (i, up) = first argmin of f over I_up: a per-thread scan of its E slots, a DPP reduction inside each wavefront,
//      the wavefronts' candidates through LDS;
//   2. row K[i, .] of the gathered ws x ws block (coalesced);
//   3. j2 = first argmin of -b^2/a over I_low with f > up: same reduction shape;
//   4. the two-variable step, row K[j2, .], f -= l * (K[j2, .] - K[i, .]).
//
// What bounds it: one chain of dependent instructions.  With one wavefront per SIMD an instruction takes four cycles
// whatever it does, an LDS access fifty, a block row 250 (from the L2), a value that crosses to the scalar unit and
// comes back about forty, a branch around a few instructions about forty-five, and a write or a broadcast read by all
// 256 threads takes the LDS four wavefronts' worth of cycles.  Hence: no branches inside the loop; what one lane knows is written by that
// lane alone (exec set to one bit around the write); every wavefront keeps its own copy of alpha; each lane reads one
// wavefront's candidate and two DPP steps compare them; the winner's index by ballot instead of a second reduction; the
// exit test folded into the loop's branch (the last round computes a step that is not taken); and everything that does
// not need the row on its way pinned in front of the first instruction that does.
// Measured on a call of 483 iterations with ws = 1024: 1.37 us per iteration before that, 1.08 with it (2,590 cycles);
// 0.97 with the scores ranked in float where that decides (c_smo_iterate_rounded); a tenth less since its chains are single blocks
// (epsilon-SVR 40000x90, launches' starts and ends included: 1.08 -> 0.98 a step).
//
// Reductions are lexicographic (value, element index) minima, so ties go to the lowest
// index exactly as the reference's serial loops resolve them, and all arithmetic is the reference's
// expression order in IEEE double (the library is compiled with -ffp-contract=off; the one fused
// operation, f -= l*(kJ - kI), is an explicit fma as gcc -O3 contracts it on an FMA host, and
// kd_i + kd_t - 2*K_it is written as fma(-2, K_it, kd_i + kd_t), which rounds identically because
// the product by 2 is exact).
#include "../../include/thundersvm_amd.h"
#include "tsvm_device.h"
#include "smo_local.h"
#include "tsvm_internal.h"

#include <algorithm>
#include <map>
#include <mutex>
#include <utility>

#define TSVM_INF __builtin_inf()
#define MAX_WS 1024
#define SV_LD 256          // smallest row stride of the ws x ws block

// kws[r*ldk + t] = K_r[working_set[t]] for t < ws, 0 for ws <= t < ldk: the ws x ws block the solver
// reads, gathered once per call so that the two row reads per inner iteration
// (smo_kernel.cpp:50-52,107-110) are contiguous; rows are padded to the solver's thread x slot grid
// so every thread can load without a bounds test.
// TB: element type of the block.  Float kernel rows give a float block: the same values in half the bytes, widened
// again when the solver loads them.
template <typename TK, typename TB>
__global__ void gather_ws_block_kernel(const TK *__restrict__ k_rows, const int *__restrict__ slots, int64_t ld,
                                       const int *__restrict__ working_set, int ws, int ldk, TB *__restrict__ kws) {
    const int r = blockIdx.x;
    const TK *row = k_rows + (int64_t) (slots ? slots[r] : r) * ld;
    for (int t = threadIdx.x; t < ldk; t += blockDim.x) kws[(int64_t) r * ldk + t] = t < ws ? (TB) row[working_set[t]] : (TB) 0;
}

// The same block when a table names the slot of every instance's row (a row cache that holds them all): row r
// is the one of instance ids[r]; its slot is also written to slots_out[r], for update_f.
template <typename TK, typename TB>
__global__ void gather_ws_block_by_id_kernel(const TK *__restrict__ k_rows, const int *__restrict__ slot_of_id, int64_t ld,
                                             const int *__restrict__ ids, int ws, int ldk, TB *__restrict__ kws,
                                             int *__restrict__ slots_out) {
    const int r = blockIdx.x;
    const int slot = slot_of_id[ids[r]];
    if (threadIdx.x == 0) slots_out[r] = slot;
    const TK *row = k_rows + (int64_t) slot * ld;
    for (int t = threadIdx.x; t < ldk; t += blockDim.x) kws[(int64_t) r * ldk + t] = t < ws ? (TB) row[ids[t]] : (TB) 0;
}

// Slots for a working set's new rows when the row store has a slot for every instance (nothing is ever
// evicted, so the bookkeeping needs no host): instances seen for the first time take the next free slots in the
// order of the list.  One workgroup; ids_new are distinct.
//   slot_of_id[i]  slot of instance i's row, -1 while it has none           (updated)
//   state[0]       slots in use                                              (updated)
//   state[1]       number of rows to compute for this working set            (written)
//   miss_ids / miss_slots [0 .. state[1])  the instances to compute and where their rows go
//   slots_ws[t]    slot of ids_ws[t], t < ws
//   info[0..1]     state[1], state[0] for the host (pinned host memory or device memory)
#define RA_T 1024
__global__ __launch_bounds__(RA_T) void row_slots_assign_kernel(const int *__restrict__ ids_new, int n_new,
                                                                int *__restrict__ slot_of_id, int *__restrict__ state,
                                                                int *__restrict__ miss_ids, int *__restrict__ miss_slots,
                                                                const int *__restrict__ ids_ws, int ws, int *__restrict__ slots_ws,
                                                                int *__restrict__ info) {
    __shared__ int wave_total[RA_T / 64];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int id = tid < n_new ? ids_new[tid] : 0;
    const bool miss = tid < n_new && slot_of_id[id] < 0;
    const unsigned long long b = __ballot(miss);
    const int before = __popcll(b & ((1ull << lane) - 1ull));
    if (lane == 0) wave_total[wave] = __popcll(b);
    __syncthreads();
    int rank = before, total = 0;
    for (int w = 0; w < RA_T / 64; ++w) {
        const int c = wave_total[w];
        if (w < wave) rank += c;
        total += c;
    }
    const int base = state[0];
    if (miss) {
        slot_of_id[id] = base + rank;
        miss_ids[rank] = id;
        miss_slots[rank] = base + rank;
    }
    __syncthreads();   // the table's new entries are read back below by other threads of this workgroup
    if (tid == 0) {
        state[0] = base + total;
        state[1] = total;
        info[0] = total;
        info[1] = base + total;
    }
    if (tid < ws) slots_ws[tid] = slot_of_id[ids_ws[tid]];
}

// What a solve starts from besides its vectors, in one launch: zeroed alpha_diff, the block's columns beyond ws (the
// solver reads them), no slot for any instance, zeroed counters and gate.
template <typename TB>
__global__ void smo_start_kernel(double *alpha_diff, int n_diff, TB *kws, int ws, int ldk, int *slot_of_id, int n_ids, int *state, int *gate) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x, stride = (int64_t) gridDim.x * blockDim.x;
    for (int64_t i = gid; i < n_diff; i += stride) alpha_diff[i] = 0.0;
    for (int64_t i = gid; i < n_ids; i += stride) slot_of_id[i] = -1;
    if (ws < ldk)
        for (int64_t i = gid; i < (int64_t) ws * ldk; i += stride) kws[i] = (TB) 0;
    if (state && gid < 2) state[gid] = 0;
    if (gate && gid < 4) gate[gid] = 0;
}

// Reads the block on one XCD, so that the rows a solver on that XCD asks for are in its L2 (written by kernels on all
// XCDs, they are in none: a row then takes some 700 cycles instead of 250).  Workgroup b runs on XCD b % 8 as a rule;
// those on another one leave.  One call of 455 iterations at ws = 1024: 1.22 us per iteration on a block that has just
// been written, 1.09 after this kernel, which takes about 6 us.
#define SV_L2_BYTES (4u << 20)   // (warm_block_kernel leaves larger blocks alone; warm_share)
#define SV_WARM_SLICES 32
__global__ __launch_bounds__(256) void warm_block_kernel(const uint4 *__restrict__ p, unsigned n16, int xcd, int *__restrict__ sink) {
    if ((int) __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)) != xcd) return;   // XCC_ID
    const unsigned per = (n16 + SV_WARM_SLICES - 1) / SV_WARM_SLICES, lo = (blockIdx.x >> 3) * per, hi = lo + per < n16 ? lo + per : n16;
    unsigned any = 0;
    for (unsigned i = lo + threadIdx.x; i < hi; i += 256) {
        const uint4 v = p[i];
        any |= v.x & v.y & v.z & v.w;
    }
    if (any == 0xfff5a5a5u) *sink = 0;   // (keeps the loads; no kernel value has these bits)
}

// A thread's E consecutive elements of a block row: one 4E- or 8E-byte load.
template <int E, typename TB>
__device__ __forceinline__ void load_row_elems(const TB *__restrict__ row, int tid, TB (&out)[E]) {
    if constexpr (E == 1) {
        out[0] = row[tid];
    } else {
        typedef TB vec_t __attribute__((ext_vector_type(E)));
        const vec_t v = *(const vec_t *) (row + tid * E);
#pragma unroll
        for (int e = 0; e < E; ++e) out[e] = v[e];
    }
}

// The same by buffer loads: the row's offset in bytes is a scalar operand of the load, without an addition of addresses in front of it.
template <int E, typename TB>
struct BlockRows {
    __amdgpu_buffer_rsrc_t block;
    int at;
    __device__ __forceinline__ BlockRows(const TB *kws, unsigned n, int tid)
        : block(__builtin_amdgcn_make_buffer_rsrc((void *) kws, 0, (int) (n * sizeof(TB)), 0x00027000)), at(tid * E * (int) sizeof(TB)) {}
    __device__ __forceinline__ void load(int row, TB (&out)[E]) const {
        constexpr int BYTES = E * (int) sizeof(TB);
        static_assert(BYTES == 8 || BYTES % 16 == 0, "two or four elements");
        typedef unsigned v2u __attribute__((ext_vector_type(2)));
        typedef unsigned v4u __attribute__((ext_vector_type(4)));
        if constexpr (BYTES == 8) {
            const v2u v = __builtin_amdgcn_raw_buffer_load_b64(block, at, row, 0);
            __builtin_memcpy(out, &v, 8);
        } else {
#pragma unroll
            for (int b = 0; b < BYTES / 16; ++b) {
                const v4u v = __builtin_amdgcn_raw_buffer_load_b128(block, at + 16 * b, row, 0);
                __builtin_memcpy((char *) out + 16 * b, &v, 16);
            }
        }
    }
};

// One solver on a chosen XCD.  A kernel of one workgroup runs on whichever XCD its stream's hardware queue starts
// dealing at; launched as eight workgroups under a CU mask with one CU per XCD, one workgroup lands on every XCD, and
// the one that finds itself on target_xcd does the work while the others leave at once.  Exactly one workgroup is
// elected whatever the dealing: the workgroup on the target claims the launch (gate[0]: the number of the last launch
// claimed, epoch = that number + 1 for this launch), and the last of the eight to arrive (gate[1] counts arrivals,
// eight per launch) claims it if nobody has.  gate[2] tells the host where the solver ran.  Launches that share a gate
// must be ordered (one stream); gate starts as zeros, epoch at 1.
#define TSVM_SOLVER_GRID_ON_XCD 8
__device__ __forceinline__ int own_xcd() { return (int) __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11)); }   // XCC_ID
__device__ __forceinline__ int own_cu() { return (int) __builtin_amdgcn_s_getreg(4 | (8 << 6) | (7 << 11)); }     // HW_ID: CU, SH and SE
__device__ __forceinline__ bool solver_elected(int *gate, int epoch, int target_xcd) {
    __shared__ int s_elected;
    if (threadIdx.x == 0) {
        const int xcd = own_xcd();
        bool won = false;
        if (xcd == target_xcd) won = atomicCAS(&gate[0], epoch - 1, epoch) == epoch - 1;
        __threadfence();
        const unsigned arrived = atomicAdd((unsigned *) &gate[1], 1u);
        if (!won && (arrived % TSVM_SOLVER_GRID_ON_XCD) == TSVM_SOLVER_GRID_ON_XCD - 1) {
            __threadfence();
            won = atomicCAS(&gate[0], epoch - 1, epoch) == epoch - 1;
        }
        if (won) gate[2] = xcd;
        s_elected = won;
    }
    __syncthreads();
    return s_elected != 0;
}

// One solver on a chosen CU, for a launch on a stream that has every CU.  As many workgroups as the chip has CUs, each asking for a whole CU's
// LDS: one lands on every CU (256 different ones of 256 in every launch looked at), and the one on the CU that the row kernels'
// stream leaves out does the work.  The kernels before and behind it are then on its own stream, without the two markers
// that a solver on a stream of its own needs (some 11 us each).  Election as above (the last to arrive claims a launch that nobody has
// claimed, wherever it is); every atomic has come back before the next is made.  The others on that XCD read the block
// into its L2 before they leave (in place of warm_block_kernel, 10 us in front of the solver).  `started` tells the host that
// the solver has its CU: rows that take the other CUs before that keep those workgroups, and with them the block, out
// (20000 x 784, solver beside 340 us of rows 337 us, 427 when they came first).
// The launch has ended when every workgroup has found a CU with all of its LDS free: beside kernels of other streams, the caller's own
// or another solve's, it waits for more than eight workgroups on CUs of their own did, each of which waited at two markers, though.  A
// call in ms, when the solver had a stream of its own / now (the steps themselves are 10 % shorter now):
//   beside                          nothing      products of 2,048    of 6,144 (bf16)   copies of 256 MB   another call
//   epsilon-SVR 40000x90          78.6 / 65.9       203 /   84          249 /  121         266 / 139         159 / 134
//   nu-SVC 5001x23                3.50 / 3.08      4.46 / 3.89         11.0 / 10.4        7.98 / 7.14       7.00 / 6.03
//   C-SVC 20000x784               34.1 / 31.6      44.4 / 38.0         76.0 / 72.4        70.8 / 62.9       69.8 / 65.0
#define TSVM_SOLVER_GRID_ON_CU 256
__device__ __forceinline__ bool solver_elected_on_cu(int *gate, int epoch, bool on_target, int *started) {
    __shared__ int s_elected;
    if (threadIdx.x == 0) {
        int won = 0, seen = epoch - 1;
        if (on_target) won = __hip_atomic_compare_exchange_strong(&gate[0], &seen, epoch, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(won) :: "memory");
        // (unsigned: 8.4 million launches take the count beyond the largest int)
        unsigned arrived = __hip_atomic_fetch_add((unsigned *) &gate[1], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(arrived) :: "memory");
        if (!won && arrived % TSVM_SOLVER_GRID_ON_CU == TSVM_SOLVER_GRID_ON_CU - 1) {
            seen = epoch - 1;
            won = __hip_atomic_compare_exchange_strong(&gate[0], &seen, epoch, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (won) {
            gate[2] = own_xcd();
            __hip_atomic_store(started, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        s_elected = won;
    }
    __syncthreads();
    return s_elected != 0;
}
// Workgroup b is number b / 8 of its XCD's thirty-two, as a rule.
// Of a block that is larger than the L2 (1,024 rows of doubles, 8 MB), what has been selected last, the most violating first: the rows behind
// the half that the working set keeps, three quarters of an L2 of them.  Linear text, 18,000 rows, a call: none 32.4 ms, 384 of those rows
// 31.5 (448 as much, all 512 a little less), 448 of the kept ones 32.3.
// (LARGE: a variant of its own, as the test in the others moved their loops: the nu variant's steps took 3 % longer.)
template <bool LARGE>
__device__ __forceinline__ void warm_share(const void *block, unsigned bytes, int *gate) {
    const uint4 *p = (const uint4 *) block;
    if (bytes > SV_L2_BYTES) {
        if (!LARGE) return;
        p += bytes / 2 / 16;
        bytes = bytes / 2 < SV_L2_BYTES / 4 * 3 ? bytes / 2 : SV_L2_BYTES / 4 * 3;
    }
    const unsigned n16 = bytes / 16, per = (n16 + SV_WARM_SLICES - 1) / SV_WARM_SLICES, lo = (blockIdx.x >> 3) * per, hi = lo + per < n16 ? lo + per : n16;
    unsigned any = 0;
    for (unsigned i = lo + threadIdx.x; i < hi; i += blockDim.x) {
        const uint4 v = p[i];
        any |= v.x & v.y & v.z & v.w;
    }
    if (any == 0xfff5a5a5u) gate[3] = 0;   // (keeps the loads; no kernel value has these bits)
}

// The CU every workgroup runs on: XCD in the upper half, CU in the lower.
__global__ __launch_bounds__(64) void where_kernel(int *out) {
    if (threadIdx.x == 0) out[blockIdx.x] = own_xcd() << 16 | own_cu();
}

// What a thread's elements start from.  Every load is made (for positions beyond ws the last element's: f, alpha and the label are
// zero and the diagonal 1 there) and none waits for another but for its id; E * 4 loads behind a test each were a chain of sixteen
// misses.  A whole call of one step 12.0 -> 10.9 us; epsilon-SVR on 40,000 rows (212 launches) 98.8 -> 98.0 ms.
template <int E>
__device__ __forceinline__ void gather_elems(const int *__restrict__ working_set, int ws, const double *__restrict__ f_val, const double *alpha_val,
                                             const int *__restrict__ labels, const double *__restrict__ k_diag, double (&f)[E], double (&alpha)[E],
                                             double (&kd)[E], int (&label)[E]) {
    int id[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int t = (int) threadIdx.x * E + e;
        id[e] = working_set[t < ws ? t : ws - 1];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        f[e] = f_val[id[e]];
        alpha[e] = alpha_val[id[e]];
        label[e] = labels[id[e]];
        kd[e] = k_diag[id[e]];
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool active = (int) threadIdx.x * E + e < ws;
        f[e] = active ? f[e] : 0.0;
        alpha[e] = active ? alpha[e] : 0.0;
        label[e] = active ? label[e] : 0;
        kd[e] = active ? kd[e] : 1.0;
    }
}

// Whether this workgroup of a launch is the one that solves, with what its elements start from.  (What is gathered is on its way during
// the election; those that can only be elected last gather behind it.)
template <int E, bool LARGE>
__device__ __forceinline__ bool solver_begins(int *gate, int epoch, int target_xcd, int target_cu, int *started, const void *block, unsigned bytes,
                                              const int *__restrict__ working_set, int ws, const double *__restrict__ f_val, const double *alpha_val,
                                              const int *__restrict__ labels, const double *__restrict__ k_diag, double (&f)[E], double (&alpha)[E],
                                              double (&kd)[E], int (&label)[E]) {
    const bool on_xcd = target_cu < 0 || own_xcd() == target_xcd, likely = on_xcd && (target_cu < 0 || own_cu() == target_cu);
    if (likely) gather_elems<E>(working_set, ws, f_val, alpha_val, labels, k_diag, f, alpha, kd, label);
    if (!gate) return true;
    if (target_cu < 0) return solver_elected(gate, epoch, target_xcd);
    if (!solver_elected_on_cu(gate, epoch, likely, started)) {
        if (on_xcd) warm_share<LARGE>(block, bytes, gate);
        return false;
    }
    if (!likely) gather_elems<E>(working_set, ws, f_val, alpha_val, labels, k_diag, f, alpha, kd, label);
    return true;
}

// What the solvers keep in LDS per element of the working set (inactive elements: both bounds zero, so neither in I_up nor in
// I_low).  Bounds and diagonal are read by one address.
// (A workgroup that only passes by, of another lane's launch, has to find room beside a solver: at most half of the CU's 160 KB.  With
// 82 KB in place of 73 every launch waited for the others' solvers, and seven classes of 92,000 rows took 20 % longer.)
struct __align__(32) SvElem {
    SvBound bound;
    double kd, f;             // f: c_smo_iterate's alone, at the wavefronts' candidates for j2 (the others are not written)
};
template <int N, int W>
struct SvShared {
    SvElem elem[N];
    double z[W][N];           // alpha times its label: every wavefront keeps a copy of its own, which needs no barrier
};

// What c_smo_solve keeps.
template <int N, int W>
struct SvState {
    SvElem elem[N];
    double z[W][N];           // every wavefront keeps a copy of its own, which needs no barrier
    double k[N];              // row i at the elements of the wavefronts' candidates for j2 (as f)
};

// The iterations of c_smo_solve.  Four wavefronts compare by rows of sixteen lanes (block_first_min), as c_smo_iterate_rounded does: the same
// eight steps as over a wavefront and then over four, without the way through the scalar unit in between, worth its sixteen records
// since the chains are single blocks (3200x32, where nothing is decided by rounded scores: 2.58 -> 2.53 ms a call; z and in_low
// left to the next step's waits, as there: 2.55).
// An element that violates may have no score: the threshold is not positive and its f not above
// `up`, or the score is infinite or NaN (an a that is negative with a b^2 beyond the largest double; kernel values that are no
// numbers).  The reference's j2 then stays 0 (smo_kernel.cpp:78).  NONE: that is done here.  Without it such a step goes
// wrong, and `no_score` is set for the caller to start over; one instruction, where a way out of the loop in front of the
// step costs 5 %.
// Takes up to `left` steps, counted in n_iter; returns whether the solve has ended (nothing violates, or max_iter).
template <int E, int W, int LDK, bool NONE, typename TB>
__device__ __forceinline__ bool c_smo_iterate(SvState<E * 64 * W, W> &sh, SvCand *s_i, SvCand *s_j, int ws, const TB *kws,
                                              const double (&kd)[E], double (&f)[E], unsigned &in_up, unsigned &in_low, double local_eps,
                                              int max_iter, int &n_iter, int left, bool &no_score) {
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const BlockRows<E, TB> rows(kws, (unsigned) ws * (unsigned) LDK, tid);
    auto load_row = [&](int r, TB (&out)[E]) {
        if constexpr (W == 4) rows.load(r * (LDK * (int) sizeof(TB)), out);
        else load_row_elems<E, TB>(kws + (unsigned) r * (unsigned) LDK, tid, out);
    };
    int own[E];   // (whoever is chosen without being a candidate is one that exists)
#pragma unroll
    for (int e = 0; e < E; ++e) own[e] = tid * E + e < ws ? tid * E + e : ws - 1;
    bool go_on;
    double min_t = -TSVM_INF;
    int worst = 0;   // high word of the largest score that a step was taken on
    do {
        if (!NONE) worst = imax_sel(worst, __double2hiint(min_t));
        // i = first argmin of f over I_up (smo_kernel.cpp:41-59); with an empty I_up any i does, since nothing violates then
        double fu[E];
#pragma unroll
        for (int e = 0; e < E; ++e) fu[e] = keep_or_none<0>(in_up << (31 - e), f[e]);
        double up_value, m;
        int at, i, j2, go;
        if constexpr (W == 4) {
            block_first_min<E>(s_i, fu, own, 0, [](uint64_t) {}, up_value, i, go);
        } else {
            const int win_i = wave_first_argmin<E>(fu, tid * E, up_value, m, at);
            i = __builtin_amdgcn_readlane(at, win_i);
            i = i < ws ? i : ws - 1;   // (without a candidate the index may be an inactive element's)
        }
        TB kI[E];
        load_row(i, kI);
        SV_PIN_MEMORY;
        const double kd_i = sh.elem[i].kd, z_i = sh.z[wave][i];
        const SvBound bound_i = sh.elem[i].bound;
        double a_part[E], b_low[E], b_max = -TSVM_INF;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            a_part[e] = kd_i + kd[e];
            b_low[e] = keep_or_none<1>(in_low << (31 - e), -up_value + f[e]);
            b_max = e == 0 ? b_low[e] : fmax_f64(b_max, b_low[e]);
        }
        // some I_low element still violates: low - up >= local_eps (smo_kernel.cpp:68)
        go = __builtin_amdgcn_ballot_w64(!(b_max < local_eps)) != 0;
        double up_i = bound_i.hi - z_i;
        asm("" : "+v"(up_i));
        SV_PIN;   // (all of this while the row is on its way)
        // j2 = first argmin of -b^2/a over I_low with f > up (smo_kernel.cpp:77-90)
        double qs[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double aIJ = __builtin_fma(-2.0, (double) kI[e], a_part[e]);
            const double q = -b_low[e] * b_low[e] / aIJ;
            // (-up > -f in the reference: f > up, which is b > 0; outside I_low b is negative and q of no use)
            qs[e] = __hiloint2double(b_low[e] > 0.0 ? __double2hiint(q) : SV_NONE_HI, __double2loint(q));
        }
        if constexpr (W == 4) {
            block_first_min<E>(s_j, qs, own, go, [&](uint64_t lanes) { publish_row<E, TB, 4>(&sh.elem[tid * E].f, sh.k + tid * E, lanes, f, kI); }, min_t, j2, go);
        } else {
            const int win_j = wave_first_argmin<E>(qs, tid * E, min_t, m, at);
            publish_row<E, TB, 4>(&sh.elem[tid * E].f, sh.k + tid * E, 1ull << win_j, f, kI);
            j2 = __builtin_amdgcn_readlane(at, win_j);
        }
        if (NONE && is_none(min_t)) {
            j2 = 0;
            __syncthreads();
            if (tid == 0) { sh.elem[0].f = f[0]; *(TB *) sh.k = kI[0]; }
            __syncthreads();
        }
        if constexpr (W != 4) j2 = j2 < ws ? j2 : ws - 1;
        TB kJ[E];
        load_row(j2, kJ);
        SV_PIN_MEMORY;
        const SvBound bound_j = sh.elem[j2].bound;
        const double kd_j = sh.elem[j2].kd, z_j = sh.z[wave][j2], f_j = sh.elem[j2].f;
        const double kIj = (double) *(const TB *) (sh.k + j2);
        SV_PIN;   // the row is on its way while the step is computed
        // two-variable step (smo_kernel.cpp:92-103; the last round computes one that is not taken)
        go_on = go && !(n_iter > max_iter);
        const double q2 = (-up_value + f_j) / __builtin_fma(-2.0, kIj, kd_i + kd_j);
        const double l = fmin_f64(up_i, fmin_f64(z_j - bound_j.lo, q2));
        const double nz_i = z_i + l, nz_j = (NONE && j2 == i ? nz_i : z_j) - l;
        const unsigned bit_i = own_bit<E>(tid, i), bit_j = own_bit<E>(tid, j2);
        const unsigned up_i_on = same_in_all_lanes(nz_i < bound_i.hi), low_i_on = same_in_all_lanes(nz_i > bound_i.lo);
        const unsigned up_j_on = same_in_all_lanes(nz_j < bound_j.hi), low_j_on = same_in_all_lanes(nz_j > bound_j.lo);
        in_up = put_bits(put_bits(in_up, bit_i, up_i_on), bit_j, up_j_on);
        in_low = put_bits(put_bits(in_low, bit_i, low_i_on), bit_j, low_j_on);
        write_by_lane0(go_on, &sh.z[wave][i], nz_i, &sh.z[wave][j2], nz_j);
        SV_PIN;   // (nothing above waits for the row)
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = __builtin_fma(-l, (double) kJ[e] - (double) kI[e], f[e]);
        n_iter += go_on;
    } while (go_on && --left > 0);
    if (!NONE) no_score |= __builtin_amdgcn_readfirstlane(go_on ? imax_sel(worst, __double2hiint(min_t)) : worst) >= SV_NONE_HI;
    return !go_on;
}

// The same iterations for four wavefronts with j2 chosen by b^2/a rounded to float, as long as that decides: the largest
// score has to beat the second by more than both can be off, and to be in float's range.  A score is off by at most
// 4.2e-7 (b, a, the two products 2^-24 each, b twice; the reciprocal 2^-23), so a lead of 2^-19 = 1.9e-6 is proof, and the
// winner is then the reference's j2.  Otherwise the function returns false before the step, which c_smo_iterate then takes.
// (Scores are floored at 2^-80, which makes smaller ones ties; a score without a lead includes every tie, no candidate at
// all, negative a, and NaN.  What falls to the floor although it is larger: an a of 2^126 and more, whose reciprocal is a
// denormal, that is zero; and a b that is zero or a denormal in float, with an a so small that b^2/a is not, zero times
// infinity.  Such a b is the difference of an f and an `up` below 2^-73: anything above is a multiple of 2^-126.  A thread that
// meets either stands for an infinite second-best score, and nothing is decided: 740 steps 727 -> 728 us, 755 -> 768 on a block of
// doubles.)
// That replaces E divisions of some fourteen instructions by six each, and the reduction over doubles by one over floats.
// Rows of sixteen lanes are reduced by DPP and publish themselves, and after the barrier every lane reads one of the
// sixteen rows and four more steps compare them: the same eight steps as over a wavefront and then over four of them, without
// the way through the scalar unit in between.
// A step is bound by the issue of its instructions, so it is counted in them: 351 and 35 wait states -> 300 and 15 with the chains of
// DPP steps in one block each, membership bits changed by masks (put_bits), rows read at a scalar offset (BlockRows), one
// address for an element's bounds and diagonal, a limit of steps that shares the way out with the stopping test, and z and in_low
// written while the next step waits for its candidates.  A whole call: epsilon-SVR 40000x90 (54,594 steps) 74.8 -> 69.1 ms, sparse text
// 18000 (24,020) 34.0 -> 32.0, 20,000 x 784 (32,880) 39.2 -> 37.8.
template <int E, int LDK, typename TB>
__device__ __forceinline__ bool c_smo_iterate_rounded(SvState<E * 256, 4> &sh, SvCand *s_i, SvScoreStep *s_j, int ws, const TB *kws,
                                                      const double (&kd)[E], double (&f)[E], unsigned &in_up, unsigned &in_low,
                                                      double local_eps, int max_iter, int &n_iter) {
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned my_i = lds_at(s_i + (tid >> 4)), my_j = lds_at(s_j + (tid >> 4));
    unsigned my_z = lds_at(&sh.z[wave][0]);
    asm("" : "+v"(my_z));
    const BlockRows<E, TB> rows(kws, (unsigned) ws * (unsigned) LDK, tid);
    int at_of[E];   // (whoever is chosen without being a candidate is one that exists)
#pragma unroll
    for (int e = 0; e < E; ++e) at_of[e] = tid * E + e < ws ? tid * E + e : ws - 1;
    uint64_t go;
    // what a step leaves to the waits of the next: its changes to in_low, and the two elements' new z
    unsigned bit_i = 0, bit_j = 0, low_i = 0, low_j = 0, z_at_i = my_z, z_at_j = my_z;
    double nz_i = 0, nz_j = 0;
    int pending = 0;
    for (;;) {
        double fu[E];
#pragma unroll
        for (int e = 0; e < E; ++e) fu[e] = keep_or_none<0>(in_up << (31 - e), f[e]);
        SvWords cand;
        uint64_t has;
        row_first_candidate<E>(fu, at_of, cand, has);
        publish_words(my_i, lowest_of_rows(has), cand);
        lds_barrier();
        const SvCand ci = s_i[lane & 15];
        write_by_lane0(pending, z_at_i, nz_i, z_at_j, nz_j);
        in_low = put_bits(put_bits(in_low, bit_i, low_i), bit_j, low_j);
        double up_value;
        uint64_t first;
        row_min_and_who(ci.v, up_value, first);
        const int i = __builtin_amdgcn_readlane(ci.at, __builtin_ctzll(first));
        TB kI[E];
        rows.load(i * (LDK * (int) sizeof(TB)), kI);
        SV_PIN_MEMORY;
        z_at_i = my_z + 8u * (unsigned) i;
        const SvBound bound_i = sh.elem[i].bound;
        const double kd_i = sh.elem[i].kd, z_i = lds_f64(z_at_i);
        bit_i = own_bit<E>(tid, i);
        asm("" : "+v"(bit_i));
        double a_part[E], b_low[E], b_max = -TSVM_INF;
        float b32[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            b_low[e] = keep_or_none<1>(in_low << (31 - e), -up_value + f[e]);
            b_max = e == 0 ? b_low[e] : fmax_f64(b_max, b_low[e]);
            b32[e] = __builtin_fmaxf((float) b_low[e], 0.0f);
            a_part[e] = kd_i + kd[e];
        }
        const int violates = (__builtin_amdgcn_ballot_w64(!(b_max < local_eps)) != 0) & (n_iter <= max_iter);   // (the way out is one test)
        double up_i = bound_i.hi - z_i;
        asm("" : "+v"(up_i));
        int a_max = __builtin_fabs(up_value) < SV_UP_LEAST ? 0x7f800000 : 0;   // (as the bits of a float)
        asm("" : "+v"(a_max));
        SV_PIN;
        double aIJ[E];
        float q[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            aIJ[e] = __builtin_fma(-2.0, (double) kI[e], a_part[e]);
            const float a32 = (float) aIJ[e];
            a_max = __float_as_int(a32) > a_max ? __float_as_int(a32) : a_max;
            q[e] = __builtin_fmaxf(b32[e] * (b32[e] * __builtin_amdgcn_rcpf(a32)), 0x1p-80f);
        }
        float mine, second;
        if constexpr (E == 4) {
            const float h0 = __builtin_fmaxf(q[0], q[1]), h1 = __builtin_fmaxf(q[2], q[3]);
            mine = __builtin_fmaxf(h0, h1);
            second = __builtin_fmaxf(__builtin_fmaxf(__builtin_fminf(h0, h1), __builtin_fminf(q[0], q[1])), __builtin_fminf(q[2], q[3]));
        } else {
            static_assert(E == 2, "elements per thread");
            mine = __builtin_fmaxf(q[0], q[1]);
            second = __builtin_fminf(q[0], q[1]);
        }
        int at = at_of[E - 1];
        double b_at = b_low[E - 1], a_at = aIJ[E - 1];
#pragma unroll
        for (int e = E - 2; e >= 0; --e) {
            const bool is = q[e] == mine;
            at = is ? at_of[e] : at;
            b_at = is ? b_low[e] : b_at;
            a_at = is ? aIJ[e] : a_at;
        }
        second = a_max < SV_A_BITS ? second : __builtin_inff();
        float best, next;
        uint64_t who;   // (several only if nothing will be decided)
        row_best_two_and_who(mine, second, best, next, who);
        publish_score(my_j, who, best, next, at, violates, b_at, a_at);
        lds_barrier();
        const SvScoreStep cj = s_j[lane & 15];
        uint64_t won;
        row_best_two_and_who(cj.score.best, cj.score.second, best, next, won);
        const int row = __builtin_ctzll(won);
        const int j2 = __builtin_amdgcn_readlane(cj.score.at, row);
        TB kJ[E];
        rows.load(j2 * (LDK * (int) sizeof(TB)), kJ);
        SV_PIN_MEMORY;
        z_at_j = my_z + 8u * (unsigned) j2;
        const SvBound bound_j = sh.elem[j2].bound;
        const double z_j = lds_f64(z_at_j);
        SV_PIN;
        const double steps = cj.step.b / cj.step.a;   // (every row's, while the bounds are read)
        const double q2 = readlane_f64(steps, row);
        bit_j = own_bit<E>(tid, j2);
        // (the two comparisons come out the same in every lane)
        go = __builtin_amdgcn_ballot_w64(cj.score.go != 0);
        const uint64_t sure = __builtin_amdgcn_ballot_w64(next < best * (1.0f - 0x1p-19f)) & __builtin_amdgcn_ballot_w64(best < 0x1p80f);
        if ((go & sure) == 0) break;
        SV_PIN;
        const double l = fmin_f64(fmin_f64(up_i, z_j - bound_j.lo), q2);
        nz_i = z_i + l;
        nz_j = z_j - l;
        const unsigned up_i_on = same_in_all_lanes(nz_i < bound_i.hi), up_j_on = same_in_all_lanes(nz_j < bound_j.hi);
        low_i = same_in_all_lanes(nz_i > bound_i.lo);
        low_j = same_in_all_lanes(nz_j > bound_j.lo);
        in_up = put_bits(put_bits(in_up, bit_i, up_i_on), bit_j, up_j_on);
        pending = 1;
        SV_PIN;
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = __builtin_fma(-l, (double) kJ[e] - (double) kI[e], f[e]);
        ++n_iter;
    }
    return go == 0;
}

// Elements beyond ws are given y = 0, which puts them in neither I_up nor I_low.
// E elements per thread, W wavefronts; LDK: row stride of the block (E * 64 * W <= LDK).
template <int E, int W, int LDK, typename TB>
__global__ __launch_bounds__(64 * W) void c_smo_solve_kernel(
    const int *__restrict__ label, const double *__restrict__ f_val, double *__restrict__ alpha,
    double *__restrict__ alpha_diff, const int *__restrict__ working_set, int ws, double Cp, double Cn,
    const TB *kws, const double *__restrict__ k_diag, double eps, double *__restrict__ diff,
    int max_iter, int *__restrict__ gate, int epoch, int target_xcd, int target_cu) {
    double f[E], a_old[E], kd[E];
    int y_of[E];
    if (!solver_begins<E, (sizeof(TB) * LDK * LDK > SV_L2_BYTES)>(gate, epoch, target_xcd, target_cu, (int *) (diff + 2), kws, (unsigned) (ws * LDK * sizeof(TB)), working_set, ws, f_val, alpha, label, k_diag, f, a_old, kd,
                          y_of))
        return;
    constexpr int N = E * 64 * W;
    __shared__ SvState<N, W> sh;
    __shared__ double s_red[2][W];
    __shared__ SvCand s_i[4 * W], s_j[4 * W];
    __shared__ SvScoreStep s_score[4 * W];
    static_assert(sizeof(sh) + sizeof(s_red) + sizeof(s_i) + sizeof(s_j) + sizeof(s_score) <= 80 * 1024, "two workgroups on a CU");

    // This workgroup is a chain of dependent operations; when a chip-wide kernel runs next to it on
    // another stream its wavefronts must not wait behind that kernel's for issue slots.
    __builtin_amdgcn_s_setprio(3);
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned in_up, in_low, plus;   // bit e: element e is in I_up, in I_low, has a label > 0
    int n_iter;
    for (bool with_none = false;;) {
        in_up = in_low = plus = 0;
        n_iter = 0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int t = tid * E + e;
            const double y = (double) y_of[e];
            sh.elem[t].kd = kd[e];
            sh.elem[t].bound.hi = y > 0 ? Cp : 0.0;
            sh.elem[t].bound.lo = y < 0 ? -Cn : 0.0;
            plus |= (y > 0 ? 1u : 0u) << e;
#pragma unroll
            for (int w = 0; w < W; ++w) sh.z[w][t] = a_old[e] * y;
            in_up |= (is_I_up(a_old[e], y, Cp, Cn) ? 1u : 0u) << e;
            in_low |= (is_I_low(a_old[e], y, Cp, Cn) ? 1u : 0u) << e;
        }
        // The initial gap fixes the local stopping threshold (smo_kernel.cpp:61-66).  It is the only place
        // where the value of low = max of f over I_low is needed: inside the loop the stopping test
        // low - up < local_eps is evaluated per element, as "no I_low element has f - up >= local_eps"
        // (the same decision, since rounding the subtraction is monotone), which costs a ballot instead of
        // a second cross-lane reduction per iteration.
        double local_eps;
        {
            double mn = TSVM_INF, mx = -TSVM_INF;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                mn = fmin_f64(mn, (in_up >> e) & 1u ? f[e] : TSVM_INF);
                mx = fmax_f64(mx, (in_low >> e) & 1u ? f[e] : -TSVM_INF);
            }
            mn = wave_min_f64(mn);
            mx = wave_max_f64(mx);
            if (lane == 0) { s_red[0][wave] = mn; s_red[1][wave] = mx; }
            __syncthreads();
            double up0 = s_red[0][0];
#pragma unroll
            for (int w = 1; w < W; ++w) up0 = fmin_f64(up0, s_red[0][w]);
            const double local_diff = block_max<W>(s_red[1]) - up0;
            const double t = 0.1f * local_diff;   // float literal, as in the reference (smo_kernel.cpp:64)
            local_eps = t > eps ? t : eps;
            if (tid == 0) diff[0] = local_diff;
        }
        bool no_score = false;
        if (with_none || !__builtin_amdgcn_readfirstlane(local_eps > 0.0 ? 1 : 0)) {
            c_smo_iterate<E, W, LDK, true, TB>(sh, s_i, s_j, ws, kws, kd, f, in_up, in_low, local_eps, max_iter, n_iter, 0x7fffffff, no_score);
        } else if constexpr (W == 4) {
            // One step in a hundred or two is not decided by rounded scores (epsilon-SVR, pixels): four exact steps, then rounded
            // ones again.  Where they go on not deciding (far apart points of equal f) the exact stretch grows
            // eightfold each time the rounded one has been the shorter of the two.  Stretches from 64 on, doubling / from
            // 8, doubling / from 4, times eight: SVR 40000x90 98.0 / 96.7 / 96.8 ms, pixels 20000x784 53.5 / 52.5 / 52.7,
            // blobs 3200x32 (nothing is decided) 3.128 / 3.160 / 3.139.
            bool done;
            int stretch = 4;
            do {
                const int before = n_iter;
                done = c_smo_iterate_rounded<E, LDK, TB>(sh, s_i, s_score, ws, kws, kd, f, in_up, in_low, local_eps, max_iter, n_iter);
                if (done) break;
                stretch = n_iter - before > stretch ? 4 : stretch < 1024 ? 8 * stretch : stretch;
                done = c_smo_iterate<E, W, LDK, false, TB>(sh, s_i, s_j, ws, kws, kd, f, in_up, in_low, local_eps, max_iter, n_iter, stretch, no_score);
            } while (!done && !no_score);
        } else {
            c_smo_iterate<E, W, LDK, false, TB>(sh, s_i, s_j, ws, kws, kd, f, in_up, in_low, local_eps, max_iter, n_iter, 0x7fffffff, no_score);
        }
        if (!no_score) break;
        with_none = true;   // (nothing has been written yet: once more from the start)
        __syncthreads();
        gather_elems<E>(working_set, ws, f_val, alpha, label, k_diag, f, a_old, kd, y_of);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int t = tid * E + e;
        if (t < ws) {
            const double y = (plus >> e) & 1u ? 1.0 : -1.0;
            const double a = sh.z[wave][t] * y + 0.0;   // (+ 0.0: a zero comes out as +0, as from alpha +- l)
            alpha_diff[t] = -(a - a_old[e]) * y;
            alpha[working_set[t]] = a;
        }
    }
    // diff may be host memory that a waiting host thread polls: diff[1] is the kernel's last word, and everything
    // written before it (diff[0] in particular) has to be visible system-wide first
    if (tid == 0) {
        __threadfence_system();
        diff[1] = (double) n_iter;
    }
}

// nu variant (smo_kernel.cpp:127-287): four extrema, two second-order candidates.  Keeps the CPU
// code's j2n score, which uses kd[ip] and K[ip, .] (smo_kernel.cpp:239), and leaves diff[1] alone.
// Membership bits per element: 0 = y>0 & a<C (I_up, positive), 1 = y<0 & a>0 (I_up, negative),
// 2 = y>0 & a>0 (I_low, positive), 3 = y<0 & a<C (I_low, negative).
__device__ __forceinline__ unsigned nu_member_bits(double z, const SvBound &bound) {
    const unsigned b = (z < bound.hi ? 1u : 0u) | (z > bound.lo ? 4u : 0u);
    return bound.hi > 0 ? b : b << 1;
}

// The iterations of nu_smo_solve.  Takes up to `left` steps, counted in n_iter; returns whether the solve has ended.
template <int E, int W, int LDK, typename TB>
__device__ __forceinline__ bool nu_iterate(SvShared<E * 64 * W, W> &sh, double (&s_f)[2][E * 4 * W], double (&s_k)[2][E * 4 * W], SvCand *s_ip, SvCand *s_in,
                                           SvCand *s_jp, SvCand *s_jn, int ws, const TB *kws, const double (&kd)[E], double (&f)[E], unsigned &member,
                                           double local_eps, int max_iter, int &n_iter, int left) {
    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const BlockRows<E, TB> rows(kws, (unsigned) ws * (unsigned) LDK, tid);
    auto load_row = [&](int r, TB (&out)[E]) {
        if constexpr (W == 4) rows.load(r * (LDK * (int) sizeof(TB)), out);
        else load_row_elems<E, TB>(kws + (unsigned) r * (unsigned) LDK, tid, out);
    };
    int own[E];
#pragma unroll
    for (int e = 0; e < E; ++e) own[e] = tid * E + e < ws ? tid * E + e : ws - 1;
    const int row_at = (tid >> 4) * E;   // where this lane publishes its elements when it is its row's candidate
    for (; left > 0; --left) {
        double fup[E], fun[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            fup[e] = keep_or_none<0>(member << (31 - 4 * e), f[e]);
            fun[e] = keep_or_none<0>(member << (30 - 4 * e), f[e]);
        }
        double up_value_p, up_value_n, m_p, m_n;
        int ip, in, at_p, at_n, go;
        if constexpr (W == 4) {
            block_first_mins<E>(s_ip, s_in, fup, fun, own, 0, [](uint64_t, uint64_t) {}, up_value_p, up_value_n, ip, in, go);
        } else {
            const int win_ip = wave_first_argmin<E>(fup, tid * E, up_value_p, m_p, at_p);
            const int win_in = wave_first_argmin<E>(fun, tid * E, up_value_n, m_n, at_n);
            ip = __builtin_amdgcn_readlane(at_p, win_ip);
            in = __builtin_amdgcn_readlane(at_n, win_in);
        }
        // (an empty side's index stays 0: its row enters the other side's scores, smo_kernel.cpp:239)
        ip = is_none(up_value_p) ? 0 : ip;
        in = is_none(up_value_n) ? 0 : in;
        TB kIp[E], kIn[E];
        load_row(ip, kIp);
        load_row(in, kIn);
        SV_PIN_MEMORY;
        const double kd_ip = sh.elem[ip].kd, kd_in = sh.elem[in].kd;
        double a_part[E], lp[E], ln[E], b_max = -TSVM_INF;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            a_part[e] = kd_ip + kd[e];
            lp[e] = keep_or_none<1>(member << (29 - 4 * e), -up_value_p + f[e]);
            ln[e] = keep_or_none<1>(member << (28 - 4 * e), -up_value_n + f[e]);
            b_max = fmax_f64(e == 0 ? lp[e] : fmax_f64(b_max, lp[e]), ln[e]);
        }
        // max(low_p - up_p, low_n - up_n) >= local_eps (smo_kernel.cpp:185)
        go = __builtin_amdgcn_ballot_w64(!(b_max < local_eps)) != 0;
        SV_PIN;   // (all of this while the rows are on their way)
        double qp[E], qn[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const double aIJ = __builtin_fma(-2.0, (double) kIp[e], a_part[e]);
            const double q_p = -lp[e] * lp[e] / aIJ, q_n = -ln[e] * ln[e] / aIJ;
            // (-up > -f in the reference: f > up)
            qp[e] = __hiloint2double(lp[e] > 0.0 ? __double2hiint(q_p) : SV_NONE_HI, __double2loint(q_p));
            qn[e] = __hiloint2double(ln[e] > 0.0 ? __double2hiint(q_n) : SV_NONE_HI, __double2loint(q_n));
        }
        double f_val_j2p, f_val_j2n;
        int j2p, j2n;
        if constexpr (W == 4) {
            block_first_mins<E>(s_jp, s_jn, qp, qn, own, go, [&](uint64_t lanes_p, uint64_t lanes_n) {
                publish_row<E, TB>(s_f[0] + row_at, s_k[0] + row_at, lanes_p, f, kIp);
                publish_row<E, TB>(s_f[1] + row_at, s_k[1] + row_at, lanes_n, f, kIn);
            }, f_val_j2p, f_val_j2n, j2p, j2n, go);
        } else {
            const int win_jp = wave_first_argmin<E>(qp, tid * E, f_val_j2p, m_p, at_p);
            const int win_jn = wave_first_argmin<E>(qn, tid * E, f_val_j2n, m_n, at_n);
            publish_row<E, TB>(s_f[0] + row_at, s_k[0] + row_at, 1ull << win_jp, f, kIp);
            publish_row<E, TB>(s_f[1] + row_at, s_k[1] + row_at, 1ull << win_jn, f, kIn);
            j2p = __builtin_amdgcn_readlane(at_p, win_jp);
            j2n = __builtin_amdgcn_readlane(at_n, win_jn);
        }
        // (two sides without a candidate are equal, whatever the low words of their values hold)
        const bool take_p = __builtin_amdgcn_readfirstlane(f_val_j2p < f_val_j2n && f_val_j2p < SV_NONE ? 1 : 0) != 0;
        const int side = take_p ? 0 : 1;
        const int i = take_p ? ip : in;
        int j2 = take_p ? j2p : j2n;
        if (is_none(take_p ? f_val_j2p : f_val_j2n)) {   // (as in c_smo_iterate)
            j2 = 0;
            __syncthreads();
            if (tid == 0) { s_f[side][0] = f[0]; *(TB *) s_k[side] = take_p ? kIp[0] : kIn[0]; }
            __syncthreads();
        }
        if constexpr (W != 4) j2 = j2 < ws ? j2 : ws - 1;
        TB kJ[E];
        load_row(j2, kJ);
        SV_PIN_MEMORY;
        const int j2_at = j2 / (16 * E) * E + j2 % E;   // (the lane that has published it is the only one of its row)
        const double kd_j = sh.elem[j2].kd, z_j = sh.z[wave][j2], z_i = sh.z[wave][i], f_j = s_f[side][j2_at];
        const SvBound bound_i = sh.elem[i].bound, bound_j = sh.elem[j2].bound;
        const double kIj = (double) *(const TB *) (s_k[side] + j2_at);
        SV_PIN;   // the row is on its way while the exit test and the step are computed
        if (n_iter > max_iter || !go) return true;
        const double up_value = take_p ? up_value_p : up_value_n;
        const double q2 = (-up_value + f_j) / __builtin_fma(-2.0, kIj, (take_p ? kd_ip : kd_in) + kd_j);
        const double l = fmin_f64(bound_i.hi - z_i, fmin_f64(z_j - bound_j.lo, q2));
        const double nz_i = z_i + l, nz_j = (j2 == i ? nz_i : z_j) - l;
        const unsigned bit_i = own_bit<E, 4>(tid, i) << (bound_i.hi > 0 ? 0 : 1), bit_j = own_bit<E, 4>(tid, j2) << (bound_j.hi > 0 ? 0 : 1);
        const unsigned up_i_on = same_in_all_lanes(nz_i < bound_i.hi), low_i_on = same_in_all_lanes(nz_i > bound_i.lo);
        const unsigned up_j_on = same_in_all_lanes(nz_j < bound_j.hi), low_j_on = same_in_all_lanes(nz_j > bound_j.lo);
        member = put_bits(put_bits(member, bit_i, up_i_on), bit_i << 2, low_i_on);
        member = put_bits(put_bits(member, bit_j, up_j_on), bit_j << 2, low_j_on);
        write_by_lane0(1, &sh.z[wave][i], nz_i, &sh.z[wave][j2], nz_j);
        SV_PIN;   // (nothing above waits for the row)
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = __builtin_fma(-l, (double) kJ[e] - (double) (take_p ? kIp[e] : kIn[e]), f[e]);
        ++n_iter;
    }
    return false;
}

// The same iterations for four wavefronts with the side and its j2 chosen by b^2/a rounded to float, as long as that decides
// (c_smo_iterate_rounded: the same bounds, over the scores of both sides, whose largest has to beat every other; a side without
// a candidate for i leaves it undecided).  Both sides' scores have row ip's a (smo_kernel.cpp:239), the step the chosen
// side's own.  Bound by the issue of its instructions: eight divisions of doubles and two reductions over them become four
// reciprocals and one over floats.  1024 elements, 401 steps: 672 -> 539 us; a nu-SVC training of 5001x23: 4.00 -> 3.56 ms.  With the two
// sides' chains of DPP steps interleaved (each fills the other's wait states) and the rest as in c_smo_iterate_rounded 3.14 -> 3.02.
template <int E, int LDK, typename TB>
__device__ __forceinline__ bool nu_iterate_rounded(SvShared<E * 256, 4> &sh, SvCand *s_ip, SvCand *s_in, SvScoreStep *s_j, int ws, const TB *kws,
                                                   const double (&kd)[E], double (&f)[E], unsigned &member, double local_eps, int max_iter,
                                                   int &n_iter) {
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int SIDE_N = 1 << 16;   // in an element's number: the score is the negative side's
    const unsigned my_ip = lds_at(s_ip + (tid >> 4)), my_in = lds_at(s_in + (tid >> 4)), my_j = lds_at(s_j + (tid >> 4));
    unsigned my_z = lds_at(&sh.z[wave][0]);
    asm("" : "+v"(my_z));
    const BlockRows<E, TB> rows(kws, (unsigned) ws * (unsigned) LDK, tid);
    int own[E];
#pragma unroll
    for (int e = 0; e < E; ++e) own[e] = tid * E + e < ws ? tid * E + e : ws - 1;
    uint64_t go;
    // (as in c_smo_iterate_rounded)
    unsigned bit_i = 0, bit_j = 0, low_i = 0, low_j = 0, z_at_i = my_z, z_at_j = my_z;
    double nz_i = 0, nz_j = 0;
    int pending = 0;
    for (;;) {
        double fup[E], fun[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            fup[e] = keep_or_none<0>(member << (31 - 4 * e), f[e]);
            fun[e] = keep_or_none<0>(member << (30 - 4 * e), f[e]);
        }
        SvWords cand_p, cand_n;
        uint64_t has_p, has_n;
        row_first_candidates<E>(fup, fun, own, cand_p, cand_n, has_p, has_n);
        publish_words(my_ip, lowest_of_rows(has_p), cand_p);
        publish_words(my_in, lowest_of_rows(has_n), cand_n);
        lds_barrier();
        const SvCand cp = s_ip[lane & 15], cn = s_in[lane & 15];
        write_by_lane0(pending, z_at_i, nz_i, z_at_j, nz_j);
        member = put_bits(put_bits(member, bit_i, low_i), bit_j, low_j);
        double up_p, up_n;
        uint64_t who_p, who_n;
        row_mins_and_who(cp.v, cn.v, up_p, up_n, who_p, who_n);
        const int ip = __builtin_amdgcn_readlane(cp.at, __builtin_ctzll(who_p)), in = __builtin_amdgcn_readlane(cn.at, __builtin_ctzll(who_n));
        TB kIp[E], kIn[E];
        rows.load(ip * (LDK * (int) sizeof(TB)), kIp);
        rows.load(in * (LDK * (int) sizeof(TB)), kIn);
        SV_PIN_MEMORY;
        const double kd_ip = sh.elem[ip].kd, kd_in = sh.elem[in].kd;
        double a_part[E], lp[E], ln[E], b_max = -TSVM_INF;
        float p32[E], n32[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            a_part[e] = kd_ip + kd[e];
            lp[e] = keep_or_none<1>(member << (29 - 4 * e), -up_p + f[e]);
            ln[e] = keep_or_none<1>(member << (28 - 4 * e), -up_n + f[e]);
            b_max = fmax_f64(e == 0 ? lp[e] : fmax_f64(b_max, lp[e]), ln[e]);
            p32[e] = __builtin_fmaxf((float) lp[e], 0.0f);
            n32[e] = __builtin_fmaxf((float) ln[e], 0.0f);
        }
        const int violates = (__builtin_amdgcn_ballot_w64(!(b_max < local_eps)) != 0) & (n_iter <= max_iter);
        // (as the bits of a float: nothing is decided with an `up` of no candidate or too close to zero)
        const int hp = __double2hiint(up_p) & 0x7fffffff, hn = __double2hiint(up_n) & 0x7fffffff;
        int a_max = hp < SV_UP_LEAST_HI || hp >= SV_NONE_HI || hn < SV_UP_LEAST_HI || hn >= SV_NONE_HI ? 0x7f800000 : 0;
        asm("" : "+v"(a_max));
        SV_PIN;
        float q[E], low = 0x1p-80f;
        TB k_of[E];
        double b_of[E];
        int at_of[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const float a32 = (float) __builtin_fma(-2.0, (double) kIp[e], a_part[e]);
            a_max = __float_as_int(a32) > a_max ? __float_as_int(a32) : a_max;
            const float r = __builtin_amdgcn_rcpf(a32);
            const float qp = __builtin_fmaxf(p32[e] * (p32[e] * r), 0x1p-80f), qn = __builtin_fmaxf(n32[e] * (n32[e] * r), 0x1p-80f);
            q[e] = __builtin_fmaxf(qp, qn);
            low = __builtin_fmaxf(low, __builtin_fminf(qp, qn));
            const bool n_side = qn > qp;
            b_of[e] = n_side ? ln[e] : lp[e];
            k_of[e] = n_side ? kIn[e] : kIp[e];
            at_of[e] = n_side ? own[e] | SIDE_N : own[e];
        }
        float mine, second;
        if constexpr (E == 4) {
            const float h0 = __builtin_fmaxf(q[0], q[1]), h1 = __builtin_fmaxf(q[2], q[3]);
            mine = __builtin_fmaxf(h0, h1);
            second = __builtin_fmaxf(__builtin_fmaxf(__builtin_fminf(h0, h1), __builtin_fminf(q[0], q[1])), __builtin_fminf(q[2], q[3]));
        } else {
            static_assert(E == 2, "elements per thread");
            mine = __builtin_fmaxf(q[0], q[1]);
            second = __builtin_fminf(q[0], q[1]);
        }
        second = __builtin_fmaxf(second, low);
        int at = at_of[E - 1];
        double b_at = b_of[E - 1], kd_at = kd[E - 1];
        TB k_at = k_of[E - 1];
#pragma unroll
        for (int e = E - 2; e >= 0; --e) {
            const bool is = q[e] == mine;
            at = is ? at_of[e] : at;
            b_at = is ? b_of[e] : b_at;
            k_at = is ? k_of[e] : k_at;
            kd_at = is ? kd[e] : kd_at;
        }
        const double a_at = __builtin_fma(-2.0, (double) k_at, (at & SIDE_N ? kd_in : kd_ip) + kd_at);
        second = a_max < SV_A_BITS ? second : __builtin_inff();
        float best, next;
        uint64_t who;   // (several only if nothing will be decided)
        row_best_two_and_who(mine, second, best, next, who);
        publish_score(my_j, who, best, next, at, violates, b_at, a_at);
        lds_barrier();
        const SvScoreStep cj = s_j[lane & 15];
        uint64_t first;
        row_best_two_and_who(cj.score.best, cj.score.second, best, next, first);
        const int row = __builtin_ctzll(first);
        const int won = __builtin_amdgcn_readlane(cj.score.at, row);
        const bool n_side = (won & SIDE_N) != 0;
        const int j2 = won & (SIDE_N - 1), i = n_side ? in : ip;
        TB kJ[E];
        rows.load(j2 * (LDK * (int) sizeof(TB)), kJ);
        SV_PIN_MEMORY;
        z_at_i = my_z + 8u * (unsigned) i;
        z_at_j = my_z + 8u * (unsigned) j2;
        const SvBound bound_i = sh.elem[i].bound, bound_j = sh.elem[j2].bound;
        const double z_i = lds_f64(z_at_i), z_j = lds_f64(z_at_j);
        SV_PIN;
        const double steps = cj.step.b / cj.step.a;   // (every row's, while the bounds are read)
        const double q2 = readlane_f64(steps, row);
        // (an element that a step is taken on is of the side it was chosen for)
        const unsigned up_bit_i = own_bit<E, 4>(tid, i) << (n_side ? 1 : 0), up_bit_j = own_bit<E, 4>(tid, j2) << (n_side ? 1 : 0);
        go = __builtin_amdgcn_ballot_w64(cj.score.go != 0);
        const uint64_t sure = __builtin_amdgcn_ballot_w64(next < best * (1.0f - 0x1p-19f)) & __builtin_amdgcn_ballot_w64(best < 0x1p80f);
        if ((go & sure) == 0) break;
        SV_PIN;
        const double l = fmin_f64(fmin_f64(bound_i.hi - z_i, z_j - bound_j.lo), q2);
        nz_i = z_i + l;
        nz_j = z_j - l;
        const unsigned up_i_on = same_in_all_lanes(nz_i < bound_i.hi), up_j_on = same_in_all_lanes(nz_j < bound_j.hi);
        low_i = same_in_all_lanes(nz_i > bound_i.lo);
        low_j = same_in_all_lanes(nz_j > bound_j.lo);
        bit_i = up_bit_i << 2;
        bit_j = up_bit_j << 2;
        member = put_bits(put_bits(member, up_bit_i, up_i_on), up_bit_j, up_j_on);
        pending = 1;
        SV_PIN;
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = __builtin_fma(-l, (double) kJ[e] - (double) (n_side ? kIn[e] : kIp[e]), f[e]);
        ++n_iter;
    }
    return go == 0;
}

template <int E, int W, int LDK, typename TB>
__global__ __launch_bounds__(64 * W) void nu_smo_solve_kernel(
    const int *__restrict__ label, const double *__restrict__ f_val, double *__restrict__ alpha,
    double *__restrict__ alpha_diff, const int *__restrict__ working_set, int ws, double C,
    const TB *kws, const double *__restrict__ k_diag, double eps, double *__restrict__ diff,
    int max_iter, int *__restrict__ gate, int epoch, int target_xcd, int target_cu) {
    double f[E], a_old[E], kd[E];
    int y_of[E];
    if (!solver_begins<E, (sizeof(TB) * LDK * LDK > SV_L2_BYTES)>(gate, epoch, target_xcd, target_cu, (int *) (diff + 2), kws, (unsigned) (ws * LDK * sizeof(TB)), working_set, ws, f_val, alpha, label, k_diag, f, a_old, kd,
                          y_of))
        return;
    constexpr int N = E * 64 * W;
    __shared__ SvShared<N, W> sh;
    // f and the rows ip / in at the elements of the lanes that publish a candidate for j2, one of every sixteen.  (Slots for all elements
    // made it 98 KB, with which two lanes' launches do not fit a CU: a nu-SVC of four classes, 40,000 rows of 23 columns, 24.9 -> 21.9 ms.)
    __shared__ double s_f[2][4 * W * E], s_k[2][4 * W * E];
    __shared__ double s_red[4][W];
    __shared__ SvCand s_ip[4 * W], s_in[4 * W], s_jp[4 * W], s_jn[4 * W];
    __shared__ SvScoreStep s_score[4 * W];
    static_assert(sizeof(sh) + sizeof(s_f) + sizeof(s_k) + sizeof(s_red) + 4 * sizeof(s_ip) + sizeof(s_score) <= 80 * 1024, "two workgroups on a CU");

    __builtin_amdgcn_s_setprio(3);
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    unsigned member = 0, plus = 0;   // plus: bit e: element e has a label > 0
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int t = tid * E + e;
        const double y = (double) y_of[e];
        sh.elem[t].kd = kd[e];
        sh.elem[t].bound.hi = y > 0 ? C : 0.0;
        sh.elem[t].bound.lo = y < 0 ? -C : 0.0;
        plus |= (y > 0 ? 1u : 0u) << e;
#pragma unroll
        for (int w = 0; w < W; ++w) sh.z[w][t] = a_old[e] * y;
        member |= nu_member_bits(a_old[e] * y, sh.elem[t].bound) << (4 * e);
    }
    // initial gap -> local stopping threshold (smo_kernel.cpp:176-183); inside the loop the stopping
    // test is evaluated per element, as in the C variant
    double local_eps, first_diff;
    {
        double mnp = TSVM_INF, mnn = TSVM_INF, mxp = -TSVM_INF, mxn = -TSVM_INF;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const unsigned b = member >> (4 * e);
            mnp = fmin_f64(mnp, b & 1u ? f[e] : TSVM_INF);
            mnn = fmin_f64(mnn, b & 2u ? f[e] : TSVM_INF);
            mxp = fmax_f64(mxp, b & 4u ? f[e] : -TSVM_INF);
            mxn = fmax_f64(mxn, b & 8u ? f[e] : -TSVM_INF);
        }
        mnp = wave_min_f64(mnp);
        mnn = wave_min_f64(mnn);
        mxp = wave_max_f64(mxp);
        mxn = wave_max_f64(mxn);
        if (lane == 0) { s_red[0][wave] = mnp; s_red[1][wave] = mnn; s_red[2][wave] = mxp; s_red[3][wave] = mxn; }
        __syncthreads();
        double up_p0 = s_red[0][0], up_n0 = s_red[1][0];
#pragma unroll
        for (int w = 1; w < W; ++w) { up_p0 = fmin_f64(up_p0, s_red[0][w]); up_n0 = fmin_f64(up_n0, s_red[1][w]); }
        const double dp = block_max<W>(s_red[2]) - up_p0, dn = block_max<W>(s_red[3]) - up_n0;
        const double local_diff = dp < dn ? dn : dp;
        const double t = 0.1 * local_diff;
        local_eps = t > eps ? t : eps;
        first_diff = local_diff;
    }
    __syncthreads();
    int n_iter = 0;
    if constexpr (W == 4) {
        if (__builtin_amdgcn_readfirstlane(local_eps > 0.0 ? 1 : 0)) {
            bool done;
            int stretch = 4;   // (as in c_smo_solve_kernel)
            do {
                const int before = n_iter;
                done = nu_iterate_rounded<E, LDK, TB>(sh, s_ip, s_in, s_score, ws, kws, kd, f, member, local_eps, max_iter, n_iter);
                if (done) break;
                stretch = n_iter - before > stretch ? 4 : stretch < 1024 ? 8 * stretch : stretch;
                done = nu_iterate<E, W, LDK, TB>(sh, s_f, s_k, s_ip, s_in, s_jp, s_jn, ws, kws, kd, f, member, local_eps, max_iter, n_iter, stretch);
            } while (!done);
        } else {
            nu_iterate<E, W, LDK, TB>(sh, s_f, s_k, s_ip, s_in, s_jp, s_jn, ws, kws, kd, f, member, local_eps, max_iter, n_iter, 0x7fffffff);
        }
    } else {
        nu_iterate<E, W, LDK, TB>(sh, s_f, s_k, s_ip, s_in, s_jp, s_jn, ws, kws, kd, f, member, local_eps, max_iter, n_iter, 0x7fffffff);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int t = tid * E + e;
        if (t < ws) {
            const double y = (plus >> e) & 1u ? 1.0 : -1.0;
            const double a = sh.z[wave][t] * y + 0.0;   // (+ 0.0: a zero comes out as +0, as from alpha +- l)
            alpha_diff[t] = -(a - a_old[e]) * y;
            alpha[working_set[t]] = a;
        }
    }
    // diff[0] is the only word this variant reports (smo_kernel.cpp:283 leaves diff[1] alone).  It is written last,
    // behind a system-wide fence, so that a host thread polling it in host memory sees the kernel's end.
    if (tid == 0) {
        __threadfence_system();
        diff[0] = first_diff;
    }
}

// The solver workgroup asks for the rest of the CU's 160 KB of LDS as (unused) dynamic shared memory:
// no other workgroup can then be placed on its CU, so a kernel running concurrently on another
// stream cannot take issue slots, LDS bandwidth or L1 space away from the latency-bound solver.
static hipError_t reserve_cu(const void *kernel, size_t static_lds, size_t *dyn) {
    const size_t cu_lds = 160 * 1024;
    *dyn = cu_lds > static_lds + 1024 ? cu_lds - static_lds - 1024 : 0;
    return hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int) *dyn);
}

// The dynamic LDS a solver kernel is launched with on the current device.  The attribute query and the opt-in are made
// once per kernel and device (whichever host thread comes first), not per launch.
static int solver_dyn_lds(const void *kernel, size_t *dyn) {
    static std::mutex mu;
    static std::map<std::pair<const void *, int>, size_t> table;
    int dev = 0;
    TSVM_HIP(hipGetDevice(&dev));
    std::lock_guard<std::mutex> lock(mu);
    auto it = table.find(std::make_pair(kernel, dev));
    if (it == table.end()) {
        hipFuncAttributes fa;
        TSVM_HIP(hipFuncGetAttributes(&fa, kernel));
        size_t d = 0;
        TSVM_HIP(reserve_cu(kernel, fa.sharedSizeBytes, &d));
        it = table.emplace(std::make_pair(kernel, dev), d).first;
    }
    *dyn = it->second;
    return 0;
}

extern "C" {

static int solver_ldk(int ws_size) { return ws_size <= SV_LD ? SV_LD : (ws_size <= 2 * SV_LD ? 2 * SV_LD : 4 * SV_LD); }

size_t tsvm_smo_solve_workspace(int ws_size) {
    if (ws_size < 0) return 0;
    return sizeof(double) * (size_t) ws_size * (size_t) solver_ldk(ws_size) + 256;
}

// A float block needs float rows (a double row's values would be rounded).
static bool block_type_ok(int block_type, int row_type) {
    return block_type == TSVM_ROW_F64 || (block_type == TSVM_ROW_F32 && row_type == TSVM_ROW_F32);
}

static int launch_gather(const void *k_rows, int row_type, const int *slots, int64_t ld, const int *working_set, int ws,
                         void *workspace, int block_type, hipStream_t s) {
    TSVM_REQUIRE(row_type == TSVM_ROW_F64 || row_type == TSVM_ROW_F32, "smo_solve: unknown row type %d", row_type);
    TSVM_REQUIRE(block_type_ok(block_type, row_type), "smo_solve: block type %d not valid for row type %d", block_type, row_type);
    if (row_type == TSVM_ROW_F32 && block_type == TSVM_ROW_F32)
        hipLaunchKernelGGL((gather_ws_block_kernel<float, float>), dim3(ws), dim3(256), 0, s, (const float *) k_rows, slots, ld,
                           working_set, ws, solver_ldk(ws), (float *) workspace);
    else if (row_type == TSVM_ROW_F32)
        hipLaunchKernelGGL((gather_ws_block_kernel<float, double>), dim3(ws), dim3(256), 0, s, (const float *) k_rows, slots, ld,
                           working_set, ws, solver_ldk(ws), (double *) workspace);
    else
        hipLaunchKernelGGL((gather_ws_block_kernel<double, double>), dim3(ws), dim3(256), 0, s, (const double *) k_rows, slots, ld,
                           working_set, ws, solver_ldk(ws), (double *) workspace);
    TSVM_LAUNCH_CHECK();
    return 0;
}

#define TSVM_LAUNCH_SOLVER(KERNEL, TB, EVAL, WVAL, LDKVAL, ...)                                                \
    do {                                                                                                       \
        size_t dyn_ = 0;                                                                                       \
        if (solver_grid_ != TSVM_SOLVER_GRID_ON_XCD) {                                                         \
            const int rc_ = solver_dyn_lds(reinterpret_cast<const void *>(KERNEL<EVAL, WVAL, LDKVAL, TB>), &dyn_); \
            if (rc_) return rc_;                                                                               \
        }                                                                                                      \
        hipLaunchKernelGGL((KERNEL<EVAL, WVAL, LDKVAL, TB>), dim3(solver_grid_), dim3(64 * WVAL), dyn_, s, __VA_ARGS__); \
    } while (0)

// Up to 256 elements one wavefront alone, without a barrier (0.59 / 0.65 / 0.76 us per iteration at 64 / 128 / 256
// elements; four wavefronts take 0.95 / 0.90 / 0.87); above that four, two or four elements per thread (two wavefronts
// of four elements at 512: 0.99 us, four of two: 0.95).
#define TSVM_DISPATCH_E_T(KERNEL, TB, ...)                                                      \
    do {                                                                                        \
        if (ws_size <= 64) TSVM_LAUNCH_SOLVER(KERNEL, TB, 1, 1, SV_LD, __VA_ARGS__);            \
        else if (ws_size <= 128) TSVM_LAUNCH_SOLVER(KERNEL, TB, 2, 1, SV_LD, __VA_ARGS__);      \
        else if (ws_size <= SV_LD) TSVM_LAUNCH_SOLVER(KERNEL, TB, 4, 1, SV_LD, __VA_ARGS__);    \
        else if (ws_size <= 2 * SV_LD) TSVM_LAUNCH_SOLVER(KERNEL, TB, 2, 4, 2 * SV_LD, __VA_ARGS__); \
        else TSVM_LAUNCH_SOLVER(KERNEL, TB, 4, 4, 4 * SV_LD, __VA_ARGS__);                      \
    } while (0)

// (kws_: the block; block_type_: its element type)
#define TSVM_DISPATCH_E(KERNEL, PRE, POST)                                                                           \
    do {                                                                                                             \
        if (block_type_ == TSVM_ROW_F32) {                                                                           \
            const float *kws = (const float *) kws_;                                                                 \
            TSVM_DISPATCH_E_T(KERNEL, float, TSVM_UNPACK PRE, kws, TSVM_UNPACK POST);                                \
        } else {                                                                                                     \
            const double *kws = (const double *) kws_;                                                               \
            TSVM_DISPATCH_E_T(KERNEL, double, TSVM_UNPACK PRE, kws, TSVM_UNPACK POST);                               \
        }                                                                                                            \
    } while (0)
#define TSVM_UNPACK(...) __VA_ARGS__

int tsvm_c_smo_solve(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                     int ws_size, double Cp, double Cn, const void *k_rows, int row_type, const int *slots, int64_t ld,
                     const double *k_diag, double eps, double *diff, int max_iter, void *workspace,
                     tsvm_stream stream) {
    TSVM_REQUIRE(y && f_val && alpha && alpha_diff && working_set && k_rows && k_diag && diff && workspace,
                 "tsvm_c_smo_solve: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_c_smo_solve: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    hipStream_t s = tsvm_s(stream);
    int *gate_ = nullptr;
    const int epoch_ = 0, target_xcd_ = 0, target_cu_ = -1, solver_grid_ = 1;
    const int block_type_ = row_type;   // the block keeps the rows' element type
    int rc = launch_gather(k_rows, row_type, slots, ld, working_set, ws_size, workspace, block_type_, s);
    if (rc) return rc;
    const void *kws_ = workspace;
    TSVM_DISPATCH_E(c_smo_solve_kernel, (y, f_val, alpha, alpha_diff, working_set, ws_size, Cp, Cn),
                    (k_diag, eps, diff, max_iter, gate_, epoch_, target_xcd_, target_cu_));
    TSVM_LAUNCH_CHECK();
    return 0;
}

// c_smo_solve for callers that cannot allocate: the ws x ws block that tsvm_c_smo_solve gathers into the caller's
// workspace goes into a file-scope device array instead (8 MiB, held by every device the library runs on until the
// process ends).  Its device address is looked up once per device; host code never uses the array's name otherwise.
static __device__ __align__(256) double g_solver_block[(size_t) MAX_WS * MAX_WS];
#define TSVM_MAX_DEVICES 64
static double *g_solver_block_ptr[TSVM_MAX_DEVICES];
static std::mutex g_solver_block_mutex;

static int solver_block_address(double **out) {
    int dev = 0;
    TSVM_HIP(hipGetDevice(&dev));
    TSVM_REQUIRE(dev >= 0 && dev < TSVM_MAX_DEVICES, "tsvm_c_smo_solve_static: device ordinal %d outside [0, %d)", dev,
                 TSVM_MAX_DEVICES);
    std::lock_guard<std::mutex> lock(g_solver_block_mutex);
    if (!g_solver_block_ptr[dev]) {
        double *p = nullptr;
        TSVM_HIP(hipGetSymbolAddress((void **) &p, HIP_SYMBOL(g_solver_block)));
        TSVM_REQUIRE(p != nullptr, "tsvm_c_smo_solve_static: no device address for the static block");
        g_solver_block_ptr[dev] = p;
    }
    *out = g_solver_block_ptr[dev];
    return 0;
}

int tsvm_c_smo_solve_static_init(void) {
    double *block = nullptr;
    int rc = solver_block_address(&block);
    if (rc) return rc;
    size_t dyn = 0;
#define SV_EVERY(TB)                                                                                                         \
    reinterpret_cast<const void *>(c_smo_solve_kernel<1, 1, SV_LD, TB>), reinterpret_cast<const void *>(c_smo_solve_kernel<2, 1, SV_LD, TB>), \
        reinterpret_cast<const void *>(c_smo_solve_kernel<4, 1, SV_LD, TB>), reinterpret_cast<const void *>(c_smo_solve_kernel<2, 4, 2 * SV_LD, TB>), \
        reinterpret_cast<const void *>(c_smo_solve_kernel<4, 4, 4 * SV_LD, TB>)
    const void *kernels[] = {SV_EVERY(float), SV_EVERY(double)};
#undef SV_EVERY
    for (const void *k : kernels) {
        rc = solver_dyn_lds(k, &dyn);
        if (rc) return rc;
    }
    return 0;
}

int tsvm_c_smo_solve_static(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                            int ws_size, double Cp, double Cn, const void *k_rows, int row_type, const int *slots, int64_t ld,
                            const double *k_diag, double eps, double *diff, int max_iter, tsvm_stream stream) {
    TSVM_REQUIRE(y && f_val && alpha && alpha_diff && working_set && k_rows && k_diag && diff,
                 "tsvm_c_smo_solve_static: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_c_smo_solve_static: ws_size %d outside [1, %d] (the static block holds %d x %d values)",
                 ws_size, MAX_WS, MAX_WS, MAX_WS);
    double *block = nullptr;
    int rc = solver_block_address(&block);
    if (rc) return rc;
    hipStream_t s = tsvm_s(stream);
    int *gate_ = nullptr;
    const int epoch_ = 0, target_xcd_ = 0, target_cu_ = -1, solver_grid_ = 1;
    // the gather writes every element of the ws x ldk block the solver reads (columns beyond ws as zeros), so
    // nothing of the previous call's content is read
    const int block_type_ = row_type;
    rc = launch_gather(k_rows, row_type, slots, ld, working_set, ws_size, block, block_type_, s);
    if (rc) return rc;
    const void *kws_ = block;
    TSVM_DISPATCH_E(c_smo_solve_kernel, (y, f_val, alpha, alpha_diff, working_set, ws_size, Cp, Cn),
                    (k_diag, eps, diff, max_iter, gate_, epoch_, target_xcd_, target_cu_));
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_smo_solve_block_ld(int ws_size) { return ws_size < 1 ? 0 : solver_ldk(ws_size); }

int tsvm_smo_gather_block(const void *k_rows, int row_type, const int *slots, int64_t ld, const int *cols, int ws_size,
                          void *kws, int block_type, tsvm_stream stream) {
    TSVM_REQUIRE(k_rows && cols && kws, "tsvm_smo_gather_block: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_smo_gather_block: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    return launch_gather(k_rows, row_type, slots, ld, cols, ws_size, kws, block_type, tsvm_s(stream));
}

int tsvm_smo_gather_block_by_id(const void *k_rows, int row_type, const int *slot_of_id, int64_t ld, const int *ids,
                                int ws_size, void *kws, int block_type, int *slots_out, tsvm_stream stream) {
    TSVM_REQUIRE(k_rows && slot_of_id && ids && kws && slots_out, "tsvm_smo_gather_block_by_id: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_smo_gather_block_by_id: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    TSVM_REQUIRE(row_type == TSVM_ROW_F64 || row_type == TSVM_ROW_F32, "tsvm_smo_gather_block_by_id: unknown row type %d", row_type);
    TSVM_REQUIRE(block_type_ok(block_type, row_type), "tsvm_smo_gather_block_by_id: block type %d not valid for row type %d", block_type,
                 row_type);
    if (row_type == TSVM_ROW_F32 && block_type == TSVM_ROW_F32)
        hipLaunchKernelGGL((gather_ws_block_by_id_kernel<float, float>), dim3(ws_size), dim3(256), 0, tsvm_s(stream),
                           (const float *) k_rows, slot_of_id, ld, ids, ws_size, solver_ldk(ws_size), (float *) kws, slots_out);
    else if (row_type == TSVM_ROW_F32)
        hipLaunchKernelGGL((gather_ws_block_by_id_kernel<float, double>), dim3(ws_size), dim3(256), 0, tsvm_s(stream),
                           (const float *) k_rows, slot_of_id, ld, ids, ws_size, solver_ldk(ws_size), (double *) kws, slots_out);
    else
        hipLaunchKernelGGL((gather_ws_block_by_id_kernel<double, double>), dim3(ws_size), dim3(256), 0, tsvm_s(stream),
                           (const double *) k_rows, slot_of_id, ld, ids, ws_size, solver_ldk(ws_size), (double *) kws, slots_out);
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_row_slots_assign(const int *ids_new, int n_new, int *slot_of_id, int *state, int *miss_ids, int *miss_slots,
                          const int *ids_ws, int ws_size, int *slots_ws, int *info, tsvm_stream stream) {
    TSVM_REQUIRE(ids_new && slot_of_id && state && miss_ids && miss_slots && ids_ws && slots_ws && info,
                 "tsvm_row_slots_assign: null pointer");
    TSVM_REQUIRE(n_new >= 0 && n_new <= MAX_WS && ws_size >= 0 && ws_size <= MAX_WS, "tsvm_row_slots_assign: sizes %d, %d outside [0, %d]",
                 n_new, ws_size, MAX_WS);
    hipLaunchKernelGGL(row_slots_assign_kernel, dim3(1), dim3(RA_T), 0, tsvm_s(stream), ids_new, n_new, slot_of_id, state, miss_ids,
                       miss_slots, ids_ws, ws_size, slots_ws, info);
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_smo_start(double *alpha_diff, int n_diff, void *kws, int block_type, int ws_size, int *slot_of_id, int n_ids, int *state,
                   int *gate, tsvm_stream stream) {
    TSVM_REQUIRE(alpha_diff && kws && n_diff >= 0 && n_ids >= 0 && (n_ids == 0 || slot_of_id), "tsvm_smo_start: bad arguments");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_smo_start: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    const int ldk = solver_ldk(ws_size);
    const int64_t most = std::max<int64_t>(std::max(n_diff, n_ids), ws_size < ldk ? (int64_t) ws_size * ldk : 1);
    const dim3 grid((unsigned) std::min<int64_t>((most + 255) / 256, 1024));
    if (block_type == TSVM_ROW_F32)
        hipLaunchKernelGGL(smo_start_kernel<float>, grid, dim3(256), 0, tsvm_s(stream), alpha_diff, n_diff, (float *) kws, ws_size, ldk, slot_of_id,
                           n_ids, state, gate);
    else
        hipLaunchKernelGGL(smo_start_kernel<double>, grid, dim3(256), 0, tsvm_s(stream), alpha_diff, n_diff, (double *) kws, ws_size, ldk, slot_of_id,
                           n_ids, state, gate);
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_smo_warm_block(const void *kws, int block_type, int ws_size, int xcd, int *sink, tsvm_stream stream) {
    TSVM_REQUIRE(kws && sink, "tsvm_smo_warm_block: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_smo_warm_block: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    TSVM_REQUIRE(block_type == TSVM_ROW_F64 || block_type == TSVM_ROW_F32, "tsvm_smo_warm_block: unknown block type %d", block_type);
    TSVM_REQUIRE(xcd >= 0 && xcd < TSVM_SOLVER_GRID_ON_XCD, "tsvm_smo_warm_block: xcd %d outside [0, %d)", xcd, TSVM_SOLVER_GRID_ON_XCD);
    const size_t bytes = (size_t) ws_size * solver_ldk(ws_size) * (block_type == TSVM_ROW_F32 ? sizeof(float) : sizeof(double));
    if (bytes > SV_L2_BYTES) return 0;
    hipLaunchKernelGGL(warm_block_kernel, dim3(8 * SV_WARM_SLICES), dim3(256), 0, tsvm_s(stream), (const uint4 *) kws, (unsigned) (bytes / 16), xcd, sink);
    TSVM_LAUNCH_CHECK();
    return 0;
}

static int c_block(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set, int ws_size,
                   double Cp, double Cn, const void *kws_, int block_type_, const double *k_diag, double eps, double *diff,
                   int max_iter, int *gate_, int epoch_, int target_xcd_, int target_cu_, tsvm_stream stream) {
    TSVM_REQUIRE(y && f_val && alpha && alpha_diff && working_set && kws_ && k_diag && diff, "tsvm_c_smo_solve_block: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_c_smo_solve_block: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    TSVM_REQUIRE(block_type_ == TSVM_ROW_F64 || block_type_ == TSVM_ROW_F32, "tsvm_c_smo_solve_block: unknown block type %d", block_type_);
    hipStream_t s = tsvm_s(stream);
    const int solver_grid_ = !gate_ ? 1 : target_cu_ < 0 ? TSVM_SOLVER_GRID_ON_XCD : TSVM_SOLVER_GRID_ON_CU;
    TSVM_DISPATCH_E(c_smo_solve_kernel, (y, f_val, alpha, alpha_diff, working_set, ws_size, Cp, Cn),
                    (k_diag, eps, diff, max_iter, gate_, epoch_, target_xcd_, target_cu_));
    TSVM_LAUNCH_CHECK();
    return 0;
}

static int nu_block(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set, int ws_size,
                    double C, const void *kws_, int block_type_, const double *k_diag, double eps, double *diff, int max_iter,
                    int *gate_, int epoch_, int target_xcd_, int target_cu_, tsvm_stream stream) {
    TSVM_REQUIRE(y && f_val && alpha && alpha_diff && working_set && kws_ && k_diag && diff, "tsvm_nu_smo_solve_block: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_nu_smo_solve_block: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    TSVM_REQUIRE(block_type_ == TSVM_ROW_F64 || block_type_ == TSVM_ROW_F32, "tsvm_nu_smo_solve_block: unknown block type %d", block_type_);
    hipStream_t s = tsvm_s(stream);
    const int solver_grid_ = !gate_ ? 1 : target_cu_ < 0 ? TSVM_SOLVER_GRID_ON_XCD : TSVM_SOLVER_GRID_ON_CU;
    TSVM_DISPATCH_E(nu_smo_solve_kernel, (y, f_val, alpha, alpha_diff, working_set, ws_size, C),
                    (k_diag, eps, diff, max_iter, gate_, epoch_, target_xcd_, target_cu_));
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_c_smo_solve_block(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                           int ws_size, double Cp, double Cn, const void *kws, int block_type, const double *k_diag, double eps,
                           double *diff, int max_iter, tsvm_stream stream) {
    return c_block(y, f_val, alpha, alpha_diff, working_set, ws_size, Cp, Cn, kws, block_type, k_diag, eps, diff, max_iter, nullptr, 0,
                   0, -1, stream);
}

int tsvm_nu_smo_solve_block(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                            int ws_size, double C, const void *kws, int block_type, const double *k_diag, double eps, double *diff,
                            int max_iter, tsvm_stream stream) {
    return nu_block(y, f_val, alpha, alpha_diff, working_set, ws_size, C, kws, block_type, k_diag, eps, diff, max_iter, nullptr, 0, 0,
                    -1, stream);
}

int tsvm_c_smo_solve_block_on_xcd(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                                  int ws_size, double Cp, double Cn, const void *kws, int block_type, const double *k_diag, double eps,
                                  double *diff, int max_iter, int *gate, int epoch, int xcd, tsvm_stream stream) {
    TSVM_REQUIRE(gate && epoch >= 1 && xcd >= 0 && xcd < TSVM_SOLVER_GRID_ON_XCD, "tsvm_c_smo_solve_block_on_xcd: bad gate, epoch or xcd");
    return c_block(y, f_val, alpha, alpha_diff, working_set, ws_size, Cp, Cn, kws, block_type, k_diag, eps, diff, max_iter, gate, epoch,
                   xcd, -1, stream);
}

int tsvm_nu_smo_solve_block_on_xcd(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                                   int ws_size, double C, const void *kws, int block_type, const double *k_diag, double eps,
                                   double *diff, int max_iter, int *gate, int epoch, int xcd, tsvm_stream stream) {
    TSVM_REQUIRE(gate && epoch >= 1 && xcd >= 0 && xcd < TSVM_SOLVER_GRID_ON_XCD, "tsvm_nu_smo_solve_block_on_xcd: bad gate, epoch or xcd");
    return nu_block(y, f_val, alpha, alpha_diff, working_set, ws_size, C, kws, block_type, k_diag, eps, diff, max_iter, gate, epoch, xcd,
                    -1, stream);
}

int tsvm_c_smo_solve_block_on_cu(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                                 int ws_size, double Cp, double Cn, const void *kws, int block_type, const double *k_diag, double eps,
                                 double *diff, int max_iter, int *gate, int epoch, int xcd, int cu, tsvm_stream stream) {
    TSVM_REQUIRE(gate && epoch >= 1 && xcd >= 0 && xcd < TSVM_SOLVER_GRID_ON_XCD && cu >= 0, "tsvm_c_smo_solve_block_on_cu: bad gate, epoch, xcd or cu");
    return c_block(y, f_val, alpha, alpha_diff, working_set, ws_size, Cp, Cn, kws, block_type, k_diag, eps, diff, max_iter, gate, epoch,
                   xcd, cu, stream);
}

int tsvm_nu_smo_solve_block_on_cu(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                                  int ws_size, double C, const void *kws, int block_type, const double *k_diag, double eps,
                                  double *diff, int max_iter, int *gate, int epoch, int xcd, int cu, tsvm_stream stream) {
    TSVM_REQUIRE(gate && epoch >= 1 && xcd >= 0 && xcd < TSVM_SOLVER_GRID_ON_XCD && cu >= 0, "tsvm_nu_smo_solve_block_on_cu: bad gate, epoch, xcd or cu");
    return nu_block(y, f_val, alpha, alpha_diff, working_set, ws_size, C, kws, block_type, k_diag, eps, diff, max_iter, gate, epoch, xcd,
                    cu, stream);
}

int tsvm_where(int *out, int n, tsvm_stream stream) {
    TSVM_REQUIRE(out && n >= 0 && n <= 1024, "tsvm_where: bad arguments");
    if (n == 0) return 0;
    hipLaunchKernelGGL(where_kernel, dim3(n), dim3(64), 0, tsvm_s(stream), out);
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_nu_smo_solve(const int *y, const double *f_val, double *alpha, double *alpha_diff, const int *working_set,
                      int ws_size, double C, const void *k_rows, int row_type, const int *slots, int64_t ld,
                      const double *k_diag, double eps, double *diff, int max_iter, void *workspace,
                      tsvm_stream stream) {
    TSVM_REQUIRE(y && f_val && alpha && alpha_diff && working_set && k_rows && k_diag && diff && workspace,
                 "tsvm_nu_smo_solve: null pointer");
    TSVM_REQUIRE(ws_size >= 1 && ws_size <= MAX_WS, "tsvm_nu_smo_solve: ws_size %d outside [1, %d]", ws_size, MAX_WS);
    hipStream_t s = tsvm_s(stream);
    int *gate_ = nullptr;
    const int epoch_ = 0, target_xcd_ = 0, target_cu_ = -1, solver_grid_ = 1;
    const int block_type_ = row_type;
    int rc = launch_gather(k_rows, row_type, slots, ld, working_set, ws_size, workspace, block_type_, s);
    if (rc) return rc;
    const void *kws_ = workspace;
    TSVM_DISPATCH_E(nu_smo_solve_kernel, (y, f_val, alpha, alpha_diff, working_set, ws_size, C),
                    (k_diag, eps, diff, max_iter, gate_, epoch_, target_xcd_, target_cu_));
    TSVM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
