// CSMOSolver / NuSMOSolver: the outer SMO loop (src/thundersvm/solver/csmosolver.cpp:10-121,
// nusmosolver.cpp) driving the gfx950 kernels.  f, alpha, y, the working set and the ws x n kernel
// rows stay in HBM for the whole solve; per outer iteration the host reads back 16 bytes (diff).
#pragma once
#include <memory>
#include <string>
#include "kernelmatrix.h"

struct SolverTrace {          // optional per-iteration record (parity debugging and tests)
    int cap_iters = 0;
    std::vector<double> diff;   // [iters][2]
    std::vector<int> ws;        // [iters][ws_size]
    int ws_size = 0;
};

struct SolverStats {
    long long n_iter = 0;       // outer iterations
    long long local_iter = 0;   // inner iterations summed
    double obj = 0;
    // accumulated device time per phase in ms (only filled when profile == true)
    double ms_select = 0, ms_get_rows = 0, ms_local = 0, ms_update_f = 0;
    double ms_wall = 0, ms_setup = 0;   // host wall-clock of the whole solve / of everything before the first iteration
    // kernel-row cache
    long long cache_lookups = 0, cache_hits = 0;
    long long cache_rows = 0;     // capacity in rows (0: cache not used)
    bool cache_disabled = false;  // switched off after the warm-up because it was not hitting
    int ws_size = 0;              // working-set size of the solve
    long long rows_computed = 0;  // kernel rows get_rows produced (cache misses), summed over the outer iterations
    long long update_rows = 0;    // kernel rows update_f read (non-zero alpha_diff entries), counted only when profiling
    int solver_xcd = -1;          // several class pairs in flight: the die this pair's local solver ran on (-1: not known)
    double ms_start = 0, ms_end = 0;   // host clock at the solve's start and end, in ms since the process's first solve
};

class SolveTask;

namespace tsvm {
// Spins until *word no longer holds `pending`.  Every 200 ms `stream_state()` is asked for the state of the stream
// that is to write the word (hipSuccess: everything enqueued has run; hipErrorNotReady: still running; anything else
// is thrown as that error).  Throws std::runtime_error when the stream has drained without the word changing, or
// when timeout_ms have passed: a solver kernel that never finishes must not hang its caller for good (the
// reference's blocking copies surface such failures through CUDA_CHECK, include/thundersvm/util/common.h:33-42).
void wait_while_pending(const volatile uint64_t *word, uint64_t pending, long long timeout_ms, hipError_t (*stream_state)(void *),
                        void *stream);
long long solver_timeout_ms();   // TSVM_SOLVER_TIMEOUT_MS, default 300,000

// What a solve that has the chip to itself runs where, by the time that the rows of an iteration take (dense rows).
struct ChipSplit {
    // Of m dense rows of n values, on the whole chip.  (Every column counts.  Indicator columns are left to the epilogue, whose
    // share makes up for it: 512 x 425,000 values of 10 + 44 columns take 1.7 ps each, 1.9 by this.)
    static double rows_seconds(size_t features, long long m, long long n) { return 2.0 * (double) ((features + 15) / 16 * 16) / 6.6e13 * (double) m * (double) n; }
    // Whether the rows go ahead of the block and the solver (they are enqueued when the selection has reported, and not when the solver
    // has its CU): when they, by the previous iteration's number of them, outlast the solver's ~0.4 ms and a block that has to find
    // its CUs among them (priced as 136 of its 256 tiles on 8 CUs, some 35 times what it takes alone).  Until then they wait for the
    // solver, whose launch reads the block into its L2 from the CUs that the rows would hold.  With 512 rows computed an iteration
    // the line lies at 67,000 instances of 784 columns, 120,000 of 300 and 300,000 of 90.  A call in ms, by the rule / always ahead /
    // always behind the solver:
    //   784 columns    20,000   50.1 /  51.9 /  50.1      40,000   92.8 /  90.5 /  92.9      60,000   176 /   170 /   176      90,000   309 /   308 /   315
    //   300 columns    60,000    183 /   219 /   183     120,000    461 /   557 /   461
    //    90 columns    40,000   66.1 /  77.3 /  66.0     150,000    296 /   322 /   296     300,000   796 /   833 /   795     500,000 2,715 / 2,665 / 2,719
    // (It leaves 3 % at 784 columns below its line, and 2 % far above it at 90, where fewer rows are computed in most iterations.)
    static bool block_beside_rows(size_t features, int ws, double rows_seconds) {
        return 32.0 * 0.53 * ChipSplit::rows_seconds(features, ws, ws) + 0.4e-3 <= rows_seconds;
    }
    // (dense data only: rows_seconds prices every column, of sparse rows of 50 entries among 20,958 columns 400 times too high)
    static bool rows_ahead(bool dense, size_t features, int ws, double rows_seconds) { return dense && block_beside_rows(features, ws, rows_seconds); }
    // Whether the block is read into the solver's L2 a second time, behind the rows that stream through it beside the solver and
    // take its place there (epsilon-SVR 40000x90, rows for 42 us beside a solver of 310: 88.4 -> 81.3 ms), unless they take
    // about as long as the solver (20000x784, 340 us: 50.2 -> 50.3).  Behind rows that go ahead the block may not be there yet.
    static bool warm_behind_rows(bool block_beside, double rows_seconds) { return !block_beside && rows_seconds > 0 && rows_seconds < 0.1e-3; }
};

// Which selections of n instances are guided by the one before (tsvm_update_f_select_guided).  The first is not: the first solve moves f
// by more than a guide reaches, from values that are mostly equal.  Where the guide does not decide, one workgroup resolves
// the digits of all instances, which takes time with their number, while what a guide that decides saves hardly grows:
//   instances              20,000   40,000  100,000  300,000  1,000,000  16,000,000
//   by digits, us            33.7     32.6     39.8     52.3       71.2         471   (with update_f of one row in front)
//   guided and decided       25.4     25.2     27.7     34.3       48.9         327
//   guided and not            104      157      362    1,009      3,609      58,000
// So behind one that was not, the next go by digits, twice as many each time up to n / 1,250 (32 at least): if every guide failed they would cost
// some 4 us a selection whatever n is.  As many decided in a row, which have saved more than that failure cost, and it starts with two again.
// Above 2^20 instances, where an iteration takes a millisecond or more and a guide saves 2 % of it or less, there are none.
class GuideSchedule {
public:
    explicit GuideSchedule(long long n) : none_(n > (1 << 20)), most_(none_ ? 0 : (int) (n / 1250 > 32 ? n / 1250 : 32)) {}
    // Whether the next selection is guided; missed: a guide has failed since this was last asked.
    bool next(bool missed) {
        if (none_) return false;
        if (missed) {
            unguided_ = stretch_;
            stretch_ = 2 * stretch_ < most_ ? 2 * stretch_ : most_;
            decided_ = 0;
        }
        if (unguided_ > 0) {
            --unguided_;
            return false;
        }
        if (++decided_ == most_) stretch_ = 2;
        return true;
    }

private:
    const bool none_;
    const int most_;
    int unguided_ = 1, stretch_ = 2, decided_ = 0;
};
}  // namespace tsvm

class CSMOSolver {
public:
    virtual ~CSMOSolver() = default;
    void solve(const KernelMatrix &k_mat, const std::vector<int> &y, std::vector<float_type> &alpha, float_type &rho,
               std::vector<float_type> &f_val, float_type eps, float_type Cp, float_type Cn, int ws_size,
               int out_max_iter) const;

    mutable SolverStats stats;
    SolverTrace *trace = nullptr;
    bool profile = false;
    // Budget of the HBM kernel-row cache in bytes: -1 = nine tenths of the free device memory, 0 = no cache.
    long long cache_bytes = -1;

protected:
    friend class SolveTask;
    friend struct SmallBatch;
    virtual bool is_nu() const { return false; }
    virtual float_type calculate_rho(const std::vector<float_type> &f_val, const std::vector<int> &y,
                                     std::vector<float_type> &alpha, float_type Cp, float_type Cn) const;
    void init_f(const std::vector<float_type> &alpha, const std::vector<int> &y, const KernelMatrix &k_mat,
                float_type *d_f) const;
    float_type calculate_obj(const std::vector<float_type> &f_val, const std::vector<float_type> &alpha,
                             const std::vector<int> &y) const;
};

class NuSMOSolver : public CSMOSolver {
public:
    explicit NuSMOSolver(bool for_svr) : for_svr(for_svr) {}

protected:
    bool is_nu() const override { return true; }
    float_type calculate_rho(const std::vector<float_type> &f_val, const std::vector<int> &y,
                             std::vector<float_type> &alpha, float_type Cp, float_type Cn) const override;

private:
    bool for_svr;
};

// One SMO solve as a resumable sequence of enqueue steps.  CSMOSolver::solve runs one task to completion; a
// one-vs-one run keeps several tasks (class pairs) in flight and enqueues their steps in turn.  The local
// solver is a single workgroup bound by latency; it runs on compute units of its own (one per XCD and lane), by a stream that is restricted to
// them or, in a task that runs alone, by finding its unit itself; what runs beside it is on a stream restricted to the remaining ones, so the
// solver of an iteration runs next to that iteration's get_rows.  Where such streams cannot be had the task
// uses one ordinary stream, and the driver of several tasks keeps their solver phases apart from their
// chip-wide phases with events.  The steps of one outer iteration:
//   enqueue_select, enqueue_block, enqueue_solver, enqueue_rows, enqueue_update, finish_iteration
// (enqueue_rows before enqueue_block when the block is gathered from the stored rows: block_needs_rows()).
class SolveTask {
public:
    // pool / pool_bytes: device memory for the kernel rows (nullptr: taken from the process-wide arena
    // according to solver.cache_bytes).  lane / n_lanes: which of the tasks advanced side by side this one is;
    // every lane's local solver gets CUs of its own.
    SolveTask(const CSMOSolver &solver, const KernelMatrix &k_mat, const std::vector<int> &y, std::vector<float_type> &alpha,
              float_type &rho, std::vector<float_type> &f_val, float_type eps, float_type Cp, float_type Cn, int ws_size,
              int out_max_iter, void *pool = nullptr, size_t pool_bytes = 0, int lane = 0, int n_lanes = 1);
    ~SolveTask();
    SolveTask(const SolveTask &) = delete;
    SolveTask &operator=(const SolveTask &) = delete;

    void enqueue_select();
    void enqueue_rows();
    void enqueue_block();
    void enqueue_solver();
    void enqueue_update();
    bool finish_iteration();   // waits for this iteration's diff; true once the solve is complete and its results are written
    // For a caller that advances several tasks from one thread without blocking on any of them:
    // rows_ready(): enqueue_rows would not wait (the newly selected ids the host-side row cache needs have arrived, or
    // are not needed); iteration_done(): finish_iteration would not wait.  iteration_done() throws like the blocking
    // wait when the solver's stream has drained without a report or nothing has been heard for the time-out.
    bool rows_ready() const;
    bool iteration_done();
    bool block_needs_rows() const;
    bool split_streams() const;   // the local solver runs on CUs of its own, next to this task's (and other tasks') chip-wide kernels
    hipStream_t stream() const;
    const SolverStats &stats() const;
    static size_t min_pool_bytes(const KernelMatrix &k_mat, int ws_size);
    static bool cu_split_available();   // the device is one whose CUs this code knows how to divide

private:
    struct Impl;
    Impl *impl_;
};

// One of several small problems that are solved by one kernel launch (smo_small.hip): its y = +1 instances are n_pos rows
// of the batch's kernel matrix from row_pos on, its y = -1 instances n_neg rows from row_neg on.
struct SmallSolve {
    const CSMOSolver *solver;
    int row_pos, n_pos, row_neg, n_neg, ws_size;
    float_type Cp, Cn;
    const std::vector<int> *y;
    std::vector<float_type> *alpha, *f_val;
    float_type *rho;
    bool solved = false;        // false after run(): alpha and f_val are untouched, the problem is for a SolveTask
    SolverStats stats;

    static size_t slots(size_t n_pos, size_t n_neg);
    static bool takes(size_t n_pos, size_t n_neg, int ws_size);
    static bool takes_rows(size_t n_rows, size_t elem_size);
};
struct SmallBatch {             // problems with rows in one kernel matrix
    std::shared_ptr<const KernelMatrix> k_mat;
    std::vector<SmallSolve> solves;
    // Solves every problem of all batches, side by side as far as the row arena holds their matrices.  (All of one kind: C or
    // nu, and the same type of kernel row.)
    static void run(const std::vector<SmallBatch *> &batches, float_type eps, int out_max_iter);
    static bool is_nu(const SmallSolve &s) { return s.solver->is_nu(); }
    static void set_results(SmallSolve &s, long long n_iter, long long local_iter);   // rho and the statistics, once alpha and f are there
};
double ms_since_first_solve();   // the clock that SolverStats::ms_start and ms_end are read on
