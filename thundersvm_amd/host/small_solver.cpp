// Whole solves of small problems in one kernel (csrc/smo_small.hip): the kernel matrix of all problems' rows, one upload,
// one launch (more when a problem is not done within a launch's bound on its steps), one download.
#include "solver.h"

#include <algorithm>
#include <chrono>
#include <cstring>
#include <numeric>

using tsvm::abi_check;
using tsvm::DeviceBuffer;

size_t SmallSolve::slots(size_t n_pos, size_t n_neg) { return (n_pos + 3) / 4 * 4 + n_neg; }

// (an odd working set leaves its last place to chance in the shared window: that stays with SolveTask)
bool SmallSolve::takes(size_t n_pos, size_t n_neg, int ws_size) {
    return n_pos + n_neg >= 2 && slots(n_pos, n_neg) <= (size_t) tsvm_smo_small_max() && ws_size >= 2 && ws_size % 2 == 0 &&
           (size_t) ws_size <= n_pos + n_neg;
}

// The kernel matrix has to fit the row arena's budget; above 16,384 rows (1 GiB of floats) the pairs' own matrices are
// together no longer much more than the whole one.
bool SmallSolve::takes_rows(size_t n_rows, size_t elem_size) {
    return n_rows <= 16384 && n_rows * (n_rows + 8) * elem_size <= tsvm::RowArena::instance().auto_budget();
}

static size_t matrix_bytes(const KernelMatrix &k) {   // (three elements behind the last one are read)
    const size_t ld = (k.n_columns() + 7) / 8 * 8;
    return ((k.n_columns() * ld + 8) * k.row_elem_size() + 255) / 256 * 256;
}

static void run_together(const std::vector<SmallBatch *> &batches, float_type eps, int out_max_iter, size_t arena_bytes) {
    const auto wall0 = std::chrono::steady_clock::now();
    const double start_ms = ms_since_first_solve();
    hipStream_t stream = tsvm::work_stream();
    char *const arena = (char *) tsvm::RowArena::instance().acquire(arena_bytes, true);
    // alpha | f | states | problems | row numbers
    std::vector<tsvm_small_problem> host;
    std::vector<SmallSolve *> solves;
    std::vector<char *> matrices;
    size_t total = 0;
    int max_slots = 1, max_rows = 0;
    char *k = arena;
    for (SmallBatch *b : batches) {
        const int n_rows = (int) b->k_mat->n_columns();
        max_rows = std::max(max_rows, n_rows);
        matrices.push_back(k);
        for (SmallSolve &s : b->solves) {
            host.push_back({k, b->k_mat->diag(), (int64_t) (n_rows + 7) / 8 * 8, (int64_t) total, n_rows, s.row_pos, s.n_pos, s.row_neg, s.n_neg,
                            s.ws_size, std::max(100000, 100 * s.ws_size), 0, s.Cp, s.Cn});
            solves.push_back(&s);
            total += (size_t) s.n_pos + s.n_neg;
            max_slots = std::max(max_slots, (int) SmallSolve::slots(s.n_pos, s.n_neg));
        }
        k += matrix_bytes(*b->k_mat);
    }
    const int n_problems = (int) host.size(), row_type = batches[0]->k_mat->row_type();
    const bool nu = SmallBatch::is_nu(*solves[0]);
    std::vector<int> iota(max_rows);
    std::iota(iota.begin(), iota.end(), 0);
    const auto align = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t vec = align(total * sizeof(float_type)), states_at = 2 * vec, problems_at = states_at + align(n_problems * sizeof(tsvm_small_state));
    const size_t iota_at = problems_at + align(n_problems * sizeof(tsvm_small_problem)), bytes = iota_at + (size_t) max_rows * sizeof(int);
    DeviceBuffer<char> d(bytes);
    DeviceBuffer<int> d_ws((size_t) n_problems * tsvm_smo_small_max());
    std::vector<tsvm::HostStaging::Part> parts;
    for (int p = 0; p < n_problems; ++p) parts.push_back({solves[p]->alpha->data(), solves[p]->alpha->size() * sizeof(float_type), host[p].at * sizeof(float_type)});
    for (int p = 0; p < n_problems; ++p) parts.push_back({solves[p]->f_val->data(), solves[p]->f_val->size() * sizeof(float_type), vec + host[p].at * sizeof(float_type)});
    parts.push_back({host.data(), n_problems * sizeof(tsvm_small_problem), problems_at});
    parts.push_back({iota.data(), max_rows * sizeof(int), iota_at});
    tsvm::HostStaging::instance().upload(d.data(), parts, stream);
    const int *const d_iota = (const int *) (d.data() + iota_at);
    for (size_t b = 0; b < batches.size(); ++b) {
        const KernelMatrix &K = *batches[b]->k_mat;
        const int n_rows = (int) K.n_columns(), chunk = K.dense_layout() ? n_rows : 1024;   // (rows that are not stored dense are staged a few at a time)
        const int64_t ld = (int64_t) (n_rows + 7) / 8 * 8;
        for (int r = 0; r < n_rows; r += chunk)
            K.get_rows(d_iota + r, std::min(chunk, n_rows - r), matrices[b] + (size_t) r * ld * K.row_elem_size(), ld, nullptr, stream);
    }
    std::vector<char> got(problems_at);
    const tsvm_small_state *const states = (const tsvm_small_state *) (got.data() + states_at);
    // The kernel's own loops are bounded and every launch makes at least one outer iteration of a problem that is not done, so
    // what is not bounded is what the outer loop of SolveTask is not either: the iterations a problem needs.  Each launch is
    // waited for no longer than SolveTask waits for a solver, and has to have got further.
    for (long long done_before = -1, more = true; more;) {
        const bool first = done_before < 0;
        abi_check(tsvm_smo_solve_small(row_type, (const tsvm_small_problem *) (d.data() + problems_at), n_problems, max_slots,
                                       (tsvm_small_state *) (d.data() + states_at), d_ws.data(), (double *) d.data(), (double *) (d.data() + vec), nu,
                                       eps, out_max_iter, first, stream));
        try {
            tsvm::HostStaging::instance().download(d.data(), problems_at, [&](const char *from, size_t off, size_t len) {
                tsvm::parallel_memcpy(got.data() + off, from, len);
            }, stream, tsvm::solver_timeout_ms());
        } catch (...) {   // (the device may still be using them)
            d.abandon();
            d_ws.abandon();
            throw;
        }
        more = std::any_of(states, states + n_problems, [](const tsvm_small_state &s) { return s.status == 0; });
        const long long done = std::accumulate(states, states + n_problems, 0ll, [](long long sum, const tsvm_small_state &s) { return sum + s.iter; });
        if (more && done <= done_before) throw std::runtime_error("SmallBatch: a launch made no progress");
        done_before = done;
    }
    d.release(true);
    d_ws.release(true);
    const double wall = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - wall0).count();
#pragma omp parallel for schedule(dynamic, 1) num_threads(threads_for(total))
    for (int p = 0; p < n_problems; ++p) {
        SmallSolve &s = *solves[p];
        const tsvm_small_state &st = states[p];
        s.solved = st.status == 1;
        if (!s.solved) continue;
        const size_t n = s.alpha->size();
        memcpy(s.alpha->data(), got.data() + host[p].at * sizeof(float_type), n * sizeof(float_type));
        memcpy(s.f_val->data(), got.data() + vec + host[p].at * sizeof(float_type), n * sizeof(float_type));
        SmallBatch::set_results(s, st.iter, st.local_iter);
        SolverStats &o = s.stats;
        o.solver_xcd = st.xcd;
        o.ms_wall = wall;
        o.ms_start = start_ms;
        o.ms_end = start_ms + wall;
    }
    for (int p = 0; p < n_problems; ++p)
        if (solves[p]->solved)
            TSVM_LOG << "global iter = " << states[p].iter - 1 << ", total local iter = " << states[p].local_iter << ", diff = " << states[p].diff
                     << ", obj = " << solves[p]->stats.obj;
}

void SmallBatch::set_results(SmallSolve &s, long long n_iter, long long local_iter) {
    *s.rho = s.solver->calculate_rho(*s.f_val, *s.y, *s.alpha, s.Cp, s.Cn);
    SolverStats &o = s.stats;
    o.n_iter = n_iter;
    o.local_iter = local_iter;
    o.obj = s.solver->calculate_obj(*s.f_val, *s.alpha, *s.y);
    o.ws_size = s.ws_size;
    o.cache_rows = o.rows_computed = s.row_pos == s.row_neg ? s.n_pos : s.n_pos + s.n_neg;
    o.cache_lookups = o.cache_hits = s.ws_size + (n_iter - 1) * (s.ws_size / 2);   // (every row is there before the first lookup)
}

void SmallBatch::run(const std::vector<SmallBatch *> &batches, float_type eps, int out_max_iter) {
    std::vector<SmallBatch *> together;
    size_t bytes = 0;
    const auto flush = [&] {
        if (!together.empty()) run_together(together, eps, out_max_iter, bytes);
        together.clear();
        bytes = 0;
    };
    for (SmallBatch *b : batches) {
        if (b->solves.empty()) continue;
        const size_t mine = matrix_bytes(*b->k_mat);
        if (!together.empty() && bytes + mine > tsvm::RowArena::instance().auto_budget()) flush();
        together.push_back(b);
        bytes += mine;
    }
    flush();
}
