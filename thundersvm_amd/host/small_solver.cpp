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

// (an odd working set leaves its last place to chance in the shared window, and NaNs are nobody's problem: both stay
// with SolveTask)
bool SmallSolve::takes(size_t n_pos, size_t n_neg, int ws_size) {
    return n_pos + n_neg >= 2 && slots(n_pos, n_neg) <= (size_t) tsvm_smo_small_max() && ws_size >= 2 && ws_size % 2 == 0 &&
           (size_t) ws_size <= n_pos + n_neg;
}

// The kernel matrix has to fit the row arena's budget; above 16,384 rows (1 GiB of floats) the pairs' own matrices are
// together no longer much more than the whole one.
bool SmallSolve::takes_rows(size_t n_rows, size_t elem_size) {
    return n_rows <= 16384 && n_rows * (n_rows + 8) * elem_size <= tsvm::RowArena::instance().auto_budget();
}

void SmallSolve::run(const KernelMatrix &k_mat, std::vector<SmallSolve> &problems, float_type eps, int out_max_iter) {
    if (problems.empty()) return;
    const auto wall0 = std::chrono::steady_clock::now();
    const double start_ms = ms_since_first_solve();
    const int n_rows = (int) k_mat.n_columns(), n_problems = (int) problems.size();
    const int64_t ld = ((int64_t) n_rows + 7) / 8 * 8;
    const bool nu = problems[0].solver->is_nu();
    hipStream_t stream = tsvm::work_stream();
    char *const k = (char *) tsvm::RowArena::instance().acquire(((size_t) n_rows * ld + 8) * k_mat.row_elem_size(), true);

    // alpha | f | states | problems | row numbers
    std::vector<tsvm_small_problem> host(n_problems);
    size_t total = 0;
    int max_slots = 1;
    for (int p = 0; p < n_problems; ++p) {
        SmallSolve &s = problems[p];
        host[p] = {s.row_pos, s.n_pos, s.row_neg, s.n_neg, s.ws_size, std::max(100000, 100 * s.ws_size), s.Cp, s.Cn, (int64_t) total};
        total += (size_t) s.n_pos + s.n_neg;
        max_slots = std::max(max_slots, (int) slots(s.n_pos, s.n_neg));
    }
    std::vector<int> iota(n_rows);
    std::iota(iota.begin(), iota.end(), 0);
    const auto align = [](size_t v) { return (v + 255) / 256 * 256; };
    const size_t vec = align(total * sizeof(float_type)), states_at = 2 * vec, problems_at = states_at + align(n_problems * sizeof(tsvm_small_state));
    const size_t iota_at = problems_at + align(n_problems * sizeof(tsvm_small_problem)), bytes = iota_at + (size_t) n_rows * sizeof(int);
    DeviceBuffer<char> d(bytes);
    DeviceBuffer<int> d_ws((size_t) n_problems * tsvm_smo_small_max());
    std::vector<tsvm::HostStaging::Part> parts;
    for (int p = 0; p < n_problems; ++p) parts.push_back({problems[p].alpha->data(), problems[p].alpha->size() * sizeof(float_type), host[p].at * sizeof(float_type)});
    for (int p = 0; p < n_problems; ++p) parts.push_back({problems[p].f_val->data(), problems[p].f_val->size() * sizeof(float_type), vec + host[p].at * sizeof(float_type)});
    parts.push_back({host.data(), n_problems * sizeof(tsvm_small_problem), problems_at});
    parts.push_back({iota.data(), n_rows * sizeof(int), iota_at});
    tsvm::HostStaging::instance().upload(d.data(), parts, stream);
    // (rows that are not stored dense are staged a few at a time)
    const int chunk = k_mat.dense_layout() ? n_rows : 1024;
    const int *const d_iota = (const int *) (d.data() + iota_at);
    for (int r = 0; r < n_rows; r += chunk)
        k_mat.get_rows(d_iota + r, std::min(chunk, n_rows - r), k + (size_t) r * ld * k_mat.row_elem_size(), ld, nullptr, stream);
    std::vector<tsvm_small_state> states(n_problems);
    for (bool first = true, more = true; more; first = false) {
        abi_check(tsvm_smo_solve_small(k, k_mat.row_type(), ld, n_rows, k_mat.diag(), (const tsvm_small_problem *) (d.data() + problems_at),
                                       n_problems, max_slots, (tsvm_small_state *) (d.data() + states_at), d_ws.data(), (double *) d.data(),
                                       (double *) (d.data() + vec), nu, eps, out_max_iter, first, stream));
        std::vector<char> got(problems_at);
        tsvm::HostStaging::instance().download(d.data(), problems_at, [&](const char *from, size_t off, size_t len) {
            tsvm::parallel_memcpy(got.data() + off, from, len);
        }, stream);
        memcpy(states.data(), got.data() + states_at, n_problems * sizeof(tsvm_small_state));
        more = std::any_of(states.begin(), states.end(), [](const tsvm_small_state &s) { return s.status == 0; });
        if (more) continue;
        for (int p = 0; p < n_problems; ++p) {
            SmallSolve &s = problems[p];
            s.solved = states[p].status == 1;
            if (!s.solved) continue;
            const size_t n = s.alpha->size();
            memcpy(s.alpha->data(), got.data() + host[p].at * sizeof(float_type), n * sizeof(float_type));
            memcpy(s.f_val->data(), got.data() + vec + host[p].at * sizeof(float_type), n * sizeof(float_type));
        }
    }
    d.release(true);
    d_ws.release(true);
    const double wall = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - wall0).count();
    for (int p = 0; p < n_problems; ++p) {
        SmallSolve &s = problems[p];
        if (!s.solved) continue;
        const tsvm_small_state &st = states[p];
        *s.rho = s.solver->calculate_rho(*s.f_val, *s.y, *s.alpha, s.Cp, s.Cn);
        SolverStats &o = s.stats;
        o.n_iter = st.iter;
        o.local_iter = st.local_iter;
        o.obj = s.solver->calculate_obj(*s.f_val, *s.alpha, *s.y);
        o.ws_size = s.ws_size;
        o.cache_rows = o.rows_computed = s.row_pos == s.row_neg ? s.n_pos : s.n_pos + s.n_neg;
        o.cache_lookups = o.cache_hits = s.ws_size + (st.iter - 1LL) * (s.ws_size / 2);   // (every row is there before the first lookup)
        o.solver_xcd = st.xcd;
        o.ms_wall = wall;
        o.ms_start = start_ms;
        o.ms_end = start_ms + wall;
        TSVM_LOG << "global iter = " << st.iter - 1 << ", total local iter = " << st.local_iter << ", diff = " << st.diff << ", obj = " << o.obj;
    }
}
