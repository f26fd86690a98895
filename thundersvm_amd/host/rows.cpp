#include "rows.h"

#include <omp.h>

#include <algorithm>
#include <cstring>

namespace {
const int g_threads_at_start = omp_get_max_threads();
thread_local int t_threads_asked = 0;   // (omp_set_num_threads is the calling thread's, too)
}  // namespace

void set_threads(int n) {
    t_threads_asked = n;
    omp_set_num_threads(n > 0 ? n : g_threads_at_start);
}
int thread_limit() {
    const int n = omp_get_max_threads();
    return n == t_threads_asked || n != g_threads_at_start ? n : (3 * n + 3) / 4;
}
int threads_for(size_t entries) { return (int) std::max<size_t>(1, std::min<size_t>((size_t) thread_limit(), entries / 32768)); }

// (none of the arrays is value-initialised: whoever fills them does so on many threads, which also take the page faults)
RowStore::RowStore(size_t n, size_t nnz)
    : n_(n), own_ptr_(new int64_t[n + 1]), own_col_(new int[nnz]), own_val_(new kernel_type[nnz]) {
    ptr_ = own_ptr_.get();
    col_ = own_col_.get();
    val_ = own_val_.get();
    own_ptr_[0] = 0;
    own_ptr_[n] = (int64_t) nnz;
}

RowStore::RowStore(size_t n, const int64_t *ptr, const int *col, const kernel_type *val) : n_(n), ptr_(ptr), col_(col), val_(val) {}

std::shared_ptr<RowStore> RowStore::copy_of(size_t n, const int64_t *ptr, const int *col, const kernel_type *val) {
    const int64_t first = ptr[0];
    const size_t nnz = (size_t) (ptr[n] - first);
    auto s = std::make_shared<RowStore>(n, nnz);
    for (size_t i = 0; i <= n; ++i) s->own_ptr_[i] = ptr[i] - first;
    const long pieces = (long) ((nnz + 32767) / 32768);
#pragma omp parallel for schedule(static) num_threads(threads_for(nnz))
    for (long p = 0; p < pieces; ++p) {
        const size_t lo = (size_t) p * 32768, len = std::min<size_t>(32768, nnz - lo);
        memcpy(s->own_col_.get() + lo, col + first + lo, len * sizeof(int));
        memcpy(s->own_val_.get() + lo, val + first + lo, len * sizeof(kernel_type));
    }
    return s;
}

std::shared_ptr<RowStore> RowStore::from_nodes(const node2d &nodes) {
    size_t nnz = 0;
    for (const auto &r : nodes) nnz += r.size();
    auto s = std::make_shared<RowStore>(nodes.size(), nnz);
    for (size_t i = 0; i < nodes.size(); ++i) s->own_ptr_[i + 1] = s->own_ptr_[i] + (int64_t) nodes[i].size();
#pragma omp parallel for schedule(static) num_threads(threads_for(nnz))
    for (size_t i = 0; i < nodes.size(); ++i) {
        int64_t e = s->own_ptr_[i];
        for (const RowNode &nd : nodes[i]) {
            s->own_col_[e] = nd.index;
            s->own_val_[e++] = nd.value;
        }
    }
    return s;
}

std::shared_ptr<RowStore> RowStore::gather(const int *ids, size_t n_ids) const {
    size_t nnz = 0;
    for (size_t i = 0; i < n_ids; ++i) nnz += row_size((size_t) ids[i]);
    auto s = std::make_shared<RowStore>(n_ids, nnz);
    for (size_t i = 0; i < n_ids; ++i) s->own_ptr_[i + 1] = s->own_ptr_[i] + (int64_t) row_size((size_t) ids[i]);
#pragma omp parallel for schedule(static) num_threads(threads_for(nnz))
    for (size_t i = 0; i < n_ids; ++i) {
        const size_t len = row_size((size_t) ids[i]);
        memcpy(s->own_col_.get() + s->own_ptr_[i], col_ + ptr_[ids[i]], len * sizeof(int));
        memcpy(s->own_val_.get() + s->own_ptr_[i], val_ + ptr_[ids[i]], len * sizeof(kernel_type));
    }
    return s;
}

const RowStore::node2d &RowStore::nodes() const {
    std::call_once(nodes_once_, [this] {
        nodes_.resize(n_);
#pragma omp parallel for schedule(static) num_threads(threads_for(nnz()))
        for (size_t i = 0; i < n_; ++i) {
            std::vector<RowNode> &r = nodes_[i];
            r.reserve(row_size(i));
            for (int64_t e = ptr_[i]; e < ptr_[i + 1]; ++e) r.emplace_back(col_[e], val_[e]);
        }
    });
    return nodes_;
}
