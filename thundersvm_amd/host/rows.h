// The rows of a data set (or a model's support vectors) in host memory, as three flat arrays: row i's entries are
// col / val [ptr[i], ptr[i + 1]).  The reference keeps a vector of vectors of (index, value) nodes
// (include/thundersvm/dataset.h:17-27): one allocation per row, which made taking rows in, handing them to the device
// and copying support vectors cost more than a small training run.  That form is still available, built when it is first
// asked for.
#pragma once
#include <cstdint>
#include <memory>
#include <mutex>
#include <vector>

#include "thundersvm.h"

struct RowNode {
    RowNode(int index, kernel_type value) : index(index), value(value) {}
    int index;
    kernel_type value;
};

class RowStore {
public:
    typedef std::vector<std::vector<RowNode>> node2d;

    // room for n rows with nnz entries; ptr()[0 .. n] and the entries are the caller's to fill through the mutable pointers
    RowStore(size_t n, size_t nnz);
    // the caller's arrays, not copied: they have to outlive the store
    RowStore(size_t n, const int64_t *ptr, const int *col, const kernel_type *val);
    static std::shared_ptr<RowStore> copy_of(size_t n, const int64_t *ptr, const int *col, const kernel_type *val);
    static std::shared_ptr<RowStore> from_nodes(const node2d &nodes);
    // rows ids[0 .. n_ids), copied
    std::shared_ptr<RowStore> gather(const int *ids, size_t n_ids) const;

    size_t size() const { return n_; }
    size_t nnz() const { return (size_t) (ptr_[n_] - ptr_[0]); }
    const int64_t *ptr() const { return ptr_; }
    const int *col() const { return col_; }
    const kernel_type *val() const { return val_; }
    size_t row_size(size_t i) const { return (size_t) (ptr_[i + 1] - ptr_[i]); }
    int64_t *ptr_mut() { return own_ptr_.get(); }
    int *col_mut() { return own_col_.get(); }
    kernel_type *val_mut() { return own_val_.get(); }
    const node2d &nodes() const;

private:
    size_t n_ = 0;
    const int64_t *ptr_ = nullptr;
    const int *col_ = nullptr;
    const kernel_type *val_ = nullptr;
    std::unique_ptr<int64_t[]> own_ptr_;
    std::unique_ptr<int[]> own_col_;
    std::unique_ptr<kernel_type[]> own_val_;
    mutable std::once_flag nodes_once_;
    mutable node2d nodes_;
};

// The most threads of a training or prediction call's parallel regions: as many as the caller has asked for (set_threads, or
// omp_set_num_threads in a program of its own), else three quarters of what there is.  The team goes on spinning
// for some 75 ms behind a region, so calls that follow one another faster keep all of it busy, the thread that waits for the
// device and the runtime's own among it; with a thread for every CPU that a container has been given its scheduler then
// stops the process for tens of milliseconds (epsilon-SVR 40000x90 with 16 threads on 16 CPUs: one call in
// three takes 78 to 190 ms in place of 75).
int thread_limit();
void set_threads(int n);   // -o, n_jobs, for the calling thread's regions; 0: nobody has asked
// Threads that pay for a loop over `entries` row entries: a parallel region costs some ten microseconds to enter.
int threads_for(size_t entries);
