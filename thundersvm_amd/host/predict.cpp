// SvmModel::predict_dec_values (src/thundersvm/model/svmmodel.cpp:74-117): decision values of a set of rows against
// the model's support vectors.  With dense support vectors the kernel values are reduced where they are computed
// (tsvm_predict_dec_values_dense) and never written out; otherwise kernel rows per batch, then
// tsvm_sum_kernel_values, as the reference does.
#include <algorithm>
#include <cmath>
#include <cstdlib>
#include <cstring>
#include <memory>

#include "models.h"

using tsvm::abi_check;
using tsvm::DeviceBuffer;

namespace {
struct OneUpload {   // several arrays that go to the device in one copy, each at a multiple of 256 bytes
    std::vector<tsvm::HostStaging::Part> parts;
    size_t at = 0;
    size_t add(const void *from, size_t bytes) {
        const size_t here = at;
        if (bytes) parts.push_back({from, bytes, at});
        at = (at + bytes + 255) / 256 * 256;
        return here;
    }
    template <typename T>
    size_t add(const std::vector<T> &v) { return add(v.data(), v.size() * sizeof(T)); }
    const char *send(DeviceBuffer<char> &to) const {
        to.resize(std::max<size_t>(at, 256));
        tsvm::HostStaging::instance().upload(to.data(), parts, tsvm::work_stream());
        return to.data();
    }
};
}  // namespace

// A request of a few rows goes by one launch as long as its sums and its rows fit a page-locked block each and what the workgroups
// read over the link, every row once per 128 support vectors, is no more than this.  Calls by one launch / by the kernels for many,
// us: 770 support vectors of 32 columns, one row 19 / 34, 64 rows 24 / 37, 200 rows (0.2 MB) 35 / 61; 2,050, 64 rows 26 / 39;
// 5,740 of 60 columns in six classes, 16 rows (0.2 MB) 29 / 45; 3,550 of 120, one row 25 / 46, 32 rows (0.48 MB) 35 / 53.
constexpr size_t FEW_LINK_BYTES = (size_t) 512 << 10;

struct SvmModel::PredictPlan {
    DeviceBuffer<char> arrays;      // all of the following, uploaded together
    // for both paths
    const float_type *rho = nullptr;
    // unfused path: the reference's arrays as they are
    const int *sv_start = nullptr, *sv_count = nullptr;
    const float_type *coef = nullptr;
    // fused path: every class's support vectors start on a multiple of 128 columns
    int stride = 0;                 // coefficients stored per padded column (0: the fused kernels do not take this model)
    int64_t n_pad = 0;
    std::vector<int> class_tile;    // [n_classes + 1]: first 128-column tile of every class
    const int *col_map = nullptr;   // padded column -> support vector
    const float_type *coef_t = nullptr;   // [n_pad][stride]
    bool many_features = false;     // the 128 x 128 tile kernel (d > 128, no indicator columns)
    // chunk table of the last call, rebuilt when the batch size changes
    mutable size_t chunks_for_m = 0;
    mutable int n_chunks = 0;
    mutable DeviceBuffer<int> chunk_table;   // class_chunk_start, then the chunks
    // the batch rows' indicator masks (grown as needed, kept between calls)
    mutable DeviceBuffer<uint64_t> mask_a;
    mutable DeviceBuffer<int> mask_max;
};

// The padded columns of the support vectors (class_tile: first 128-column tile of every class, n_classes + 1) appended to
// col_map and coef_t.
void SvmModel::pad_classes(int stride, std::vector<int> &class_tile, std::vector<int> &col_map, std::vector<float_type> &coef_t) const {
    const size_t T = sv->size(), first = col_map.size();
    class_tile.assign(n_classes + 1, 0);
    for (int c = 0; c < n_classes; ++c) class_tile[c + 1] = class_tile[c] + (n_sv[c] + 127) / 128;
    const size_t n_pad = (size_t) class_tile[n_classes] * 128;
    col_map.resize(first + n_pad, 0);
    coef_t.resize((first + n_pad) * stride, 0.0);
    int sv_start = 0;
    for (int c = 0; c < n_classes; ++c) {
        const size_t p0 = first + (size_t) class_tile[c] * 128, p1 = first + (size_t) class_tile[c + 1] * 128;
        for (size_t p = p0; p < p1; ++p) {
            const int t = (int) (p - p0);
            if (t < n_sv[c]) {
                const int l = sv_start + t;
                col_map[p] = l;
                for (int r = 0; r < n_classes - 1; ++r) coef_t[p * stride + r] = coef[(size_t) r * T + l];
            } else {
                col_map[p] = sv_start;   // a valid row; its coefficients stay zero
            }
        }
        sv_start += n_sv[c];
    }
}

const SvmModel::PredictPlan &SvmModel::predict_plan() const {
    if (predict_plan_) return *predict_plan_;
    // the support vectors' device copy is built by the first predict call and kept for the next ones (the
    // reference rebuilds it per call, svmmodel.cpp:84)
    if (!sv_k_mat) sv_k_mat.reset(new KernelMatrix(*sv, param));
    auto plan = std::make_shared<PredictPlan>();
    PredictPlan &P = *plan;
    const DeviceRows &R = sv_k_mat->rows();
    std::vector<int> sv_start(n_classes, 0);
    for (int c = 1; c < n_classes; ++c) sv_start[c] = sv_start[c - 1] + n_sv[c - 1];
    std::vector<int> col_map;
    std::vector<float_type> coef_t;
    const bool masks = R.dense && R.ind_first >= 0;
    const int d = masks ? R.ind_first : (int) R.n_features;
    P.stride = R.dense ? tsvm_predict_nc_stride(n_classes, d, masks) : 0;
    if (P.stride > 0) {
        P.many_features = d > 128 && !masks;
        pad_classes(P.stride, P.class_tile, col_map, coef_t);
        P.n_pad = (int64_t) P.class_tile[n_classes] * 128;
    }
    // (eight arrays, most of them some bytes: uploads of 10 us each)
    OneUpload up;
    const auto add = [&](const void *from, size_t bytes) { return up.add(from, bytes); };
    const size_t rho_at = add(rho.data(), rho.size() * sizeof(float_type)), start_at = add(sv_start.data(), sv_start.size() * sizeof(int));
    const size_t count_at = add(n_sv.data(), n_sv.size() * sizeof(int)), coef_at = add(coef.data(), coef.size() * sizeof(float_type));
    const size_t map_at = add(col_map.data(), col_map.size() * sizeof(int)), coef_t_at = add(coef_t.data(), coef_t.size() * sizeof(float_type));
    const char *const base = up.send(P.arrays);
    P.rho = (const float_type *) (base + rho_at);
    P.sv_start = (const int *) (base + start_at);
    P.sv_count = (const int *) (base + count_at);
    P.coef = (const float_type *) (base + coef_at);
    P.col_map = (const int *) (base + map_at);
    P.coef_t = (const float_type *) (base + coef_t_at);
    predict_plan_ = plan;
    return *predict_plan_;
}

// Chunks: runs of column tiles inside one class, short enough that the workgroups walking the same chunk side by
// side keep its support vectors in their XCD's L2, and numerous enough to fill the chip when the batch is small.
static void build_chunks(const std::vector<int> &class_tile, size_t row_blocks, int max_tiles, std::vector<int> &chunks,
                         std::vector<int> &class_chunk_start) {
    const int n_classes = (int) class_tile.size() - 1;
    const int64_t total = class_tile[n_classes];
    const int64_t per = std::max<int64_t>(1, std::min<int64_t>(max_tiles, total * (int64_t) row_blocks / 2048));
    chunks.clear();
    class_chunk_start.assign(n_classes + 1, 0);
    for (int c = 0; c < n_classes; ++c) {
        const int t0 = class_tile[c], nt = class_tile[c + 1] - t0;
        const int pieces = (int) ((nt + per - 1) / per);
        for (int q = 0; q < pieces; ++q) {   // as even as possible
            chunks.push_back(t0 + (int) ((int64_t) nt * q / pieces));
            chunks.push_back(t0 + (int) ((int64_t) nt * (q + 1) / pieces));
        }
        class_chunk_start[c + 1] = class_chunk_start[c] + pieces;
    }
}

bool SvmModel::predict_batch_fused(const PredictPlan &P, const kernel_type *a, int64_t lda, const kernel_type *sd_a, size_t m,
                                   bool indicator_values, float_type *dec_out, int *winner_out) const {
    const DeviceRows &R = sv_k_mat->rows();
    // (TSVM_PREDICT_UNFUSED: the two-call form for every batch, to compare the two)
    if (P.stride == 0 || getenv("TSVM_PREDICT_UNFUSED")) return false;
    const bool plan_masks = R.ind_first >= 0;
    if (plan_masks && !indicator_values) return false;   // (the coefficient layout was made for the kernel with masks)
    const int d = plan_masks ? R.ind_first : (int) R.n_features;
    if (lda < (int64_t) ((R.n_features + 7) / 8 * 8)) return false;
    if (P.chunks_for_m != m) {
        std::vector<int> chunks, ccs;
        build_chunks(P.class_tile, P.many_features ? (m + 127) / 128 : (m + 63) / 64, P.many_features ? 8 : 32, chunks, ccs);
        P.n_chunks = (int) chunks.size() / 2;
        ccs.insert(ccs.end(), chunks.begin(), chunks.end());
        P.chunk_table.upload(ccs);
        P.chunks_for_m = m;
    }
    if (plan_masks) {
        if (P.mask_a.size() < m) P.mask_a.resize(m);
        if (P.mask_max.size() < 1) P.mask_max.resize(1);
        abi_check(tsvm_indicator_masks(a, lda, (int64_t) m, R.ind_first, (int) R.n_features - R.ind_first, P.mask_a.data(),
                                       P.mask_max.data(), tsvm::work_stream()));
    }
    const int km1 = n_classes - 1;
    // partial sums, decision values and winners: from the persistent row arena (no allocation per call)
    const size_t part_doubles = (size_t) std::max(P.n_chunks, 1) * m * km1, dec_doubles = m * (size_t) n_binary_models;
    float_type *d_part = (float_type *) tsvm::RowArena::instance().acquire((part_doubles + dec_doubles) * sizeof(float_type) + m * sizeof(int), false);
    float_type *d_dec = d_part + part_doubles;
    // a request of a few rows has its decision values written straight to page-locked host memory: no copy behind the kernels
    std::unique_ptr<tsvm::ResultBlock> direct;
    if (!winner_out && dec_doubles * sizeof(float_type) <= tsvm::PINNED_BLOCK) {
        direct.reset(new tsvm::ResultBlock(tsvm::work_stream()));
        d_dec = (float_type *) direct->dev();
    }
    // (a batch row may set more indicator columns than any support vector does: its matches are bounded by the
    // support vectors' count all the same)
    abi_check(tsvm_predict_dec_values_dense(R.x.data(), R.ld, d, R.self_dot.data(), plan_masks ? R.ind_mask.data() : nullptr,
                                            P.col_map, P.n_pad, P.coef_t, P.chunk_table.data() + n_classes + 1, P.n_chunks,
                                            P.chunk_table.data(), P.rho, n_classes, a, lda, (int64_t) m, sd_a,
                                            plan_masks ? P.mask_a.data() : nullptr, R.ind_max_ones, (int) param.kernel_type,
                                            param.gamma, param.coef0, param.degree, d_part, d_dec, tsvm::work_stream()));
    if (direct) {
        memcpy(dec_out, direct->wait(), dec_doubles * sizeof(float_type));
    } else {
        fetch_predictions(d_dec, m, dec_out, winner_out);
    }
    return true;
}

bool SvmModel::predict_few(const PredictPlan &P, const RowStore &rows, size_t first, size_t m, float_type *dec_out) const {
    const DeviceRows &R = sv_k_mat->rows();
    const int d = (int) R.n_features, nc = n_classes - 1;
    const size_t tiles = (size_t) P.n_pad / 128, sums = tiles * m * nc, in_bytes = m <= 4096 ? tsvm_predict_few_rows_bytes((int) m, d) : 0;
    if (P.stride == 0 || P.many_features || tiles == 0 || in_bytes == 0 || in_bytes > tsvm::PINNED_BLOCK || sums * sizeof(float_type) > tsvm::PINNED_BLOCK)
        return false;
    if (tiles * in_bytes > FEW_LINK_BYTES) return false;
    tsvm::ResultBlock in(tsvm::work_stream()), out(tsvm::work_stream());
    float *const dense = (float *) in.host();
    double *const sd = (double *) (dense + (m * d + 1) / 2 * 2);
    std::fill(dense, dense + (m * d + 1) / 2 * 2, 0.0f);
    const int64_t *const ptr = rows.ptr() + first;
    for (size_t r = 0; r < m; ++r) {
        double s = 0.0;
        for (int64_t e = ptr[r]; e < ptr[r + 1]; ++e) {
            const double v = rows.val()[e];
            const int c = rows.col()[e];
            // (other values than finite floats: the square below would not be exact, or a product with an absent column not zero)
            if (!((double) (float) v == v) || std::isinf(v) || c < 0) {
                in.unused();
                out.unused();
                return false;
            }
            if (c < d) dense[r * d + c] = (float) v;
            s += v * v;   // (the square of a float is exact: what fma(v, v, s) gives)
        }
        sd[r] = s;
    }
    out.expect(sums);
    abi_check(tsvm_predict_few_rows(R.x.data(), R.ld, d, R.self_dot.data(), P.col_map, P.n_pad, P.coef_t, P.stride, nc, dense, (const float *) in.dev(),
                                    (int) m, (int) param.kernel_type, param.gamma, param.coef0, param.degree, (float_type *) out.dev(),
                                    tsvm::work_stream()));
    const float_type *const part = out.wait_for(sums);
    in.unused();   // (whoever wrote the sums has read the rows)
    // every pair's two classes, tile after tile, as predict_combine_kernel adds them
    for (size_t r = 0; r < m; ++r) {
        float_type *to = dec_out + r * n_binary_models;
        for (int i = 0, p = 0; i < n_classes; ++i)
            for (int j = i + 1; j < n_classes; ++j, ++p) {
                double s = 0.0, t = 0.0;
                for (int tile = P.class_tile[i]; tile < P.class_tile[i + 1]; ++tile) s += part[((size_t) tile * m + r) * nc + (j - 1)];
                for (int tile = P.class_tile[j]; tile < P.class_tile[j + 1]; ++tile) t += part[((size_t) tile * m + r) * nc + i];
                to[p] = (s + t) - rho[p];
            }
    }
    return true;
}

void SvmModel::fetch_predictions(float_type *d_dec, size_t m, float_type *dec_out, int *winner_out) const {
    const size_t dec_bytes = m * (size_t) n_binary_models * sizeof(float_type);
    int *const d_winner = (int *) ((char *) d_dec + dec_bytes);
    if (winner_out) abi_check(tsvm_predict_votes(d_dec, (int64_t) m, n_classes, d_winner, tsvm::work_stream()));
    tsvm::HostStaging::instance().download(d_dec, dec_bytes + (winner_out ? m * sizeof(int) : 0), [=](const char *from, size_t off, size_t len) {
        if (off < dec_bytes) tsvm::parallel_memcpy((char *) dec_out + off, from, std::min(len, dec_bytes - off));
        if (off + len > dec_bytes) {
            const size_t lo = std::max(off, dec_bytes);
            memcpy((char *) winner_out + (lo - dec_bytes), from + (lo - off), off + len - lo);
        }
    }, tsvm::work_stream());
}

void SvmModel::predict_dec_values(const RowStore &rows, std::vector<float_type> &dec, int batch_size, std::vector<int> *winner) const {
    const size_t n_rows = rows.size();
    dec.resize(n_rows * (size_t) n_binary_models);   // (every element is written below)
    if (winner) winner->clear();
    if (n_rows == 0) return;
    const size_t T = sv->size();
    if (T == 0) {
        for (size_t r = 0; r < n_rows; ++r)
            for (int p = 0; p < n_binary_models; ++p) dec[r * n_binary_models + p] = -rho[p];
        return;
    }
    const PredictPlan &P = predict_plan();
    const KernelMatrix &k_mat = *sv_k_mat;
    const bool fused = P.stride > 0 && !getenv("TSVM_PREDICT_UNFUSED");
    if (batch_size == -1) {
        if (fused) {
            // no batch x support-vector matrix exists: a batch only needs its own rows on the device
            batch_size = 65536;
        } else {
            const size_t used = tsvm::device_bytes_in_use();
            const size_t free_mem = param.max_mem_size > used ? param.max_mem_size - used : 0;
            batch_size = (int) std::min(free_mem / sizeof(float_type) / (T + k_mat.n_features()), size_t(10000));
        }
        if (batch_size < 1) batch_size = 1;
    }
    const size_t bmax = std::min((size_t) batch_size, n_rows);
    void *d_k = nullptr;
    const int64_t ldk = ((int64_t) T + 15) / 16 * 16;   // (rows padded to 16 elements: get_rows writes whole aligned vectors)
    DeviceBuffer<float_type> d_dec;
    if (winner) winner->resize(n_rows);
    for (size_t b0 = 0; b0 < n_rows; b0 += batch_size) {
        const size_t bm = std::min((size_t) batch_size, n_rows - b0);
        if (fused) {
            if (!winner && predict_few(P, rows, b0, bm, dec.data() + b0 * n_binary_models)) continue;
            const KernelMatrix::StagedBatch b = k_mat.stage_batch(rows, b0, bm);
            if (predict_batch_fused(P, b.a, b.lda, b.sd, bm, b.indicator_values, dec.data() + b0 * n_binary_models,
                                    winner ? winner->data() + b0 : nullptr))
                continue;
        }
        // kernel values of one batch (taken from the persistent row arena), then the reduction
        if (!d_k) {
            d_k = tsvm::RowArena::instance().acquire(bmax * (size_t) ldk * k_mat.row_elem_size(), false);
            d_dec.resize(bmax * n_binary_models + (winner ? (bmax + 1) / 2 : 0));
        }
        k_mat.get_rows(rows, b0, bm, d_k, ldk);
        abi_check(tsvm_sum_kernel_values(P.coef, (int) T, P.sv_start, P.sv_count, P.rho, d_k,
                                         k_mat.row_type(), ldk, d_dec.data(), n_classes, (int64_t) bm, tsvm::work_stream()));
        fetch_predictions(d_dec.data(), bm, dec.data() + b0 * n_binary_models, winner ? winner->data() + b0 : nullptr);
    }
}

void SvmModel::predict_dec_values(const DataSet &dataset, std::vector<float_type> &dec, int batch_size, std::vector<int> *winner) const {
    const std::shared_ptr<void> &slot = dataset.device_cache();
    if (slot && sv->size() > 0 && dataset.n_instances() > 0) {
        const DeviceRows &A = *std::static_pointer_cast<DeviceRows>(slot);
        const PredictPlan &P = predict_plan();
        const DeviceRows &R = sv_k_mat->rows();
        if (A.dense && P.stride > 0 && A.n == dataset.n_instances()) {
            // do the batch's values in the support vectors' indicator columns qualify?  (counted once per DataSet)
            bool indicator_values = false;
            if (R.ind_first >= 0) {
                const std::vector<int> &st = A.column_stats();
                indicator_values = true;
                for (size_t c = (size_t) R.ind_first; c < std::min(R.n_features, A.n_features); ++c)
                    if (st[A.n_features + c] != 0) indicator_values = false;
            }
            dec.resize(dataset.n_instances() * (size_t) n_binary_models);   // (every element is written below, or by the call at the end)
            if (winner) winner->resize(dataset.n_instances());
            const size_t step = batch_size > 0 ? (size_t) batch_size : A.n;
            bool ok = true;
            for (size_t b0 = 0; b0 < A.n && ok; b0 += step) {
                const size_t bm = std::min(step, A.n - b0);
                ok = predict_batch_fused(P, A.x.data() + b0 * (size_t) A.ld, A.ld, A.self_dot.data() + b0, bm, indicator_values,
                                         dec.data() + b0 * n_binary_models, winner ? winner->data() + b0 : nullptr);
            }
            if (ok) return;
        }
    }
    predict_dec_values(dataset.rows(), dec, batch_size, winner);
}

bool SvmModel::predict_folds(const DeviceRows &all, const std::vector<FoldRows> &folds, std::vector<std::vector<float_type>> &dec) {
    const SvmModel &first = *folds[0].model;
    const int k = first.n_classes, P = first.n_binary_models, d = (int) all.n_features;
    const int stride = all.dense && d <= 128 && !getenv("TSVM_PREDICT_UNFUSED") ? tsvm_predict_nc_stride(k, d, 0) : 0;
    if (stride == 0 || P != k * (k - 1) / 2 || first.param.kernel_type == SvmParam::PRECOMPUTED) return false;
    for (const FoldRows &f : folds)
        if (f.model->n_classes != k || f.model->n_binary_models != P || f.model->sv->size() == 0) return false;
    // A group is a fold's batch of rows, as its own call would take them; the chunks of columns are cut for it as there.
    std::vector<int> col_map, rows, row_group, chunks, chunk_start;
    std::vector<float_type> coef_t, rho;
    std::vector<tsvm_predict_task> tasks;
    int most_parts = 0, group = 0;
    for (const FoldRows &f : folds) {
        const SvmModel &m = *f.model;
        const size_t col0 = col_map.size();
        std::vector<int> class_tile;
        m.pad_classes(stride, class_tile, col_map, coef_t);
        for (size_t p = col0; p < col_map.size(); ++p) col_map[p] = (*f.train_idx)[m.sv_indices[col_map[p]]];
        for (size_t b0 = 0; b0 < f.test_idx->size(); b0 += FOLD_BATCH, ++group) {
            const int row0 = (int) rows.size(), bm = (int) std::min<size_t>(FOLD_BATCH, f.test_idx->size() - b0), chunk0 = (int) chunks.size() / 2;
            rows.insert(rows.end(), f.test_idx->begin() + b0, f.test_idx->begin() + b0 + bm);
            row_group.insert(row_group.end(), bm, group);
            std::vector<int> mine, starts;
            build_chunks(class_tile, (bm + 63) / 64, 32, mine, starts);
            const int parts = (int) mine.size() / 2;
            for (int part = 0; part < parts; ++part)
                for (int r = 0; r < bm; r += 64) tasks.push_back({row0 + r, row0 + bm, chunk0 + part, part});
            for (int tile : mine) chunks.push_back((int) (col0 / 128) + tile);
            chunk_start.insert(chunk_start.end(), starts.begin(), starts.end());
            rho.insert(rho.end(), m.rho.begin(), m.rho.begin() + P);
            most_parts = std::max(most_parts, parts);
        }
    }
    const size_t m_all = rows.size(), part_doubles = (size_t) std::max(most_parts, 1) * m_all * (k - 1), dec_bytes = m_all * P * sizeof(float_type);
    dec.resize(folds.size());
    for (size_t i = 0; i < folds.size(); ++i) dec[i].resize(folds[i].test_idx->size() * P);
    if (m_all == 0) return true;
    OneUpload up;
    const size_t tasks_at = up.add(tasks), rows_at = up.add(rows), group_at = up.add(row_group), map_at = up.add(col_map), coef_at = up.add(coef_t);
    const size_t chunks_at = up.add(chunks), start_at = up.add(chunk_start), rho_at = up.add(rho);
    DeviceBuffer<char> arrays;
    const char *const at = up.send(arrays);
    float_type *const d_part = (float_type *) tsvm::RowArena::instance().acquire(part_doubles * sizeof(float_type) + dec_bytes, false);
    float_type *d_dec = d_part + part_doubles;
    std::unique_ptr<tsvm::ResultBlock> direct;
    if (dec_bytes <= tsvm::PINNED_BLOCK) {   // (straight to page-locked host memory, as a request of a few rows)
        direct.reset(new tsvm::ResultBlock(tsvm::work_stream()));
        d_dec = (float_type *) direct->dev();
    }
    const SvmParam &p = first.param;
    abi_check(tsvm_predict_groups_dense(all.x.data(), all.ld, d, all.self_dot.data(), (const int *) (at + map_at), (int64_t) col_map.size(),
                                        (const float_type *) (at + coef_at), (const int *) (at + chunks_at), (const tsvm_predict_task *) (at + tasks_at),
                                        (int) tasks.size(), (const int *) (at + rows_at), (int64_t) m_all, (const int *) (at + group_at),
                                        (const int *) (at + start_at), (const float_type *) (at + rho_at), k, (int) p.kernel_type, p.gamma, p.coef0,
                                        p.degree, d_part, d_dec, tsvm::work_stream()));
    std::vector<float_type> all_dec(m_all * P);
    if (direct)
        memcpy(all_dec.data(), direct->wait(), dec_bytes);
    else
        tsvm::HostStaging::instance().download(d_dec, dec_bytes, [&](const char *from, size_t off, size_t len) {
            tsvm::parallel_memcpy((char *) all_dec.data() + off, from, len);
        }, tsvm::work_stream());
    size_t from = 0;
    for (std::vector<float_type> &v : dec) {
        std::copy(all_dec.begin() + from, all_dec.begin() + from + v.size(), v.begin());
        from += v.size();
    }
    return true;
}

namespace {
struct ClearAtEnd {   // (a prediction's winners are no other call's)
    std::vector<int> &v;
    ~ClearAtEnd() { v.clear(); }
};
}  // namespace

std::vector<float_type> SvmModel::predict(const DataSet::node2d &instances, int batch_size) {   // svmmodel.cpp:157-171
    const ClearAtEnd clear{vote_winner};
    predict_dec_values(*RowStore::from_nodes(instances), dec_values, batch_size, votes_on_device(instances.size()) ? &vote_winner : nullptr);
    return finish_predict((int) instances.size());
}

std::vector<float_type> SvmModel::predict(const DataSet &dataset, int batch_size) {
    const ClearAtEnd clear{vote_winner};
    predict_dec_values(dataset, dec_values, batch_size, votes_on_device(dataset.n_instances()) ? &vote_winner : nullptr);
    return finish_predict((int) dataset.n_instances());
}
