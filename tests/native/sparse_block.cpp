// The staging matrices of a sparse solve's blocks (KernelMatrix::get_block) where the device has room for two, where it has not, and
// where they are large: a program of its own whose definitions of the HIP calls and of the kernels stand in for the real ones, hand
// out host memory up to a limit and compute on it.  Exits with 0, or prints what went wrong.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <vector>

#include "../../thundersvm_amd/host/kernelmatrix.h"

static int g_failures = 0, g_refused = 0, g_puts = 0;
static size_t g_in_use = 0, g_memory = ~(size_t) 0;
static hipError_t g_last = hipSuccess;
static std::map<void *, size_t> g_size;

static void expect(bool ok, const char *what) {
    if (ok) return;
    ++g_failures;
    fprintf(stderr, "sparse block: %s\n", what);
}
template <typename T>
static hipError_t make(T *out, size_t bytes) {
    if (bytes > g_memory - g_in_use) {
        ++g_refused;
        return g_last = hipErrorOutOfMemory;
    }
    *out = (T) calloc(1, bytes);
    g_size[*out] = bytes;
    g_in_use += bytes;
    return hipSuccess;
}
static hipError_t drop(void *p) {
    g_in_use -= g_size[p];
    g_size.erase(p);
    free(p);
    return hipSuccess;
}
static size_t blocks_of(size_t bytes) {   // live allocations of at least that size
    size_t n = 0;
    for (auto &kv : g_size) n += kv.second >= bytes;
    return n;
}

// rows idx[0..m) into w [features][m], or out of it
template <typename T>
static void move_rows(const double *val, const int *col, const int64_t *ptr, const int *idx, int m, T *w, bool out) {
    for (int i = 0; i < m; ++i)
        for (int64_t e = ptr[idx[i]]; e < ptr[idx[i] + 1]; ++e) {
            T &at = w[(int64_t) col[e] * m + i];
            expect(out ? at == (T) val[e] : at == 0, out ? "a row that is taken out was not in" : "the staging matrix was not empty");
            at = out ? (T) 0 : (T) val[e];
        }
}

extern "C" {
hipError_t hipGetDevice(int *d) { *d = 0; return hipSuccess; }
hipError_t hipGetLastError(void) { const hipError_t e = g_last; g_last = hipSuccess; return e; }
hipError_t hipMalloc(void **p, size_t bytes) { return make(p, bytes); }
hipError_t hipFree(void *p) { return drop(p); }
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) { *p = malloc(bytes); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize(void) { return hipSuccess; }
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t) malloc(1); return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t s) { free(s); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t) malloc(1); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { free(e); return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventQuery(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipMemcpyAsync(void *to, const void *from, size_t bytes, hipMemcpyKind, hipStream_t) { memcpy(to, from, bytes); return hipSuccess; }
hipError_t hipMemsetAsync(void *p, int v, size_t bytes, hipStream_t) { memset(p, v, bytes); return hipSuccess; }

int tsvm_csr_self_dot(const double *, const int64_t *, int64_t, double *, tsvm_stream) { return 0; }
int tsvm_kernel_diag(const double *, int64_t, int, double, double, int, double *, tsvm_stream) { return 0; }
size_t tsvm_get_rows_csr_sliced_lds(int, int, int) { return 0; }
int tsvm_csr_scatter_rows(const double *val, const int *col, const int64_t *ptr, const int *idx, int m, int, void *w, int w_type, int clear, tsvm_stream) {
    expect(w_type == TSVM_ROW_F32 && g_last == hipSuccess, "a launch behind an error that nobody has taken");
    move_rows(val, col, ptr, idx, m, (float *) w, clear != 0);
    return 0;
}
int tsvm_csr_block(const double *val, const int *col, const int64_t *ptr, const int *idx, int m, const double *, void *w, int *ids, void *w_old, const int *ids_old,
                   int m_old, int w_type, int, double, double, int, void *out, int, int64_t ldo, tsvm_stream) {
    expect(w_type == TSVM_ROW_F32 && g_last == hipSuccess, "a launch behind an error that nobody has taken");
    move_rows(val, col, ptr, idx, m, (float *) w, false);
    memcpy(ids, idx, m * sizeof(int));
    if (m_old) move_rows(val, col, ptr, ids_old, m_old, (float *) w_old, true);
    ++g_puts;
    for (int r = 0; r < m; ++r)
        for (int t = 0; t < m; ++t) {
            double s = 0.0;
            for (int64_t e = ptr[idx[r]]; e < ptr[idx[r] + 1]; ++e) s += val[e] * ((const float *) w)[(int64_t) col[e] * m + t];
            ((double *) out)[r * ldo + t] = s;
        }
    return 0;
}
}

// Blocks of a linear kernel, of 2 to m rows; the device has room for `beside` bytes beside the first staging matrix.  matrices: how many
// there are to be in the end.
static void solve(int n_features, int m, size_t beside, size_t matrices, int refused, const char *what) {
    const int n = 300, per_row = 4;
    std::vector<int64_t> ptr(1, 0);
    std::vector<int> col;
    std::vector<double> val;
    for (int i = 0; i < n; ++i) {
        for (int k = 0; k < per_row; ++k) {
            col.push_back((int) ((int64_t) n_features * k / per_row) + i * (k + 1) % (n_features / per_row));
            val.push_back(1 + i % 7 + k);
        }
        ptr.push_back((int64_t) col.size());
    }
    col[per_row * n - 1] = n_features - 1;
    const int before = g_failures;
    {
        SvmParam param;
        param.kernel_type = SvmParam::LINEAR;
        const RowStore rows(n, ptr.data(), col.data(), val.data());
        const KernelMatrix k(rows, param);
        expect(!k.dense_layout() && (int) k.n_features() == n_features, "the layout");
        const size_t bytes = (size_t) m * n_features * sizeof(float);
        std::vector<double> out((size_t) m * m);
        std::vector<int> idx(m);
        g_refused = 0;
        for (int call = 0; call < 7; ++call) {
            const int now = call == 3 ? 2 : m;   // (a smaller working set between)
            for (int t = 0; t < now; ++t) idx[t] = (t * 37 + call * 11) % n;
            k.get_block(idx.data(), now, out.data(), now);
            for (int r = 0; r < now; ++r)
                for (int t = 0; t < now; ++t) {
                    double s = 0.0;
                    for (int a = 0; a < per_row; ++a)
                        for (int b = 0; b < per_row; ++b)
                            if (col[idx[r] * per_row + a] == col[idx[t] * per_row + b]) s += val[idx[r] * per_row + a] * val[idx[t] * per_row + b];
                    if (out[r * now + t] != s) return expect(false, what);
                }
            if (call == 0) g_memory = beside == ~(size_t) 0 ? beside : g_in_use + beside;
        }
        expect(blocks_of(bytes) == matrices, what);
        expect(g_refused <= refused, "memory is asked for again and again");
        g_memory = ~(size_t) 0;
    }
    tsvm::DevicePool::instance().flush();
    if (g_failures > before) fprintf(stderr, "sparse block: %s: %zu matrices, %d refusals\n", what, matrices, g_refused);
}

int main() {
    solve(4000, 64, ~(size_t) 0, 2, 0, "two matrices in turn");
    solve(4000, 64, 100000, 1, 2, "no room for a second matrix");
    solve(300000, 128, ~(size_t) 0, 1, 0, "a large matrix, alone");
    solve(300000, 128, 0, 1, 0, "a large matrix and no room beside it");
    expect(g_puts == 28, "blocks");
    if (g_failures == 0) puts("ok");
    return g_failures != 0;
}
