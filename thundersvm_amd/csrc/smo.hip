// SMO device kernels for gfx950: update_f, the single-workgroup local solvers and the fused
// sort_f + select_working_set.
//
// Reference behaviour restated here: src/thundersvm/kernel/smo_kernel.cpp:12-332,
// src/thundersvm/solver/csmosolver.cpp:123-165, src/thundersvm/solver/nusmosolver.cpp:48-118
// (the USE_CUDA=OFF, USE_DOUBLE=ON build: first-index tie breaks, serial summation order).
#include "../../include/thundersvm_amd.h"
#include "tsvm_device.h"
#include "tsvm_internal.h"

#define TSVM_INF __builtin_inf()
#define MAX_WS 1024

// ------------------------------------------------------------------------------------------------
// Fused sort_f + select_working_set.
//
// The reference sorts (f, index) pairs ascending (smo_kernel.cpp:321-332) and then walks the
// sorted order from both ends, alternately taking the next unmarked I_up element from the low end
// and the next unmarked I_low element from the high end (csmosolver.cpp:123-165).  Only the first
// n_select candidates from each end can ever be taken, so instead of sorting n pairs this selects,
// per side, the n_select smallest composite keys (f-bits, index) among that side's candidates with
// an MSB-first radix select (11-bit digits, one pass over the keys per digit, early exit once the
// boundary bucket is exactly consumed), sorts those <= 1024 entries in LDS with a bitonic network
// and replays the alternating scan on them.  The high end is handled by complementing key and
// index, so every side is an ascending selection.  Composite keys are unique, which makes the
// result independent of any thread ordering.
//
// Sides: C-SMO 0 = I_up (ascending), 1 = I_low (descending);
//        nu-SMO 0 = I_up&y>0, 1 = I_up&y<0 (ascending), 2 = I_low&y>0, 3 = I_low&y<0 (descending).
// ------------------------------------------------------------------------------------------------
#define SEL_BINS 2048
#define SEL_DIGIT 11
#define SEL_MAX_PASS 9
#define SEL_FULL_MAX 4   // digits that are counted by the whole chip, at most
#define SEL_MAX_SIDES 4
#define SEL_T 256
#define SEL_EACH 4   // instances of a thread whose loads are on their way together
#define SEL_GUIDE_BINS 512

struct SelState {
    uint64_t pk;      // resolved high bits of the key part
    uint32_t pi;      // resolved high bits of the index part
    uint32_t k_rem;   // entries still to take from inside the boundary bucket
    uint32_t done;    // 1: selection decided; entries matching the prefix are all taken
    uint32_t pad;     // number of digits held by the prefix
};

struct SelWorkspace {   // device-side layout, carved from the caller's workspace
    uint64_t *keys;     // [n] order-preserving transform of f
    uint8_t *flags;     // [n] side membership bits
    uint32_t *hist;     // [SEL_MAX_PASS][SEL_MAX_SIDES][SEL_BINS]
    SelState *state;    // [SEL_MAX_PASS + 1][SEL_MAX_SIDES]
    uint32_t *count;    // [SEL_MAX_SIDES], then the workgroups of sel_final_kernel that are done
    uint64_t *list_key; // [SEL_MAX_SIDES][MAX_WS]
    uint32_t *list_idx; // [SEL_MAX_SIDES][MAX_WS]
    int2 *sorted;       // [SEL_MAX_SIDES][MAX_WS] the lists in order: instance, its place in the paired side's list or -1
    uint32_t *guide_hist; // [SEL_MAX_SIDES][SEL_GUIDE_BINS]
    uint64_t *guide;    // [SEL_MAX_SIDES][2] the keys of a side's k/2-th and k-th entry, as the last selection left them
};

static size_t sel_align(size_t v) { return (v + 255) & ~(size_t) 255; }

static size_t sel_carve(void *base, int64_t n, SelWorkspace *w) {
    size_t off = 0;
    char *b = (char *) base;
    auto take = [&](size_t bytes) { size_t o = off; off += sel_align(bytes); return b ? b + o : nullptr; };
    void *keys = take(sizeof(uint64_t) * (size_t) n);
    void *flags = take((size_t) n);
    void *hist = take(sizeof(uint32_t) * SEL_MAX_PASS * SEL_MAX_SIDES * SEL_BINS);
    void *state = take(sizeof(SelState) * (SEL_MAX_PASS + 1) * SEL_MAX_SIDES);
    void *count = take(sizeof(uint32_t) * (SEL_MAX_SIDES + 1));
    void *lk = take(sizeof(uint64_t) * SEL_MAX_SIDES * MAX_WS);
    void *li = take(sizeof(uint32_t) * SEL_MAX_SIDES * MAX_WS);
    void *so = take(sizeof(int2) * SEL_MAX_SIDES * MAX_WS);
    void *gh = take(sizeof(uint32_t) * SEL_MAX_SIDES * SEL_GUIDE_BINS);
    void *gu = take(sizeof(uint64_t) * SEL_MAX_SIDES * 2);
    if (w) {
        w->keys = (uint64_t *) keys; w->flags = (uint8_t *) flags;
        w->hist = (uint32_t *) hist; w->state = (SelState *) state; w->count = (uint32_t *) count;
        w->list_key = (uint64_t *) lk; w->list_idx = (uint32_t *) li; w->sorted = (int2 *) so;
        w->guide_hist = (uint32_t *) gh; w->guide = (uint64_t *) gu;
    }
    return off;
}

struct SelGeom {
    int n_sides;
    int n_pass;
    int idx_bits;
    uint32_t idx_mask;
    uint32_t k;   // n_select
};

// digit p of the composite (key: 6 digits of 11,11,11,11,11,9 bits; then the index digits)
__device__ __forceinline__ void sel_digit_geom(int p, int idx_bits, bool &is_key, int &shift, int &width) {
    if (p < 6) {
        is_key = true;
        width = p < 5 ? SEL_DIGIT : 9;
        shift = p < 5 ? 64 - SEL_DIGIT * (p + 1) : 0;
    } else {
        is_key = false;
        const int rb = idx_bits - SEL_DIGIT * (p - 6);
        width = rb < SEL_DIGIT ? rb : SEL_DIGIT;
        shift = rb - width;
    }
}
__device__ __forceinline__ int sel_resolved_key_bits(int p) { return p >= 6 ? 64 : SEL_DIGIT * p; }
__device__ __forceinline__ int sel_resolved_idx_bits(int p, int idx_bits) {
    if (p <= 6) return 0;
    const int r = SEL_DIGIT * (p - 6);
    return r < idx_bits ? r : idx_bits;
}

// -1 / 0 / +1: composite (k, i) versus the prefix on the bits resolved before pass p
__device__ __forceinline__ int sel_cmp_prefix(uint64_t k, uint32_t i, const SelState &st, int p, int idx_bits) {
    const int rk = sel_resolved_key_bits(p);
    if (rk > 0) {
        const uint64_t a = rk == 64 ? k : (k >> (64 - rk));
        const uint64_t b = rk == 64 ? st.pk : (st.pk >> (64 - rk));
        if (a < b) return -1;
        if (a > b) return 1;
    }
    const int ri = sel_resolved_idx_bits(p, idx_bits);
    if (ri > 0) {
        const uint32_t a = i >> (idx_bits - ri);
        const uint32_t b = st.pi >> (idx_bits - ri);
        if (a < b) return -1;
        if (a > b) return 1;
    }
    return 0;
}

__device__ __forceinline__ uint64_t f_to_key(double f) {
    if (f == 0.0) f = 0.0;  // -0.0 and +0.0 compare equal in the reference's sort
    uint64_t u = (uint64_t) __double_as_longlong(f);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

__device__ __forceinline__ double key_to_f(uint64_t key) { return __longlong_as_double((long long) ((key >> 63) ? key & 0x7fffffffffffffffull : ~key)); }

__device__ __forceinline__ bool sel_side_descending(int side, int n_sides) { return n_sides == 2 ? side == 1 : side >= 2; }

// A guided selection.  The digits of a key say little about where the k smallest of some hundred thousand end: the first is sign and
// exponent, so a second pass over the instances is always needed and near convergence a third.  A selection that follows another
// one counts once, in bins of a sixteenth of an octave of the distance from where the last one ended, its k-th entry, to either
// side, in units of how far its k/2-th was from there.  Then it is some hundred entries further to the new end, and the bin of
// that holds a sixteenth of them where f has moved little; a list has room for as many more than k as that.  The bins are monotonous in f
// (each of the operations rounds monotonously), so everything up to the k-th's bin is a superset of the k smallest whatever the
// guide was; if it does not fit the list, the digits are resolved from the first by sel_final_kernel's tail, which says so
// (`missed`; none of the 5,000 selections of seven classes of 300,000 rows but one, two of 98 of 20,000 x 784), and the caller asks
// for a selection by digits for a while.  Two launches less per outer iteration: epsilon-SVR 40000x90 69.4 -> 66.8 ms a call,
// 30,000 blobs of which thousands share a value 25.0 -> 21.4; seven classes of 300,000 rows within what their runs differ by.  Bins from the first entry on instead, in units of the k-th's distance, missed where the candidates
// crowd around the k-th (five of 42 of 20,000 x 784, 43.2 -> 44.1 ms).
struct SelGuide {
    double at, scale;
};
__device__ __forceinline__ SelGuide sel_guide(const SelWorkspace &w, int side, bool desc) {
    const uint64_t k0 = w.guide[2 * side], k1 = w.guide[2 * side + 1];
    const double half = key_to_f(desc ? ~k0 : k0);
    SelGuide g;
    g.at = key_to_f(desc ? ~k1 : k1);
    double unit = desc ? half - g.at : g.at - half;
    if (!(unit > 1e-290 && unit < 1e290)) unit = __builtin_fabs(g.at) * 0x1p-10;   // (all of them equal, or a guide from nowhere)
    g.scale = 1.0 / unit;
    if (!(unit > 1e-290 && unit < 1e290 && __builtin_fabs(g.at) < 1e290)) { g.at = 0.0; g.scale = 0.0; }   // (one bin)
    return g;
}
__device__ __forceinline__ uint32_t sel_guided_bin(double f, uint64_t side_key, const SelGuide &g, bool desc) {
    const double x = (desc ? g.at - f : f - g.at) * g.scale;
    if (x != x) return side_key >> 63 ? SEL_GUIDE_BINS - 1 : 0;   // (f is infinite or no number: where its key belongs)
    const int d = (__float_as_int(__builtin_fabsf((float) x)) >> 19) - ((127 - 8) << 4);   // from 2^-8 units on, sixteen bins an octave, sixteen octaves
    const int b = d < 0 ? 0 : d < SEL_GUIDE_BINS / 2 ? d : SEL_GUIDE_BINS / 2 - 1;
    return (uint32_t) (x < 0.0 ? SEL_GUIDE_BINS / 2 - 1 - b : SEL_GUIDE_BINS / 2 + b);
}
// One instance's count; the last bin, which holds whoever is far away, once per wavefront.
__device__ __forceinline__ void sel_guided_add(uint32_t *h, bool valid, uint32_t bin) {
    const uint64_t far = __ballot(valid && bin == SEL_GUIDE_BINS - 1);
    if (far && (int) (threadIdx.x & 63) == __builtin_ctzll(far)) atomicAdd(&h[SEL_GUIDE_BINS - 1], (uint32_t) __popcll(far));
    if (valid && bin < SEL_GUIDE_BINS - 1) atomicAdd(&h[bin], 1u);
}

// What a call needs to find in the workspace: zeroed histograms for the digits that are counted with atomics
// by the whole grid and zeroed counters.  Written by sel_init_kernel, and again
// by sel_final_kernel once it has read what it needs, so that the next call on the same workspace (same n,
// same sides) can start counting straight away.
__device__ __forceinline__ void sel_clear_hist(const SelWorkspace &w, int p_full, int64_t gid, int64_t stride) {
    for (int64_t e = gid; e < (int64_t) p_full * SEL_MAX_SIDES * SEL_BINS; e += stride) w.hist[e] = 0;
}

__global__ void sel_init_kernel(SelWorkspace w, int p_full) {
    const int64_t gid = (int64_t) blockIdx.x * blockDim.x + threadIdx.x;
    sel_clear_hist(w, p_full, gid, (int64_t) gridDim.x * blockDim.x);
    if (gid <= SEL_MAX_SIDES) w.count[gid] = 0;
    if (gid < SEL_MAX_SIDES * SEL_GUIDE_BINS) w.guide_hist[gid] = 0;
    if (gid < SEL_MAX_SIDES * 2) w.guide[gid] = 0;
}

// Computes, in LDS, the state after pass p-1's histogram has been consumed (st_out), from the
// state before it (global state[p-1]) and hist[p-1].  Every workgroup does this redundantly; the first
// SEL_T threads of the workgroup do the work, any others only join the barriers.
//
// A side is decided as soon as the boundary bucket can be taken whole: when everything up to and including
// it fits the side's list (MAX_WS entries), the list is a superset of the k smallest candidates, in which
// every extra entry is larger than all of them, and sel_final_kernel sorts the list and reads it from the
// front.  With 11-bit digits that is the normal case after the second or third pass.
template <int NS>
__device__ void sel_advance_state(const SelWorkspace &w, const SelGeom &g, int p, SelState *st_out /* LDS [NS] */,
                                  uint32_t *scratch /* LDS [NS * SEL_T / 64] */) {
    constexpr int EACH = SEL_BINS / SEL_T, WAVES = SEL_T / 64;
    const int tid = threadIdx.x;
    const bool worker = tid < SEL_T;
    const int lane = tid & 63, wave = tid >> 6;
    SelState st[NS];
    uint32_t c[NS][EACH], sum[NS], incl[NS];
    if (worker) {   // (every side's state and counts at once: one memory latency)
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            st[s] = w.state[(p - 1) * SEL_MAX_SIDES + s];
            const uint4 *h = (const uint4 *) (w.hist + ((size_t) (p - 1) * SEL_MAX_SIDES + s) * SEL_BINS + tid * EACH);
#pragma unroll
            for (int e = 0; e < EACH / 4; ++e) {
                const uint4 v = h[e];
                c[s][4 * e] = v.x; c[s][4 * e + 1] = v.y; c[s][4 * e + 2] = v.z; c[s][4 * e + 3] = v.w;
            }
        }
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            sum[s] = 0;
#pragma unroll
            for (int e = 0; e < EACH; ++e) sum[s] += c[s][e];
            incl[s] = sum[s];
#pragma unroll
            for (int d = 1; d < 64; d <<= 1) {
                const uint32_t o = __shfl_up(incl[s], d, 64);
                if (lane >= d) incl[s] += o;
            }
            if (lane == 63) scratch[s * WAVES + wave] = incl[s];
        }
    }
    __syncthreads();
    if (worker) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (st[s].done) {
                if (tid == 0) st_out[s] = st[s];
                continue;
            }
            uint32_t excl = incl[s] - sum[s], total = 0;
#pragma unroll
            for (int wv = 0; wv < WAVES; ++wv) {
                if (wv < wave) excl += scratch[s * WAVES + wv];
                total += scratch[s * WAVES + wv];
            }
            if (total < st[s].k_rem) {
                // fewer candidates than requested (only possible on the first digit): take them all
                if (tid == 0) { st[s].done = 1; st[s].k_rem = total; st_out[s] = st[s]; }
            } else if (excl < st[s].k_rem && st[s].k_rem <= excl + sum[s]) {
                uint32_t below = excl, cb = 0;
                int b = 0;
                bool in_front = true;
#pragma unroll
                for (int e = 0; e < EACH; ++e) {
                    const bool here = in_front && below + c[s][e] >= st[s].k_rem;
                    if (here) { b = tid * EACH + e; cb = c[s][e]; }
                    in_front = in_front && !here;
                    if (in_front) below += c[s][e];
                }
                const uint32_t taken = g.k - st[s].k_rem;   // entries of the buckets decided by earlier digits
                bool is_key; int shift, width;
                sel_digit_geom(p - 1, g.idx_bits, is_key, shift, width);
                if (is_key) st[s].pk |= (uint64_t) b << shift; else st[s].pi |= (uint32_t) b << shift;
                st[s].k_rem -= below;
                st[s].pad = (uint32_t) p;
                if (cb == st[s].k_rem || p == g.n_pass || taken + below + cb <= (uint32_t) MAX_WS) st[s].done = 1;
                st_out[s] = st[s];
            }
        }
    }
    __syncthreads();
}

// One count for `bin` from every lane with `valid` set, added to the LDS histogram h with one atomic per distinct
// bin of the wavefront instead of one per lane: the first digit of f (sign and exponent) is the same for most
// instances, and atomics of 64 lanes on one LDS word are carried out one after the other.  May be called in
// divergent code: only the lanes that call take part.
__device__ __forceinline__ void sel_hist_add_wave(uint32_t *h, bool valid, uint32_t bin) {
    uint64_t todo = __ballot(valid);
    while (todo) {
        const int leader = __builtin_ctzll(todo);
        const uint32_t b = (uint32_t) __builtin_amdgcn_readlane((int) bin, leader);
        const uint64_t same = __ballot(valid && bin == b);
        if ((int) (threadIdx.x & 63) == leader) atomicAdd(&h[b], (uint32_t) __popcll(same));
        todo &= ~same;
    }
}

// One candidate's contribution to the histograms of digit p: on every undecided side it belongs to, if it
// matches that side's prefix.
__device__ __forceinline__ void sel_count(const SelGeom &g, const SelState *st, uint32_t (*lhist)[SEL_BINS], int p,
                                          bool is_key, int shift, uint32_t dmask, uint64_t key, uint32_t fl, int64_t j) {
    for (int s = 0; s < g.n_sides; ++s) {
        if (!(fl & (1u << s)) || st[s].done) continue;
        const bool desc = sel_side_descending(s, g.n_sides);
        const uint64_t k2 = desc ? ~key : key;
        const uint32_t i2 = desc ? g.idx_mask - (uint32_t) j : (uint32_t) j;
        if (sel_cmp_prefix(k2, i2, st[s], p, g.idx_bits) != 0) continue;
        const uint32_t dg = is_key ? (uint32_t) (k2 >> shift) & dmask : (i2 >> shift) & dmask;
        atomicAdd(&lhist[s][dg], 1u);
    }
}

// Side membership of an unmarked instance (csmosolver.cpp:133-159, nusmosolver.cpp:60-115).
__device__ __forceinline__ uint32_t sel_flags(double a, double yy, double Cp, double Cn, int n_sides) {
    const bool up = is_I_up(a, yy, Cp, Cn), low = is_I_low(a, yy, Cp, Cn);
    if (n_sides == 2) return (up ? 1u : 0u) | (low ? 2u : 0u);
    return ((up && yy > 0) ? 1u : 0u) | ((up && yy < 0) ? 2u : 0u) | ((low && yy > 0) ? 4u : 0u) | ((low && yy < 0) ? 8u : 0u);
}

// What the selection's first pass needs besides f when update_f makes it (NS sides; see update_f_kernel).
struct SelFuse {
    SelWorkspace w;
    SelGeom g;
    const int *y;
    const double *alpha;
    double Cp, Cn;
    const int *marked;
    int n_marked;
    bool guided = false;
};

// ------------------------------------------------------------------------------------------------
// update_f: f[j] -= sum_t alpha_diff[t] * K_t[j]  (smo_kernel.cpp:300-319)
// Bandwidth-bound stream over the ws x n kernel rows.  The non-zero alpha_diff entries are
// compacted (in order) into LDS once per workgroup; rows with alpha_diff == 0 are never read.
// This kernel is for more than 65,536 columns of floats, 32,768 of doubles (update_f_narrow_kernel below for fewer).
// Each thread owns one to four adjacent columns and keeps 8 to 32 row loads in flight.  On the vector-load
// path the columns are dealt evenly to a number of workgroups that is a multiple of 248 (every CU, or every
// CU left to a stream that leaves one CU per XCD to the local solver, gets the same number of workgroups):
// with a grid of full 256-thread workgroups some CUs stream 2 and others 1, and the launch lasts as long as
// the busiest one.
// ------------------------------------------------------------------------------------------------
#define UF_T 256
#define UF_CHUNK 1024

// TK: element type of the kernel rows; COLS columns per thread (consecutive, loaded as one vector of
// COLS elements); UNROLL rows in flight.  Rows are n columns wide and f holds `repeat` stacked copies
// of the n columns, each of which receives the same sum.
//
// NS > 0: the kernel also makes the first pass of the working-set selection that follows on the updated f, over
// the n * repeat stacked instances and NS sides (what sel_pass_kernel does for digit 0: keys, side flags, the
// first digit's histogram, the state before it), while each new f value is still in a register.  The instances
// of the kept half of the working set (sf.marked) that fall among a workgroup's columns are a bit field in LDS.
#define UF_MAX_REPEAT 4
template <typename TK, int COLS, int UNROLL, int NS>
__global__ __launch_bounds__(UF_T) void update_f_kernel(double *__restrict__ f, const double *__restrict__ alpha_diff,
                                                        int ws, const TK *__restrict__ k_rows,
                                                        const int *__restrict__ slots, int64_t ld, int64_t n, int repeat,
                                                        int vec_per_wg, SelFuse sf) {
    typedef TK vec_t __attribute__((ext_vector_type(COLS)));
    __shared__ uint32_t lhist[NS > 0 ? NS : 1][NS > 0 ? SEL_BINS : 1];
    __shared__ uint32_t mark_bits[NS > 0 ? UF_MAX_REPEAT : 1][NS > 0 ? UF_T * 4 / 32 : 1];   // a workgroup owns at most UF_T * COLS <= 1024 columns
    __shared__ double s_ad[UF_CHUNK];
    __shared__ int64_t s_off[UF_CHUNK];
    __shared__ int s_wave_cnt[UF_T / 64];
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int64_t j = ((int64_t) blockIdx.x * vec_per_wg + tid) * COLS;
    const bool act = tid < vec_per_wg && j < n;   // a vector may reach past n, but never past the padded row (checked by the launcher)
    double sum[COLS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) sum[c] = 0.0;
    const int64_t col_lo = (int64_t) blockIdx.x * vec_per_wg * COLS;
    if (NS > 0) {
        for (int e = tid; e < NS * (sf.guided ? SEL_GUIDE_BINS : SEL_BINS); e += UF_T) (&lhist[0][0])[e] = 0;
        for (int e = tid; e < UF_MAX_REPEAT * (UF_T * 4 / 32); e += UF_T) (&mark_bits[0][0])[e] = 0;
        if (blockIdx.x == 0 && tid < NS) {
            SelState s0;
            s0.pk = 0; s0.pi = 0; s0.k_rem = sf.g.k; s0.done = 0; s0.pad = 0;
            sf.w.state[tid] = s0;   // the state before digit 0, for the next pass
        }
        __syncthreads();
        const int64_t col_hi = col_lo + (int64_t) vec_per_wg * COLS;
        for (int i = tid; i < sf.n_marked; i += UF_T) {
            const int64_t id = sf.marked[i];
            for (int r = 0; r < repeat; ++r) {
                const int64_t c = id - r * n;   // column, if the id lies in copy r
                if (c >= col_lo && c < col_hi && c < n) atomicOr(&mark_bits[r][(c - col_lo) >> 5], 1u << ((c - col_lo) & 31));
            }
        }
        // (the barriers of the loop below, or the one before the epilogue, order these writes before their readers)
    }
    for (int base = 0; base < ws; base += UF_CHUNK) {
        // ordered compaction of this chunk's non-zero entries: thread t owns entries 4t..4t+3
        double v[4];
        int cnt = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int t = base + tid * 4 + e;
            v[e] = t < ws ? alpha_diff[t] : 0.0;
            cnt += (v[e] != 0.0);
        }
        int incl = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        if (lane == 63) s_wave_cnt[wave] = incl;
        __syncthreads();
        int wave_base = 0, total = 0;
#pragma unroll
        for (int w = 0; w < UF_T / 64; ++w) {
            if (w < wave) wave_base += s_wave_cnt[w];
            total += s_wave_cnt[w];
        }
        int pos = wave_base + incl - cnt;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            if (v[e] != 0.0) {
                const int t = base + tid * 4 + e;
                s_ad[pos] = v[e];
                s_off[pos] = (int64_t) (slots ? slots[t] : t) * ld;
                ++pos;
            }
        }
        __syncthreads();
        if (act) {
            int u = 0;
            for (; u + UNROLL <= total; u += UNROLL) {
                vec_t k[UNROLL];
#pragma unroll
                for (int e = 0; e < UNROLL; ++e) k[e] = load_streaming((const vec_t *) (k_rows + s_off[u + e] + j));
#pragma unroll
                for (int e = 0; e < UNROLL; ++e) {
                    const double ad = s_ad[u + e];
#pragma unroll
                    for (int c = 0; c < COLS; ++c) sum[c] = __builtin_fma(ad, (double) k[e][c], sum[c]);
                }
            }
            for (; u < total; ++u) {
                const vec_t k = load_streaming((const vec_t *) (k_rows + s_off[u] + j));
                const double ad = s_ad[u];
#pragma unroll
                for (int c = 0; c < COLS; ++c) sum[c] = __builtin_fma(ad, (double) k[c], sum[c]);
            }
        }
        __syncthreads();
    }
    if (NS == 0) {
        if (act) {
            for (int r = 0; r < repeat; ++r) {
#pragma unroll
                for (int c = 0; c < COLS; ++c)
                    if (j + c < n) f[(int64_t) r * n + j + c] -= sum[c];
            }
        }
        return;
    }
    SelGuide guide[NS > 0 ? NS : 1];
#pragma unroll
    for (int s = 0; s < NS; ++s) guide[s] = sel_guide(sf.w, s, sel_side_descending(s, NS));
    __syncthreads();
    if (act) {
        for (int r = 0; r < repeat; ++r) {
            const int64_t j0 = (int64_t) r * n + j;   // the first of this thread's stacked instances in copy r
            // every load first, then the arithmetic: one memory latency for the lot
            double fo[COLS], al[COLS];
            int yv[COLS];
#pragma unroll
            for (int c = 0; c < COLS; ++c) {
                const bool in = j + c < n;
                fo[c] = in ? f[j0 + c] : 0.0;
                al[c] = in ? sf.alpha[j0 + c] : 0.0;
                yv[c] = in ? sf.y[j0 + c] : 1;
            }
            uint32_t fl_all = 0;
#pragma unroll
            for (int c = 0; c < COLS; ++c) {
                const bool in = j + c < n;
                const double fn = fo[c] - sum[c];
                const uint64_t key = f_to_key(fn);
                const int bit = (int) (j + c - col_lo);
                uint32_t fl = 0;
                if (in && !((mark_bits[r][bit >> 5] >> (bit & 31)) & 1u)) fl = sel_flags(al[c], (double) yv[c], sf.Cp, sf.Cn, NS);
                if (in) {
                    f[j0 + c] = fn;
                    sf.w.keys[j0 + c] = key;
                }
                fl_all |= fl << (8 * c);
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const bool desc = sel_side_descending(s, NS);
                    const uint64_t k2 = desc ? ~key : key;
                    if (sf.guided) sel_guided_add(&lhist[0][0] + s * SEL_GUIDE_BINS, (fl >> s) & 1u, sel_guided_bin(fn, k2, guide[s], desc));
                    else sel_hist_add_wave(lhist[s], (fl >> s) & 1u, (uint32_t) (k2 >> (64 - SEL_DIGIT)));   // digit 0: the key's top bits
                }
            }
            if (COLS == 4 && (j0 & 3) == 0 && j + COLS <= n) {
                *(uint32_t *) (sf.w.flags + j0) = fl_all;   // four flag bytes at once
            } else {
#pragma unroll
                for (int c = 0; c < COLS; ++c)
                    if (j + c < n) sf.w.flags[j0 + c] = (uint8_t) (fl_all >> (8 * c));
            }
        }
    }
    __syncthreads();
    uint32_t *const counts = sf.guided ? sf.w.guide_hist : sf.w.hist;   // [s][bin], s < NS
    for (int e = tid; e < NS * (sf.guided ? SEL_GUIDE_BINS : SEL_BINS); e += UF_T) {
        const uint32_t c = (&lhist[0][0])[e];
        if (c) atomicAdd(&counts[e], c);
    }
}

// The same for fewer columns.  One thread per column leaves most of the chip without work then, and a column's some 500
// rows come in sixteen batches one memory latency apart: 27 us for 3,200 columns and 31 for 40,000.  Here a workgroup has
// 64 * COLS columns and eight wavefronts; groups of R neighbouring rows are dealt to them in turn, so that all eight have theirs on
// their way at once, and they add them in turn: the sums of a column stay one chain in the rows' order, handed on through
// LDS.  Bound by that chain where columns are few, by HBM where they are many.  A row of the chain costs its addition and whatever stands
// between two of them: the coefficients lie in a register, a lane each, and come by v_readlane four rows ahead (read from LDS one
// pair after another, each pair behind a wait, a row took 50 cycles; 26 with the hand-overs now), and a wavefront that asks for its
// next rows (some 1,600 cycles of issue) holds up nobody, since the others wait for the turn's number and not at a barrier.  1,024 and 516
// of 1,024 float rows, us: 3,200 columns 19.6 / 11.5 -> 15.9 / 9.9, 16,384 20.2 / 12.3 -> 17.1 / 10.8; with the selection behind it,
// 516 rows: 40.1 -> 32.9 and 46.1 -> 38.5.
#define UN_WAVES 8
// The sums of a wavefront's columns on their way to the next: written, then the number of the turn (the LDS takes a wavefront's
// accesses in order), and read behind that number until it is the wanted one.  Rows stay on their way meanwhile, across no barrier.
template <int COLS>
__device__ __forceinline__ void un_pass_turn(int *turn, int next, double *slot, const double (&sum)[COLS]) {
    if constexpr (COLS == 1)
        asm volatile("ds_write_b64 %0, %1\n\tds_write_b32 %2, %3" :: "v"(lds_at(slot)), "v"(sum[0]), "v"(lds_at(turn)), "v"(next) : "memory");
    else
        asm volatile("ds_write2_b64 %0, %1, %2 offset1:1\n\tds_write_b32 %3, %4"
                     :: "v"(lds_at(slot)), "v"(sum[0]), "v"(sum[1]), "v"(lds_at(turn)), "v"(next) : "memory");
}
template <int COLS>
__device__ __forceinline__ void un_take_turn(int *turn, int mine, double *slot, double (&sum)[COLS]) {
    static_assert(COLS == 1 || COLS == 2, "columns per thread");
    typedef double v2d __attribute__((ext_vector_type(2)));
    int at;
    do {
        if constexpr (COLS == 1) {
            asm volatile("ds_read_b32 %0, %2\n\tds_read_b64 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(at), "=&v"(sum[0]) : "v"(lds_at(turn)), "v"(lds_at(slot)) : "memory");
        } else {
            v2d both;
            asm volatile("ds_read_b32 %0, %2\n\tds_read_b128 %1, %3\n\ts_waitcnt lgkmcnt(0)"
                         : "=&v"(at), "=&v"(both) : "v"(lds_at(turn)), "v"(lds_at(slot)) : "memory");
            sum[0] = both[0];
            sum[1] = both[1];
        }
    } while (__builtin_amdgcn_readfirstlane(at) != mine);
}
template <typename TK, int COLS, int R, int NS>
__global__ __launch_bounds__(64 * UN_WAVES, 4) void update_f_narrow_kernel(double *__restrict__ f, const double *__restrict__ alpha_diff,
                                                                        int ws, const TK *__restrict__ k_rows,
                                                                        const int *__restrict__ slots, int64_t ld, int64_t n, int repeat, SelFuse sf) {
    typedef TK vec_t __attribute__((ext_vector_type(COLS)));
    constexpr int T = 64 * UN_WAVES, EACH = UF_CHUNK / T;
    __shared__ uint32_t lhist[NS > 0 ? NS : 1][NS > 0 ? SEL_BINS : 1];
    __shared__ uint32_t mark_bits[NS > 0 ? UF_MAX_REPEAT : 1][2 * COLS];
    __shared__ double s_ad[UF_CHUNK];
    __shared__ int64_t s_off[UF_CHUNK];
    __shared__ __align__(16) double s_sum[64 * COLS];
    __shared__ int s_wave_cnt[UN_WAVES], s_turn;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int64_t col_lo = (int64_t) blockIdx.x * 64 * COLS, j = col_lo + lane * COLS;
    const int64_t jc = j < n ? j : (n - 1) / COLS * COLS;   // (a lane behind the last column reads that column's vector)
    // what the epilogue needs of this wavefront's copy of the columns: on its way from here on
    double fo[COLS], al[COLS];
    int yv[COLS];
    auto fetch = [&](int r) {
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            const int64_t at = (int64_t) r * n + (j + c < n ? j + c : n - 1);
            fo[c] = f[at];
            if (NS > 0) {
                al[c] = sf.alpha[at];
                yv[c] = sf.y[at];
            }
        }
    };
    // a chunk's coefficients and slots, EACH neighbouring ones per thread
    double v[EACH];
    int slot[EACH];
    auto fetch_chunk = [&](int base) {
#pragma unroll
        for (int e = 0; e < EACH; ++e) {
            const int t = base + tid * EACH + e, tc = t < ws ? t : ws - 1;
            v[e] = t < ws ? alpha_diff[tc] : 0.0;
            slot[e] = slots ? slots[tc] : tc;
        }
    };
    // (everything that waits for nothing is asked for first: as four latencies one after another it took 2 us)
    if (ws > 0) fetch_chunk(0);
    int mark = NS > 0 && tid < sf.n_marked ? sf.marked[tid] : -1;
    if (wave < repeat) fetch(wave);
    if (tid == 0) s_turn = 0;
    if (NS > 0) {
        for (int e = tid; e < NS * SEL_BINS; e += T) (&lhist[0][0])[e] = 0;
        if (tid < UF_MAX_REPEAT * 2 * COLS) (&mark_bits[0][0])[tid] = 0;
        if (blockIdx.x == 0 && tid < NS) {
            SelState s0;
            s0.pk = 0; s0.pi = 0; s0.k_rem = sf.g.k; s0.done = 0; s0.pad = 0;
            sf.w.state[tid] = s0;   // the state before digit 0, for the next pass
        }
        __syncthreads();
        for (int i = tid; i < sf.n_marked; i += T) {
            const int64_t id = i == tid ? mark : sf.marked[i];
            for (int r = 0; r < repeat; ++r) {
                const int64_t c = id - r * n;   // column, if the id lies in copy r
                if (c >= col_lo && c < col_lo + 64 * COLS && c < n) atomicOr(&mark_bits[r][(c - col_lo) >> 5], 1u << ((c - col_lo) & 31));
            }
        }
    }
    double sum[COLS];
#pragma unroll
    for (int c = 0; c < COLS; ++c) sum[c] = 0.0;
    int turns = 0;   // groups of the chunks before
    for (int base = 0; base < ws; base += UF_CHUNK) {
        // ordered compaction of this chunk's non-zero entries
        if (base > 0) fetch_chunk(base);
        int cnt = 0;
#pragma unroll
        for (int e = 0; e < EACH; ++e) cnt += (v[e] != 0.0);
        int incl = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        if (lane == 63) s_wave_cnt[wave] = incl;
        __syncthreads();
        int pos = incl - cnt, total = 0;
#pragma unroll
        for (int w = 0; w < UN_WAVES; ++w) {
            if (w < wave) pos += s_wave_cnt[w];
            total += s_wave_cnt[w];
        }
#pragma unroll
        for (int e = 0; e < EACH; ++e)
            if (v[e] != 0.0) {
                s_ad[pos] = v[e];
                s_off[pos] = (int64_t) slot[e] * ld;
                ++pos;
            }
        __syncthreads();
        // Groups of R rows are dealt to the wavefronts in turn: group g is wavefront g % UN_WAVES's, which asks for its next one as
        // soon as it has added the last.  s_turn is the group whose turn it is; a wavefront waits for its own and nothing else, so
        // that another's requests hold nobody up.
        const int groups = (total + R - 1) / R;
        vec_t k[R];
        double ad = 0.0;   // lane u's is the coefficient of the group's row u
        auto request = [&](int g) {
            ad = s_ad[g * R + (lane & (R - 1)) < total ? g * R + (lane & (R - 1)) : total - 1];
#pragma unroll
            for (int u = 0; u < R; ++u) k[u] = load_streaming((const vec_t *) (k_rows + s_off[g * R + u < total ? g * R + u : total - 1] + jc));
        };
        if (wave < groups) request(wave);
#pragma unroll 1
        for (int g = wave; g < groups; g += UN_WAVES) {
            if (turns + g > 0) un_take_turn<COLS>(&s_turn, turns + g, s_sum + lane * COLS, sum);   // the sums so far come from the wavefront before
            __builtin_amdgcn_s_setprio(2);   // (in front of the wavefronts that wait)
            const int m = total - g * R;
            if (m >= R) {
                constexpr int AHEAD = 4;   // rows whose coefficient and values are made ready while one is added
                double a[AHEAD], wide[AHEAD][COLS];
                auto ready = [&](int u) {
                    a[u % AHEAD] = readlane_f64(ad, u);
#pragma unroll
                    for (int c = 0; c < COLS; ++c) wide[u % AHEAD][c] = (double) k[u][c];
                };
#pragma unroll
                for (int u = 0; u < AHEAD; ++u) ready(u);
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < R; ++u) {
#pragma unroll
                    for (int c = 0; c < COLS; ++c) sum[c] = __builtin_fma(a[u % AHEAD], wide[u % AHEAD][c], sum[c]);
                    if (u + AHEAD < R) ready(u + AHEAD);
                    __builtin_amdgcn_sched_barrier(0);
                }
            } else {
#pragma unroll
                for (int u = 0; u < R; ++u)
                    if (u < m) {
                        const double a = readlane_f64(ad, u);
#pragma unroll
                        for (int c = 0; c < COLS; ++c) {
                            TK v = k[u][c];
                            asm("" : "+v"(v));   // (or the conversions of both branches would be made in front of them, and all be held)
                            sum[c] = __builtin_fma(a, (double) v, sum[c]);
                        }
                    }
            }
            un_pass_turn<COLS>(&s_turn, turns + g + 1, s_sum + lane * COLS, sum);
            __builtin_amdgcn_s_setprio(0);
            if (g + UN_WAVES < groups) request(g + UN_WAVES);
        }
        turns += groups;
        __syncthreads();
        if (total > 0) {   // every wavefront goes on from the chunk's sums
#pragma unroll
            for (int c = 0; c < COLS; ++c) sum[c] = s_sum[lane * COLS + c];
            __syncthreads();
        }
    }
    if (NS > 0 && ws <= 0) __syncthreads();   // (the marks)
    SelGuide guide[NS > 0 ? NS : 1];
#pragma unroll
    for (int s = 0; s < NS; ++s) guide[s] = sel_guide(sf.w, s, sel_side_descending(s, NS));
    for (int r = wave; r < repeat; r += UN_WAVES) {
        if (r != wave) fetch(r);
        const int64_t j0 = (int64_t) r * n + j;
#pragma unroll
        for (int c = 0; c < COLS; ++c) {
            const bool in = j + c < n;
            const double fn = fo[c] - sum[c];
            if (in) f[j0 + c] = fn;
            if constexpr (NS > 0) {
                const uint64_t key = f_to_key(fn);
                const int bit = lane * COLS + c;
                uint32_t fl = 0;
                if (in && !((mark_bits[r][bit >> 5] >> (bit & 31)) & 1u)) fl = sel_flags(al[c], (double) yv[c], sf.Cp, sf.Cn, NS);
                if (in) {
                    sf.w.keys[j0 + c] = key;
                    sf.w.flags[j0 + c] = (uint8_t) fl;
                }
#pragma unroll
                for (int s = 0; s < NS; ++s) {
                    const bool desc = sel_side_descending(s, NS);
                    const uint64_t k2 = desc ? ~key : key;
                    if (sf.guided) sel_guided_add(&lhist[0][0] + s * SEL_GUIDE_BINS, (fl >> s) & 1u, sel_guided_bin(fn, k2, guide[s], desc));
                    else sel_hist_add_wave(lhist[s], (fl >> s) & 1u, (uint32_t) (k2 >> (64 - SEL_DIGIT)));   // digit 0: the key's top bits
                }
            }
        }
    }
    if (NS == 0) return;
    __syncthreads();
    uint32_t *const counts = sf.guided ? sf.w.guide_hist : sf.w.hist;   // [s][bin], s < NS
    for (int e = tid; e < NS * (sf.guided ? SEL_GUIDE_BINS : SEL_BINS); e += T) {
        const uint32_t c = (&lhist[0][0])[e];
        if (c) atomicAdd(&counts[e], c);
    }
}

// f from a non-zero alpha: batches of rows, each summed and then taken from f (csmosolver.cpp:189-214).  Bound by memory
// latency: few columns (a few thousand instances), many rows, and the sums of a column one after another.  One column per
// thread in workgroups of one wavefront (5,001 columns are 79 of them), the rows one stream across the batches, the next UB
// of them on their way while UB are added: 1,010 rows of 5,001 floats 70 us, ten launches of update_f_kernel 88 and the gaps
// between them.  nu-SVC on 5,001 x 23 starts from 2,000 such rows: 5.01 -> 4.57 ms.  (With many columns update_f_kernel is
// the better one: whoever has both calls chooses.)
#define UB 32
template <typename TK>
__global__ __launch_bounds__(64) void update_f_batches_kernel(double *__restrict__ f, const double *__restrict__ coef, int n_rows, int batch,
                                                              const TK *__restrict__ k_rows, int64_t ld, int64_t n, int repeat) {
    const int64_t j = (int64_t) blockIdx.x * 64 + threadIdx.x;
    const TK *const col = k_rows + (j < n ? j : n - 1);
    double sum = 0.0;
    int left = batch;   // rows of the batch still to come
    auto add = [&](int t, double c, TK k) {
        sum = __builtin_fma(c, (double) k, sum);
        if (--left == 0 || t == n_rows - 1) {
            if (j < n)
                for (int r = 0; r < repeat; ++r) f[r * n + j] -= sum;
            sum = 0.0;
            left = batch;
        }
    };
    TK next[UB];
    double next_c[UB];
    const int whole = n_rows / UB * UB;
    auto fetch = [&](int t) {
#pragma unroll
        for (int u = 0; u < UB; ++u) next[u] = col[(int64_t) (t + u) * ld];
#pragma unroll
        for (int u = 0; u < UB; ++u) next_c[u] = coef[t + u];
    };
    if (whole > 0) fetch(0);
    for (int t = 0; t < whole; t += UB) {
        TK k[UB];
        double c[UB];
#pragma unroll
        for (int u = 0; u < UB; ++u) { k[u] = next[u]; c[u] = next_c[u]; }
        fetch(t + UB < whole ? t + UB : t);
        if (left > UB) {   // no batch ends among these rows, unless they are the last ones
#pragma unroll
            for (int u = 0; u < UB; ++u) sum = __builtin_fma(c[u], (double) k[u], sum);
            left -= UB;
            if (t + UB == n_rows && j < n)
                for (int r = 0; r < repeat; ++r) f[r * n + j] -= sum;
        } else {
#pragma unroll
            for (int u = 0; u < UB; ++u) add(t + u, c[u], k[u]);
        }
    }
    for (int t = whole; t < n_rows; ++t) add(t, coef[t], col[(int64_t) t * ld]);
}

// Pass p: histogram of digit p of the not-yet-decided candidates.  Pass 0 also builds keys and flags; there a
// workgroup walks one contiguous chunk of the instances and keeps the chunk's marked instances (the half of the
// previous working set that stays, csmosolver.cpp:65-71: never candidates) as a bit field in LDS.
#define SEL_CHUNK_MAX 65536
template <int NS>   // NS = g.n_sides: two sides need half the LDS of four, and a workgroup finds room on a busy CU sooner
__global__ __launch_bounds__(SEL_T) void sel_pass_kernel(SelWorkspace w, const double *__restrict__ f,
                                                         const int *__restrict__ y, const double *__restrict__ alpha,
                                                         int64_t n, double Cp, double Cn, SelGeom g, int p,
                                                         const int *__restrict__ marked, int n_marked) {
    __shared__ uint32_t lhist[NS][SEL_BINS];
    __shared__ SelState st[SEL_MAX_SIDES];
    __shared__ uint32_t scratch[SEL_T + 16];
    __shared__ uint32_t mark_bits[SEL_CHUNK_MAX / 32];
    const int tid = threadIdx.x;
    if (p == 0) {
        if (tid < g.n_sides) {
            SelState s0;
            s0.pk = 0; s0.pi = 0; s0.k_rem = g.k; s0.done = 0; s0.pad = 0;
            st[tid] = s0;
            if (blockIdx.x == 0) w.state[tid] = s0;   // the state before digit 0, for the next pass
        }
        __syncthreads();
    } else {
        sel_advance_state<NS>(w, g, p, st, scratch);
        if (blockIdx.x == 0 && tid < g.n_sides) w.state[p * SEL_MAX_SIDES + tid] = st[tid];
    }
    bool any = false;
    for (int s = 0; s < g.n_sides; ++s) any |= !st[s].done;
    if (!any) return;
    for (int e = tid; e < NS * SEL_BINS; e += SEL_T) (&lhist[0][0])[e] = 0;
    bool is_key; int shift, width;
    sel_digit_geom(p, g.idx_bits, is_key, shift, width);
    const uint32_t dmask = (1u << width) - 1;
    if (p == 0) {
        const int64_t chunk = (n + gridDim.x - 1) / gridDim.x;   // <= SEL_CHUNK_MAX (the host sizes the grid)
        const int64_t lo = (int64_t) blockIdx.x * chunk;
        const int64_t hi = lo + chunk < n ? lo + chunk : n;
        for (int e = tid; e < (int) ((chunk + 31) >> 5); e += SEL_T) mark_bits[e] = 0;
        __syncthreads();
        for (int i = tid; i < n_marked; i += SEL_T) {
            const int64_t id = marked[i];
            if (id >= lo && id < hi) atomicOr(&mark_bits[(id - lo) >> 5], 1u << ((id - lo) & 31));
        }
        __syncthreads();
        for (int64_t j = lo + tid; j < hi; j += SEL_T) {
            const double a = alpha[j];
            const double yy = (double) y[j];
            const uint64_t key = f_to_key(f[j]);
            uint32_t fl = 0;
            if (!((mark_bits[(j - lo) >> 5] >> ((j - lo) & 31)) & 1u)) fl = sel_flags(a, yy, Cp, Cn, g.n_sides);
            w.keys[j] = key;
            w.flags[j] = (uint8_t) fl;
            sel_count(g, st, lhist, p, is_key, shift, dmask, key, fl, j);
        }
    } else {
        __syncthreads();
        const int64_t stride = (int64_t) gridDim.x * SEL_T;
        for (int64_t j0 = (int64_t) blockIdx.x * SEL_T + tid; j0 < n; j0 += stride * SEL_EACH) {
            uint32_t fl[SEL_EACH];
            uint64_t key[SEL_EACH];
#pragma unroll
            for (int e = 0; e < SEL_EACH; ++e) {
                const int64_t j = j0 + e * stride, jc = j < n ? j : n - 1;
                fl[e] = j < n ? w.flags[jc] : 0u;
                key[e] = w.keys[jc];
            }
#pragma unroll
            for (int e = 0; e < SEL_EACH; ++e)
                if (fl[e]) sel_count(g, st, lhist, p, is_key, shift, dmask, key[e], fl[e], j0 + e * stride);
        }
    }
    __syncthreads();
    uint32_t *gh = w.hist + (size_t) p * SEL_MAX_SIDES * SEL_BINS;
    for (int e = tid; e < g.n_sides * SEL_BINS; e += SEL_T) {
        const uint32_t c = (&lhist[0][0])[e];
        if (c) atomicAdd(&gh[e], c);
    }
}

// Whether instance j is among those a side takes; st is the side's final state.
__device__ __forceinline__ bool sel_taken(const SelGeom &g, const SelState &st, uint64_t k2, uint32_t i2) {
    if (st.k_rem == 0 && st.done) return false;   // nothing to take on this side
    // compare on the digits this side consumed before it was decided
    return sel_cmp_prefix(k2, i2, st, (int) st.pad, g.idx_bits) <= 0;
}

// Appends the selected candidates among instances [lo, hi) to their sides' lists.  A workgroup counts its own first and asks for their
// places once per side and SEL_EACH instances of each thread: the thousand candidates' own atomics on two addresses took longer than
// the rest of the kernel (80,000 instances: 13.7 -> 7.4 us, 20,000: 7.2 -> 5.4).
// GUIDED: a side takes the bins up to st[].pi.
template <int NS, bool GUIDED>
__device__ __forceinline__ void sel_collect(const SelWorkspace &w, const SelGeom &g, const SelState *st, int64_t lo, int64_t hi, uint32_t *scratch) {
    SelGuide guide[NS];
    if (GUIDED)
#pragma unroll
        for (int s = 0; s < NS; ++s) guide[s] = sel_guide(w, s, sel_side_descending(s, NS));
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, waves = (int) blockDim.x >> 6, nt = (int) blockDim.x;
    for (int64_t j0 = lo; j0 < hi; j0 += (int64_t) nt * SEL_EACH) {
        uint64_t key[SEL_EACH];
        uint32_t fl[SEL_EACH];
#pragma unroll
        for (int e = 0; e < SEL_EACH; ++e) {
            const int64_t j = j0 + (int64_t) e * nt + tid;
            fl[e] = j < hi ? w.flags[j] : 0u;
            key[e] = w.keys[j < hi ? j : hi - 1];
        }
        uint64_t takes[NS][SEL_EACH];   // which lanes' instance e goes to the side's list
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const bool desc = sel_side_descending(s, NS);
            int count = 0;
#pragma unroll
            for (int e = 0; e < SEL_EACH; ++e) {
                const uint32_t j = (uint32_t) (j0 + (int64_t) e * nt + tid);
                const uint64_t k2 = desc ? ~key[e] : key[e];
                takes[s][e] = __ballot(((fl[e] >> s) & 1u) &&
                                       (GUIDED ? sel_guided_bin(key_to_f(key[e]), k2, guide[s], desc) <= st[s].pi : sel_taken(g, st[s], k2, desc ? g.idx_mask - j : j)));
                count += __popcll(takes[s][e]);
            }
            if (lane == 0) scratch[s * waves + wave] = (uint32_t) count;
        }
        __syncthreads();
        if (tid < NS) {
            uint32_t total = 0;
            for (int v = 0; v < waves; ++v) {   // (the counts become the wavefronts' first places)
                const uint32_t mine = scratch[tid * waves + v];
                scratch[tid * waves + v] = total;
                total += mine;
            }
            scratch[NS * waves + tid] = total ? atomicAdd(&w.count[tid], total) : 0u;
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const bool desc = sel_side_descending(s, NS);
            uint32_t at = scratch[NS * waves + s] + scratch[s * waves + wave];
#pragma unroll
            for (int e = 0; e < SEL_EACH; ++e) {
                const uint32_t j = (uint32_t) (j0 + (int64_t) e * nt + tid);
                const uint32_t pos = at + (uint32_t) __popcll(takes[s][e] & ((1ull << lane) - 1ull));
                if (((takes[s][e] >> lane) & 1ull) && pos < MAX_WS) {
                    w.list_key[s * MAX_WS + pos] = desc ? ~key[e] : key[e];
                    w.list_idx[s * MAX_WS + pos] = desc ? g.idx_mask - j : j;
                }
                at += (uint32_t) __popcll(takes[s][e]);
            }
        }
        __syncthreads();   // (scratch is written again)
    }
}

__device__ __forceinline__ bool sel_undecided(const SelGeom &g, const SelState *st) {
    bool any = false;
    for (int s = 0; s < g.n_sides; ++s) any |= !st[s].done;
    return any;
}

// After the grid-wide passes every side is normally decided: then this kernel appends every selected candidate
// to its side's list.  If a boundary bucket is still too large it does nothing, and sel_final_kernel goes on.
// The states of a guided selection's sides from the counts: `done` with the last bin that is taken in `pi`; if a side cannot be
// decided, all of them as they are before the first digit.
template <int NS>
__device__ void sel_guided_state(const SelWorkspace &w, const SelGeom &g, SelState *st, uint32_t *scratch) {
    static_assert(2 * SEL_T == SEL_GUIDE_BINS, "two bins per thread");
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint2 c[NS];
    uint32_t incl[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) c[s] = *(const uint2 *) (w.guide_hist + s * SEL_GUIDE_BINS + 2 * tid);
    if (tid < NS) {
        st[tid].pk = 0; st[tid].pi = SEL_GUIDE_BINS - 1; st[tid].k_rem = g.k; st[tid].done = 1; st[tid].pad = 0;   // (fewer than k: all of them)
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        incl[s] = c[s].x + c[s].y;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint32_t o = __shfl_up(incl[s], d, 64);
            if (lane >= d) incl[s] += o;
        }
        if (lane == 63) scratch[s * (SEL_T / 64) + wave] = incl[s];
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        for (int v = 0; v < wave; ++v) incl[s] += scratch[s * (SEL_T / 64) + v];
        if (incl[s] - c[s].x - c[s].y < g.k && g.k <= incl[s]) {
            const bool second = incl[s] - c[s].y < g.k;
            st[s].pi = (uint32_t) (2 * tid + (second ? 1 : 0));
            st[s].done = (second ? incl[s] : incl[s] - c[s].y) <= (uint32_t) MAX_WS;
        }
    }
    __syncthreads();
    const bool undecided = sel_undecided(g, st);
    __syncthreads();
    if (undecided && tid < NS) { st[tid].pi = 0; st[tid].done = 0; }
    __syncthreads();
}

template <int NS, bool GUIDED>
__global__ __launch_bounds__(SEL_T) void sel_compact_kernel(SelWorkspace w, int64_t n, SelGeom g, int p_full) {
    __shared__ SelState st[SEL_MAX_SIDES];
    __shared__ uint32_t scratch[SEL_T + 16];
    if constexpr (GUIDED) sel_guided_state<NS>(w, g, st, scratch);
    else sel_advance_state<NS>(w, g, p_full, st, scratch);
    if (blockIdx.x == 0 && (int) threadIdx.x < NS) w.state[p_full * SEL_MAX_SIDES + threadIdx.x] = st[threadIdx.x];
    if (sel_undecided(g, st)) return;
    const int64_t chunk = (n + gridDim.x - 1) / gridDim.x, lo = (int64_t) blockIdx.x * chunk;
    sel_collect<NS, GUIDED>(w, g, st, lo, lo + chunk < n ? lo + chunk : n, scratch);
}

// Digits p_full .. n_pass-1 and the lists, by one workgroup: only when the grid-wide digits left a boundary
// bucket too large to take whole (many equal f values, e.g. the first iteration of a training run, where the
// instance index has to break the ties).  The workgroup walks the candidates once per remaining digit: slow but
// rare, and it keeps a launch per digit out of every call.  st holds the state before digit p_full.
template <int NS>
__device__ void sel_tail(const SelWorkspace &w, int64_t n, const SelGeom &g, int p_full, SelState *st,
                         uint32_t (*lhist)[SEL_BINS], uint32_t *scratch) {
    const int tid = threadIdx.x, nt = blockDim.x;
    for (int p = p_full; p < g.n_pass && sel_undecided(g, st); ++p) {
        if (tid < g.n_sides) w.state[p * SEL_MAX_SIDES + tid] = st[tid];
        for (int e = tid; e < g.n_sides * SEL_BINS; e += nt) (&lhist[0][0])[e] = 0;
        __syncthreads();
        bool is_key; int shift, width;
        sel_digit_geom(p, g.idx_bits, is_key, shift, width);
        const uint32_t dmask = (1u << width) - 1;
        for (int64_t j = tid; j < n; j += nt) {
            const uint32_t fl = w.flags[j];
            if (fl) sel_count(g, st, lhist, p, is_key, shift, dmask, w.keys[j], fl, j);
        }
        __syncthreads();
        uint32_t *gh = w.hist + (size_t) p * SEL_MAX_SIDES * SEL_BINS;
        for (int e = tid; e < g.n_sides * SEL_BINS; e += nt) gh[e] = (&lhist[0][0])[e];
        __syncthreads();   // sel_advance_state reads state[p] and hist[p] back from memory
        sel_advance_state<NS>(w, g, p + 1, st, scratch);
    }
    sel_collect<NS, false>(w, g, st, 0, n, scratch);
    __syncthreads();
}

// The lists in order by one workgroup: when it alone has made them (sel_tail).
__device__ __forceinline__ bool comp_less(uint64_t ka, uint32_t ia, uint64_t kb, uint32_t ib) {
    return ka < kb || (ka == kb && ia < ib);
}
template <int NS>
__device__ void sel_sort_here(const SelWorkspace &w, const SelGeom &g, const int *cnt, uint64_t (*sk)[MAX_WS], uint32_t (*si)[MAX_WS],
                              int (&id_out)[NS], int (&pos_other)[NS]) {
    const int tid = threadIdx.x;
    for (int s = 0; s < NS; ++s) {
        sk[s][tid] = tid < cnt[s] ? w.list_key[s * MAX_WS + tid] : ~0ull;
        si[s][tid] = tid < cnt[s] ? w.list_idx[s * MAX_WS + tid] : ~0u;
    }
    __syncthreads();
    // Bitonic sort, ascending composite, all sides at once.  Thread t owns compare-exchange pair t & 511 of
    // side t >> 9 (and of side 2 + (t >> 9) when there are four), so every thread works in every stage.  With
    // strides up to 64 a wavefront's 64 pairs cover one closed block of 128 entries, stage after stage: such
    // stages only need the wavefront's own LDS accesses kept in order, not a workgroup barrier.
    int m_sort = 2;
    for (int s = 0; s < NS; ++s)
        while (m_sort < cnt[s]) m_sort <<= 1;   // padding entries are already in place behind the longest list
    const int pr = tid & (MAX_WS / 2 - 1);
    for (int size = 2; size <= m_sort; size <<= 1) {
        for (int strd = size >> 1; strd > 0; strd >>= 1) {
            const int lo = ((pr & ~(strd - 1)) << 1) | (pr & (strd - 1));
            const int hi = lo | strd;
            const bool asc = (lo & size) == 0;
            if (hi < m_sort) {
                for (int s = tid >> 9; s < NS; s += 2) {
                    const uint64_t ka = sk[s][lo], kb = sk[s][hi];
                    const uint32_t ia = si[s][lo], ib = si[s][hi];
                    const bool sw = asc ? comp_less(kb, ib, ka, ia) : comp_less(ka, ia, kb, ib);
                    if (sw) { sk[s][lo] = kb; sk[s][hi] = ka; si[s][lo] = ib; si[s][hi] = ia; }
                }
            }
            const int next_strd = strd > 1 ? strd >> 1 : (2 * size <= m_sort ? size : 0);
            if (strd > 64 || next_strd > 64) {
                __syncthreads();
            } else {
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup");   // LDS accesses of a wavefront complete in order
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    __syncthreads();
    // real instance ids; descending sides stored idx_mask - id
    for (int s = 0; s < NS; ++s)
        if (tid < cnt[s] && sel_side_descending(s, NS)) si[s][tid] = g.idx_mask - si[s][tid];
    __syncthreads();
    // position of each entry in the paired side's list (binary search on the paired side's order)
    constexpr int half = NS / 2;
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int o = s < half ? s + half : s - half;
        int res = -1;
        if (tid < cnt[s]) {
            // key of this instance as the paired side stores it: complement of ours (or of the complement)
            const uint64_t k_here = sk[s][tid];
            const uint64_t k_o = ~k_here;
            const uint32_t id = si[s][tid];
            const uint32_t i_o = sel_side_descending(o, NS) ? g.idx_mask - id : id;
            int lo = 0, hi = cnt[o];
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                const uint32_t im = sel_side_descending(o, NS) ? g.idx_mask - si[o][mid] : si[o][mid];
                if (comp_less(sk[o][mid], im, k_o, i_o)) lo = mid + 1; else hi = mid;
            }
            if (lo < cnt[o] && sk[o][lo] == k_o && si[o][lo] == id) res = lo;
        }
        pos_other[s] = res;
        id_out[s] = (int) si[s][tid];
    }
}

// Final step: the lists in order, the alternating scan, the selection.
//
// The order comes from counting: a wavefront takes an entry, compares it with its side's list, 64 entries at a time, and the
// entries below it are its place; the same against the paired side's list gives the place of the same instance there.  At
// most 1,024 entries a side make 32 workgroups, and the one that draws the last ticket makes the scan.  One workgroup
// that sorted the lists by a bitonic network in LDS and looked the places up by bisection took 26.8 us, 49 with four
// sides, in which the rest of the chip was idle; this takes 9 (bound by the launch and a chain of three memory latencies).  nu-SVC
// 5,001 x 23 4.39 -> 4.06 ms, epsilon-SVR 40,000 x 90 96.8 -> 92.9.  Entries per wavefront 1 / 2 / 4 / 8: 92.5 / 92.8 / 93.5 /
// 95.5 ms there.  Among lanes, whose workgroups wait for room among other pairs', more entries would be better: seven classes of
// 300,000 rows 848 / 846 / 843 / 840, of 500,000 rows 1,525 with two and 1,505 with eight (means of three and two runs; 1,498 when
// one workgroup sorted).
#define SEL_RANK_T 1024
#define SEL_RANK_EACH 2   // entries a wavefront takes
#define SEL_RANK_ENTRIES (SEL_RANK_T / 64 * SEL_RANK_EACH)

// The entries of `key` [0, count) that are below (k, i), and whether (k, i) is among them (OWN: it is); one wavefront.
template <bool OWN>
__device__ __forceinline__ int sel_place(const uint64_t *key, const uint32_t *idx, int count, uint64_t k, uint32_t i, bool &found) {
    const int lane = threadIdx.x & 63;
    int below = 0, equal = 0;
    for (int t0 = 0; t0 < count; t0 += 256) {   // (t < MAX_WS: what lies behind the list is read but not counted)
        uint64_t kt[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) kt[u] = key[t0 + u * 64 + lane];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const bool in = t0 + u * 64 + lane < count;
            below += __popcll(__ballot(in && kt[u] < k));
            equal += __popcll(__ballot(in && kt[u] == k));
        }
    }
    found = OWN;
    if (equal > (OWN ? 1 : 0))   // equal values of f: the index decides
        for (int t = lane; t - lane < count; t += 64) {
            const uint64_t kt = key[t];
            const uint32_t it = idx[t];
            below += __popcll(__ballot(t < count && kt == k && it < i));
            found |= __ballot(t < count && kt == k && it == i) != 0;
        }
    return below;
}

// Where a selection's ids go on the host, when it is to hear of them: pinned memory that the device can write, and a word behind
// them that the host polls (as report_ids_kernel below, in a launch less: epsilon-SVR on 40,000 rows 91.5 -> 90.9 ms; seven
// classes of 300,000 rows level within the 3 % that its runs differ by).
struct SelReport {
    int *ids = nullptr, *word_at = nullptr, word = 0;
    int *missed = nullptr;   // of a guided selection: becomes 1 if the guide did not decide it
};

// (fold_n > 0: the ids are also written modulo fold_n to out_folded, for problems whose instances are stacked
// copies of fold_n stored rows)
template <int NS>   // NS = g.n_sides
__global__ __launch_bounds__(SEL_RANK_T) void sel_final_kernel(SelWorkspace w, int64_t n, SelGeom g, int p_full,
                                                               int *__restrict__ out, int fold_n, int *__restrict__ out_folded, SelReport report, bool guided) {
    // a side's list and its paired side's; on the slow path every side's, and the histograms before that
    __shared__ union {
        struct { uint64_t key[NS][MAX_WS]; uint32_t idx[NS][MAX_WS]; } list;
        uint32_t hist[NS][SEL_BINS];
    } sh;
    __shared__ int cnt[SEL_MAX_SIDES];
    __shared__ int conflict, last, event[NS / 2], alone_in[NS][MAX_WS / 64];
    __shared__ SelState st[SEL_MAX_SIDES];
    __shared__ uint32_t scratch[SEL_T + 16];
    static_assert(SEL_RANK_T == MAX_WS, "one thread per entry in the scan");
    constexpr int half = NS / 2;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int s_own = (int) blockIdx.x / (MAX_WS / SEL_RANK_ENTRIES), s_paired = s_own < half ? s_own + half : s_own - half;
    // (the lists are read before it is known how long they are, and whether they are there at all: one latency for everything)
    uint64_t key[2] = {w.list_key[s_own * MAX_WS + tid], w.list_key[s_paired * MAX_WS + tid]};
    uint32_t idx[2] = {w.list_idx[s_own * MAX_WS + tid], w.list_idx[s_paired * MAX_WS + tid]};
    if (tid < NS) {
        st[tid] = w.state[p_full * SEL_MAX_SIDES + tid];
        cnt[tid] = (int) w.count[tid];
    }
    sel_clear_hist(w, p_full, (int64_t) blockIdx.x * SEL_RANK_T + tid, (int64_t) gridDim.x * SEL_RANK_T);
    if (guided && blockIdx.x == 0)
        for (int e = tid; e < NS * SEL_GUIDE_BINS; e += SEL_RANK_T) w.guide_hist[e] = 0;
    if (tid == 0) conflict = 0;
    __syncthreads();
    int si[NS], pos_other[NS];   // entry `tid` of every side's list in order: instance, its place in the paired side's list or -1
    if (sel_undecided(g, st)) {   // (sel_compact_kernel has left the lists empty)
        if (blockIdx.x != 0) return;
        sel_tail<NS>(w, n, g, p_full, st, sh.hist, scratch);
        if (guided) {   // (its digits' counts are in the place of those that a selection by digits wants to find cleared)
            sel_clear_hist(w, SEL_FULL_MAX, tid, SEL_RANK_T);
            if (tid == 0 && report.missed) __hip_atomic_store(report.missed, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        // (counted with atomics by this workgroup itself: an atomic read)
        if (tid < NS) cnt[tid] = imin_sel((int) __hip_atomic_load(&w.count[tid], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), MAX_WS);
        __syncthreads();
        sel_sort_here<NS>(w, g, cnt, sh.list.key, sh.list.idx, si, pos_other);
        if (tid < NS && cnt[tid] > 0) {
            const int last_at = imin_sel((int) g.k, cnt[tid]) - 1;
            w.guide[2 * tid] = sh.list.key[tid][last_at / 2];
            w.guide[2 * tid + 1] = sh.list.key[tid][last_at];
        }
    } else {
        if (tid < NS) cnt[tid] = imin_sel(cnt[tid], MAX_WS);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            sh.list.key[h][tid] = key[h];
            sh.list.idx[h][tid] = idx[h];
        }
        __syncthreads();
        for (int each = 0; each < SEL_RANK_EACH; ++each) {
            const int e = (int) blockIdx.x % (MAX_WS / SEL_RANK_ENTRIES) * SEL_RANK_ENTRIES + each * (SEL_RANK_T / 64) + wave;
            if (e >= cnt[s_own]) break;
            const uint64_t k = sh.list.key[0][e];
            const uint32_t i = sh.list.idx[0][e];
            bool found;
            const int at = sel_place<true>(sh.list.key[0], sh.list.idx[0], cnt[s_own], k, i, found);
            // (the paired side reads the order from the other end: it holds the complements of key and index)
            const int there = sel_place<false>(sh.list.key[1], sh.list.idx[1], cnt[s_paired], ~k, g.idx_mask - i, found);
            const int last_at = imin_sel((int) g.k, cnt[s_own]) - 1;
            if (lane == 0 && at == last_at / 2) w.guide[2 * s_own] = k;
            if (lane == 0 && at == last_at) w.guide[2 * s_own + 1] = k;
            if (lane == 0) w.sorted[s_own * MAX_WS + at] = make_int2((int) (sel_side_descending(s_own, NS) ? g.idx_mask - i : i), found ? there : -1);
        }
        // (every wavefront's entry is in the L2 before thread 0 publishes them for the others)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) last = __hip_atomic_fetch_add(&w.count[SEL_MAX_SIDES], 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
        __syncthreads();
        if (!last) return;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            const int2 v = tid < cnt[s] ? w.sorted[s * MAX_WS + tid] : make_int2(-1, -1);
            si[s] = v.x;
            pos_other[s] = v.y;
        }
    }
    if (tid <= SEL_MAX_SIDES) w.count[tid] = 0;
    auto put = [&](int at, int id) {
        out[at] = id;
        if (fold_n > 0) out_folded[at] = id < 0 ? -1 : id % fold_n;
        if (report.ids) report.ids[at] = id;
    };
    auto tell = [&] {
        if (!report.ids) return;
        // (every wavefront's ids have arrived, then one release for all: a fence in each of sixteen would write the L2 back sixteen times)
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tid == 0) __hip_atomic_store(report.word_at, report.word, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    };
    const int k = (int) g.k;
    // fast path: round r takes entry r of every side, provided no entry is already consumed by its pair
    const int per = k / NS;
    bool ok = (k % NS) == 0;
#pragma unroll
    for (int s = 0; s < NS; ++s) ok = ok && cnt[s] >= per;
    if (ok && tid < per) {
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            // the paired side has consumed `tid` entries before this pick if it runs later in the round,
            // `tid + 1` if it runs earlier
            const int consumed = s >= half ? tid + 1 : tid;
            if (pos_other[s] >= 0 && pos_other[s] < consumed) atomicOr(&conflict, 1);
        }
    }
    __syncthreads();
    if (ok && !conflict) {
        if (tid < per)
#pragma unroll
            for (int s = 0; s < NS; ++s) put(tid * NS + s, si[s]);
        tell();
        return;
    }
    // General path (the two ends of a pair of sides meet, or a side runs dry): the scan has a closed form.  Every side
    // makes one pick per round while it lasts, and takes its list from the front until the pair's first event: an entry that
    // the other side has taken, or the end of a list.  By then every instance that is in both lists has been taken
    // (those in front of the event's entry by one side, those behind it by the other), so from there on a side goes
    // on with the entries that are in its list alone.  What remains are prefix counts.  Replayed by one thread the scan took
    // 0.2 us per pick.
    // the turn of side s in round r is number 2 r + (is it a low side?) of its pair
    if (tid < half) event[tid] = 2 * cnt[tid] < 2 * cnt[tid + half] + 1 ? 2 * cnt[tid] : 2 * cnt[tid + half] + 1;
    __syncthreads();
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        const int po = pos_other[s], low = s < half ? 0 : 1;
        if (po >= 0 && po < tid + low) atomicMin(&event[s - low * half], 2 * tid + low);
    }
    __syncthreads();
    int first[NS], nth[NS];
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        first[s] = s < half ? (event[s] + 1) >> 1 : event[s - half] >> 1;   // picks before the event
        const bool alone = tid >= first[s] && tid < cnt[s] && pos_other[s] < 0;
        const uint64_t b = __ballot(alone);
        nth[s] = alone ? first[s] + __popcll(b & ((1ull << lane) - 1ull)) : -1;
        if (lane == 0) alone_in[s][wave] = __popcll(b);
    }
    __syncthreads();
    int len[NS], sum = 0;   // picks a side has to offer
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        int before = 0, total = 0;
        for (int v = 0; v < MAX_WS / 64; ++v) {
            if (v < wave) before += alone_in[s][v];
            total += alone_in[s][v];
        }
        nth[s] = tid < first[s] ? tid : nth[s] >= 0 ? nth[s] + before : -1;
        len[s] = first[s] + total;
        sum += len[s];
    }
#pragma unroll
    for (int s = 0; s < NS; ++s) {
        if (nth[s] < 0) continue;
        int at = 0;
#pragma unroll
        for (int o = 0; o < NS; ++o) at += (len[o] < nth[s] ? len[o] : nth[s]) + (o < s && len[o] > nth[s] ? 1 : 0);
        if (at < k) put(at, si[s]);
    }
    for (int t = sum + tid; t < k; t += MAX_WS) put(t, -1);
    tell();
}

// The ids a selection has just written, sent to the host by the device itself: host_ids is host memory the device
// can write (pinned, mapped); the ids go there (modulo fold_n when fold_n > 0) and then, behind a system-wide fence,
// `word` goes to host_ids[word_at], which the host polls.  One small kernel in stream order behind the selection,
// in place of a copy, an event and the wake-up of a thread that sleeps on it.
__global__ __launch_bounds__(256) void report_ids_kernel(const int *__restrict__ ids, int n_ids, int fold_n,
                                                         int *__restrict__ host_ids, int word_at, int word) {
    for (int t = threadIdx.x; t < n_ids; t += 256) {
        const int id = ids[t];
        host_ids[t] = fold_n > 0 && id >= 0 ? id % fold_n : id;
    }
    __threadfence_system();
    __syncthreads();
    if (threadIdx.x == 0) {
        __hip_atomic_store(&host_ids[word_at], word, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ------------------------------------------------------------------------------------------------
// C ABI
// ------------------------------------------------------------------------------------------------
template <typename TK, int COLS, int UNROLL, int NS>
static void launch_update_f(double *f, const double *alpha_diff, int ws_size, const void *k_rows, const int *slots,
                            int64_t ld, int64_t n, int repeat, const SelFuse &sf, hipStream_t s) {
    const int64_t vecs = (n + COLS - 1) / COLS;                        // column vectors, one per thread
    int64_t grid = (vecs + UF_T - 1) / UF_T;
    int vec_per_wg = UF_T;
    if (COLS > 1) {
        // (with one column per thread a workgroup's share has to start on a cache line, or every wavefront's
        // 256-byte read touches three lines instead of two: measured slower than the uneven grid)
        const int64_t per_cu = (vecs + 248 * UF_T - 1) / (248 * UF_T);   // workgroups per CU
        grid = 248 * per_cu;
        vec_per_wg = (int) ((vecs + grid - 1) / grid);
    }
    hipLaunchKernelGGL((update_f_kernel<TK, COLS, UNROLL, NS>), dim3((unsigned) grid), dim3(UF_T), 0, s, f, alpha_diff, ws_size,
                       (const TK *) k_rows, slots, ld, n, repeat, vec_per_wg, sf);
}

template <typename TK, int COLS, int R, int NS>
static void launch_update_f_narrow(double *f, const double *alpha_diff, int ws_size, const void *k_rows, const int *slots,
                                   int64_t ld, int64_t n, int repeat, const SelFuse &sf, hipStream_t s) {
    hipLaunchKernelGGL((update_f_narrow_kernel<TK, COLS, R, NS>), dim3((unsigned) ((n + 64 * COLS - 1) / (64 * COLS))), dim3(64 * UN_WAVES), 0, s,
                       f, alpha_diff, ws_size, (const TK *) k_rows, slots, ld, n, repeat, sf);
}

// The variant of the kernel for the row type, alignment and size at hand.
template <int NS>
static void dispatch_update_f(double *f, const double *alpha_diff, int ws_size, const void *k_rows, int row_type, const int *slots,
                              int64_t ld, int64_t n, int repeat, const SelFuse &sf, hipStream_t s) {
    // Vector loads need every row start aligned to the vector and the last vector inside the padded row.
    const size_t esz = row_type == TSVM_ROW_F32 ? 4 : 8;
    auto aligned = [&](int cols) { return (uintptr_t) k_rows % (cols * esz) == 0 && ld % cols == 0; };
    // Few columns: wavefronts that take the rows in turn, and on to 65,536 columns of floats with two columns per thread, to 32,768 of
    // doubles.  One column per thread up to 28,672 columns of floats, twice as many workgroups whose first pass of the selection then ends in
    // more atomics on the same addresses (with the selection, 516 rows, two columns / one: 20,000 43.2 / 39.5 us, 28,000
    // 44.5 / 41.8, 40,000 46.1 / 50.9), and up to 16,384 of doubles (20,000 44.4 / 45.7).  Of 2,048
    // rows in slots, us a call, one thread per column and all rows / wavefronts in turn (two columns per thread):
    //   non-zero rows     60          250          500         1,024
    //   floats  20,000   8.1 /  5.2  21.4 /  9.2  29.3 / 14.6   41.8 /  24.7   (one column per thread: 5.1, 8.6, 12.3, 18.5)
    //           65,536  15.6 /  6.9  24.9 / 15.1  34.1 / 24.6   50.0 /  44.7
    //          100,000  17.6 /  8.8  28.7 / 22.0  41.2 / 38.5   64.7 /  71.2   (here and below: four columns per thread)
    //          180,000  20.4 / 13.6  39.7 / 37.3  64.6 / 67.2  112.2 / 131.5
    //   doubles 20,000  10.2 /  6.2  23.0 / 10.5  35.5 / 16.4   62.5 /  28.4
    //           40,000  11.8 /  9.2  24.5 / 20.1  37.6 / 33.8   67.9 /  62.1
    //          100,000  15.3 / 17.2  38.5 / 41.2  67.7 / 72.4  132.1 / 137.9
    // Beyond the line rows in turn win alone where few rows are non-zero, and lose in training: calls with wavefronts in turn
    // everywhere / up to the line, ms: C-SVC 100,000 x 784 394.3 / 391.0, 200,000 x 30 483.7 / 468.0, 90,000 x 40 102.2 / 101.1,
    // epsilon-SVR 100,000 x 90 217.8 / 215.4, linear on 60,000 sparse rows 117.7 / 116.2; seven classes of 240,000 rows 596 / 584, means of
    // four calls of 574 to 608.
    const bool narrow = n <= (int64_t) 64 * 256 * (row_type == TSVM_ROW_F32 ? 4 : 2);
    if (narrow) {
        const bool one = n <= (row_type == TSVM_ROW_F32 ? 28672 : 16384) || !aligned(2);
        if (row_type == TSVM_ROW_F32) {
            if (one) launch_update_f_narrow<float, 1, 32, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
            else launch_update_f_narrow<float, 2, 16, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
        } else {
            if (one) launch_update_f_narrow<double, 1, 16, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
            else launch_update_f_narrow<double, 2, 16, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
        }
        return;
    }
    // 16-byte loads from 262,144 columns on; with fewer, one column per thread and more rows in flight keeps more of the chip busy
    const bool wide = n >= (int64_t) UF_T * 1024;
    if (row_type == TSVM_ROW_F32) {
        if (wide && aligned(4)) launch_update_f<float, 4, 8, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
        else launch_update_f<float, 1, 32, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
    } else {
        if (wide && aligned(2)) launch_update_f<double, 2, 8, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
        else launch_update_f<double, 1, 16, NS>(f, alpha_diff, ws_size, k_rows, slots, ld, n, repeat, sf, s);
    }
}

static SelGeom sel_geom(int64_t n, int n_select, int nu) {
    SelGeom g;
    g.n_sides = nu ? 4 : 2;
    int bits = 1;
    while (((int64_t) 1 << bits) < n) ++bits;
    g.idx_bits = bits;
    g.idx_mask = (uint32_t) (((uint64_t) 1 << bits) - 1);
    g.n_pass = 6 + (bits + SEL_DIGIT - 1) / SEL_DIGIT;
    g.k = (uint32_t) n_select;
    return g;
}

static SelWorkspace sel_workspace(void *workspace, int64_t n) {
    SelWorkspace w;
    sel_carve((void *) (((uintptr_t) workspace + 255) & ~(uintptr_t) 255), n, &w);
    return w;
}

// first_pass 1: digit 0 has been counted already, by update_f_kernel, on a workspace left by an earlier selection
static int select_working_set(const double *f, const int *y, const double *alpha, int64_t n, double Cp, double Cn,
                              const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace,
                              bool armed, int fold_n, int *out_folded, int first_pass, const SelReport &report, tsvm_stream stream,
                              bool guided = false) {
    TSVM_REQUIRE(f && y && alpha && out && workspace, "tsvm_select_working_set: null pointer");
    TSVM_REQUIRE(n >= 1 && n <= 0x7fffffffLL, "tsvm_select_working_set: n %lld outside [1, 2^31)", (long long) n);
    TSVM_REQUIRE(n_select >= 0 && n_select <= MAX_WS, "tsvm_select_working_set: n_select %d outside [0, %d]", n_select,
                 MAX_WS);
    TSVM_REQUIRE(n_marked >= 0 && (n_marked == 0 || marked), "tsvm_select_working_set: bad marked list");
    TSVM_REQUIRE(fold_n >= 0 && (fold_n == 0 || out_folded), "tsvm_select_working_set: bad fold arguments");
    hipStream_t s = tsvm_s(stream);
    if (n_select == 0) {   // (nothing to select, but whoever polls the word hears of it)
        if (report.ids) {
            hipLaunchKernelGGL(report_ids_kernel, dim3(1), dim3(256), 0, s, out, 0, 0, report.word_at, 0, report.word);
            TSVM_LAUNCH_CHECK();
        }
        return 0;
    }
    const SelWorkspace w = sel_workspace(workspace, n);
    const SelGeom g = sel_geom(n, n_select, nu);
    // The first three digits (33 bits of f) are counted by the whole chip, the rest (rarely needed) by one
    // workgroup.  Near convergence the free support vectors crowd within epsilon of the threshold, so the third
    // digit is usually the one that separates them.
    const int p_full = guided ? 0 : n > ((int64_t) 1 << 26) ? SEL_FULL_MAX : 3;   // < n_pass, which is at least 7
    // Every workgroup adds its histogram to the global one and asks for its candidates' places with atomics, on a few addresses that
    // most of them share, and with many workgroups those take longer than the counting they spread: four instances a thread, at
    // least 64 workgroups while there are instances for them, at most two per CU (n = 800k: 92 us per call with 1,024, 80 with 496).
    unsigned grid = (unsigned) std::min<int64_t>(std::max<int64_t>((n + SEL_T * SEL_EACH - 1) / (SEL_T * SEL_EACH),
                                                                  std::min<int64_t>((n + SEL_T - 1) / SEL_T, 64)), 496);
    if ((n + grid - 1) / grid > SEL_CHUNK_MAX) grid = (unsigned) ((n + SEL_CHUNK_MAX - 1) / SEL_CHUNK_MAX);
    if (!armed) {
        hipLaunchKernelGGL(sel_init_kernel, dim3(p_full * SEL_MAX_SIDES * SEL_BINS / 1024), dim3(256), 0, s, w, p_full);
        TSVM_LAUNCH_CHECK();
    }
    for (int p = first_pass; p < p_full; ++p) {
        if (nu) hipLaunchKernelGGL(sel_pass_kernel<4>, dim3(grid), dim3(SEL_T), 0, s, w, f, y, alpha, n, Cp, Cn, g, p, marked, n_marked);
        else hipLaunchKernelGGL(sel_pass_kernel<2>, dim3(grid), dim3(SEL_T), 0, s, w, f, y, alpha, n, Cp, Cn, g, p, marked, n_marked);
        TSVM_LAUNCH_CHECK();
    }
    if (guided && nu) hipLaunchKernelGGL((sel_compact_kernel<4, true>), dim3(grid), dim3(SEL_T), 0, s, w, n, g, p_full);
    else if (guided) hipLaunchKernelGGL((sel_compact_kernel<2, true>), dim3(grid), dim3(SEL_T), 0, s, w, n, g, p_full);
    else if (nu) hipLaunchKernelGGL((sel_compact_kernel<4, false>), dim3(grid), dim3(SEL_T), 0, s, w, n, g, p_full);
    else hipLaunchKernelGGL((sel_compact_kernel<2, false>), dim3(grid), dim3(SEL_T), 0, s, w, n, g, p_full);
    TSVM_LAUNCH_CHECK();
    if (nu) hipLaunchKernelGGL(sel_final_kernel<4>, dim3(4 * MAX_WS / SEL_RANK_ENTRIES), dim3(SEL_RANK_T), 0, s, w, n, g, p_full, out, fold_n, out_folded, report, guided);
    else hipLaunchKernelGGL(sel_final_kernel<2>, dim3(2 * MAX_WS / SEL_RANK_ENTRIES), dim3(SEL_RANK_T), 0, s, w, n, g, p_full, out, fold_n, out_folded, report, guided);
    TSVM_LAUNCH_CHECK();
    return 0;
}

static int sel_report(const char *who, int *host_ids, int word_at, int word, int n_select, SelReport *report) {
    TSVM_REQUIRE(host_ids, "%s: null pointer", who);
    TSVM_REQUIRE(word_at >= n_select, "%s: the word at %d among the %d ids", who, word_at, n_select);
    report->ids = host_ids;
    report->word_at = host_ids + word_at;
    report->word = word;
    return 0;
}

static int update_f_select(double *f, const double *alpha_diff, int ws_size, const void *k_rows, int row_type, const int *slots,
                           int64_t ld, int64_t n_cols, int repeat, const int *y, const double *alpha, double Cp, double Cn,
                           const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace, int *out_folded,
                           const SelReport &report, tsvm_stream stream, bool guided = false) {
    TSVM_REQUIRE(f && alpha_diff && k_rows, "tsvm_update_f_select: null pointer");
    TSVM_REQUIRE(ws_size >= 0 && n_cols >= 1 && ld >= n_cols && repeat >= 1 && repeat <= UF_MAX_REPEAT,
                 "tsvm_update_f_select: bad size (ws=%d n=%lld ld=%lld repeat=%d)", ws_size, (long long) n_cols, (long long) ld, repeat);
    TSVM_REQUIRE(row_type == TSVM_ROW_F64 || row_type == TSVM_ROW_F32, "tsvm_update_f_select: unknown row type %d", row_type);
    TSVM_REQUIRE(y && alpha && out && workspace, "tsvm_update_f_select: null pointer");
    TSVM_REQUIRE(n_select >= 1 && n_select <= MAX_WS, "tsvm_update_f_select: n_select %d outside [1, %d]", n_select, MAX_WS);
    TSVM_REQUIRE(n_marked >= 0 && (n_marked == 0 || marked), "tsvm_update_f_select: bad marked list");
    const int64_t n = n_cols * repeat;
    TSVM_REQUIRE(n <= 0x7fffffffLL, "tsvm_update_f_select: %lld instances, at most 2^31 - 1", (long long) n);
    SelFuse sf;
    sf.w = sel_workspace(workspace, n);
    sf.g = sel_geom(n, n_select, nu);
    sf.y = y; sf.alpha = alpha; sf.Cp = Cp; sf.Cn = Cn; sf.marked = marked; sf.n_marked = n_marked; sf.guided = guided;
    hipStream_t s = tsvm_s(stream);
    if (nu) dispatch_update_f<4>(f, alpha_diff, ws_size, k_rows, row_type, slots, ld, n_cols, repeat, sf, s);
    else dispatch_update_f<2>(f, alpha_diff, ws_size, k_rows, row_type, slots, ld, n_cols, repeat, sf, s);
    TSVM_LAUNCH_CHECK();
    return select_working_set(f, y, alpha, n, Cp, Cn, marked, n_marked, out, n_select, nu, workspace, true,
                              out_folded ? (int) n_cols : 0, out_folded, guided ? 0 : 1, report, stream, guided);
}

extern "C" {

int tsvm_update_f(double *f, const double *alpha_diff, int ws_size, const void *k_rows, int row_type, const int *slots,
                  int64_t ld, int64_t n_cols, int repeat, tsvm_stream stream) {
    TSVM_REQUIRE(f && alpha_diff && k_rows, "tsvm_update_f: null pointer");
    TSVM_REQUIRE(ws_size >= 0 && n_cols >= 0 && ld >= n_cols && repeat >= 1, "tsvm_update_f: bad size (ws=%d n=%lld ld=%lld)",
                 ws_size, (long long) n_cols, (long long) ld);
    TSVM_REQUIRE(row_type == TSVM_ROW_F64 || row_type == TSVM_ROW_F32, "tsvm_update_f: unknown row type %d", row_type);
    if (n_cols == 0 || ws_size == 0) return 0;
    dispatch_update_f<0>(f, alpha_diff, ws_size, k_rows, row_type, slots, ld, n_cols, repeat, SelFuse(), tsvm_s(stream));
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_update_f_batches(double *f, const double *coef, int n_rows, int batch, const void *k_rows, int row_type, int64_t ld,
                          int64_t n_cols, int repeat, tsvm_stream stream) {
    TSVM_REQUIRE(f && coef && k_rows, "tsvm_update_f_batches: null pointer");
    TSVM_REQUIRE(n_rows >= 0 && batch >= 1 && n_cols >= 0 && ld >= n_cols && repeat >= 1, "tsvm_update_f_batches: bad size (rows=%d batch=%d n=%lld ld=%lld)",
                 n_rows, batch, (long long) n_cols, (long long) ld);
    TSVM_REQUIRE(row_type == TSVM_ROW_F64 || row_type == TSVM_ROW_F32, "tsvm_update_f_batches: unknown row type %d", row_type);
    TSVM_REQUIRE((n_cols + 63) / 64 <= 0x7fffffffLL, "tsvm_update_f_batches: %lld columns", (long long) n_cols);
    if (n_cols == 0 || n_rows == 0) return 0;
    const dim3 grid((unsigned) ((n_cols + 63) / 64));
    if (row_type == TSVM_ROW_F32)
        hipLaunchKernelGGL(update_f_batches_kernel<float>, grid, dim3(64), 0, tsvm_s(stream), f, coef, n_rows, batch, (const float *) k_rows, ld, n_cols, repeat);
    else
        hipLaunchKernelGGL(update_f_batches_kernel<double>, grid, dim3(64), 0, tsvm_s(stream), f, coef, n_rows, batch, (const double *) k_rows, ld, n_cols, repeat);
    TSVM_LAUNCH_CHECK();
    return 0;
}

int tsvm_update_f_select(double *f, const double *alpha_diff, int ws_size, const void *k_rows, int row_type, const int *slots,
                         int64_t ld, int64_t n_cols, int repeat, const int *y, const double *alpha, double Cp, double Cn,
                         const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace, int *out_folded,
                         tsvm_stream stream) {
    return update_f_select(f, alpha_diff, ws_size, k_rows, row_type, slots, ld, n_cols, repeat, y, alpha, Cp, Cn, marked, n_marked, out,
                           n_select, nu, workspace, out_folded, SelReport(), stream);
}

int tsvm_update_f_select_report(double *f, const double *alpha_diff, int ws_size, const void *k_rows, int row_type, const int *slots,
                                int64_t ld, int64_t n_cols, int repeat, const int *y, const double *alpha, double Cp, double Cn,
                                const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace, int *out_folded,
                                int *host_ids, int word_at, int word, tsvm_stream stream) {
    SelReport report;
    if (const int rc = sel_report("tsvm_update_f_select_report", host_ids, word_at, word, n_select, &report)) return rc;
    return update_f_select(f, alpha_diff, ws_size, k_rows, row_type, slots, ld, n_cols, repeat, y, alpha, Cp, Cn, marked, n_marked, out,
                           n_select, nu, workspace, out_folded, report, stream);
}

int tsvm_update_f_select_guided(double *f, const double *alpha_diff, int ws_size, const void *k_rows, int row_type, const int *slots,
                                int64_t ld, int64_t n_cols, int repeat, const int *y, const double *alpha, double Cp, double Cn,
                                const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace, int *out_folded,
                                int *host_ids, int word_at, int word, int *missed, tsvm_stream stream) {
    TSVM_REQUIRE(missed, "tsvm_update_f_select_guided: null pointer");
    SelReport report;
    if (host_ids)
        if (const int rc = sel_report("tsvm_update_f_select_guided", host_ids, word_at, word, n_select, &report)) return rc;
    report.missed = missed;
    return update_f_select(f, alpha_diff, ws_size, k_rows, row_type, slots, ld, n_cols, repeat, y, alpha, Cp, Cn, marked, n_marked, out,
                           n_select, nu, workspace, out_folded, report, stream, true);
}

int tsvm_report_ids(const int *ids, int n_ids, int fold_n, int *host_ids, int word_at, int word, tsvm_stream stream) {
    TSVM_REQUIRE(ids && host_ids, "tsvm_report_ids: null pointer");
    TSVM_REQUIRE(n_ids >= 0 && n_ids <= MAX_WS && word_at >= n_ids && fold_n >= 0, "tsvm_report_ids: bad size (n_ids=%d word_at=%d fold_n=%d)",
                 n_ids, word_at, fold_n);
    hipLaunchKernelGGL(report_ids_kernel, dim3(1), dim3(256), 0, tsvm_s(stream), ids, n_ids, fold_n, host_ids, word_at, word);
    TSVM_LAUNCH_CHECK();
    return 0;
}

size_t tsvm_select_workspace(int64_t n) {
    if (n < 0) return 0;
    return sel_carve(nullptr, n, nullptr) + 256;
}

int tsvm_select_working_set(const double *f, const int *y, const double *alpha, int64_t n, double Cp, double Cn,
                            const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace,
                            tsvm_stream stream) {
    return select_working_set(f, y, alpha, n, Cp, Cn, marked, n_marked, out, n_select, nu, workspace, false, 0, nullptr, 0, SelReport(), stream);
}

int tsvm_select_working_set_again(const double *f, const int *y, const double *alpha, int64_t n, double Cp, double Cn,
                                  const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace,
                                  tsvm_stream stream) {
    return select_working_set(f, y, alpha, n, Cp, Cn, marked, n_marked, out, n_select, nu, workspace, true, 0, nullptr, 0, SelReport(), stream);
}

int tsvm_select_working_set_folded(const double *f, const int *y, const double *alpha, int64_t n, double Cp, double Cn,
                                   const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace,
                                   int again, int fold_n, int *out_folded, tsvm_stream stream) {
    TSVM_REQUIRE(fold_n >= 1, "tsvm_select_working_set_folded: fold_n %d < 1", fold_n);
    return select_working_set(f, y, alpha, n, Cp, Cn, marked, n_marked, out, n_select, nu, workspace, again != 0, fold_n, out_folded,
                              0, SelReport(), stream);
}

int tsvm_select_working_set_report(const double *f, const int *y, const double *alpha, int64_t n, double Cp, double Cn,
                                   const int *marked, int n_marked, int *out, int n_select, int nu, void *workspace,
                                   int again, int fold_n, int *out_folded, int *host_ids, int word_at, int word, tsvm_stream stream) {
    SelReport report;
    if (const int rc = sel_report("tsvm_select_working_set_report", host_ids, word_at, word, n_select, &report)) return rc;
    return select_working_set(f, y, alpha, n, Cp, Cn, marked, n_marked, out, n_select, nu, workspace, again != 0, fold_n, out_folded,
                              0, report, stream);
}

}  // extern "C"
