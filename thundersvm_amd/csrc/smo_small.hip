// Whole SMO solves of small problems: CSMOSolver::solve / NuSMOSolver::solve (src/thundersvm/solver/csmosolver.cpp:10-121,
// nusmosolver.cpp) with everything between the kernel matrix and the solution in one kernel, one workgroup per problem
// and as many problems as there are in one launch (the class pairs of a one-vs-one run).
//
// Why.  A problem of a few hundred instances needs some ten outer iterations of some fifty steps.  As a chain of launches
// (selection, rows, block, solver, update) an outer iteration took 150 us of which the solver's steps were 50, each
// problem another 600 us of set-up, and one host thread fed all pairs.  Here an outer iteration's selection is a sort in LDS
// of some microseconds, the kernel matrix is computed once for all pairs (it holds every pair's rows and columns), the host
// takes no part between the upload and the result, and the pairs run side by side.  Whole
// training calls: 45 pairs of 360 instances in 64 columns 31 -> 1.1 ms, 3 pairs of 100 in 4 columns 2.4 -> 0.35 ms.
//
// Shape.  At most 1,024 instances (above that a workgroup's share of update_f and of the selection outlasts what the
// chip-wide kernels take, and their launches no longer matter): W wavefronts of E neighbouring instances per thread.
// f, the local solver's f and the sets' membership live in registers, alpha in LDS.  The local solver runs on the
// instances where they are, not on a gathered working set: an instance outside the working set is in neither I_up nor I_low, a row is
// read from the kernel matrix in one piece, and ties go to the instance that comes first in the working set.
#include "../../include/thundersvm_amd.h"
#include "smo_local.h"
#include "tsvm_internal.h"

#define SS_MAX 1024            // instances of a problem (padded) at most
#define SS_MAX_ITER 256        // outer iterations per launch: the host launches again what is not finished
#define SS_MAX_INNER 300000    // and local steps per launch after which no outer iteration is begun

__device__ __forceinline__ int wave_min_i32(int v) {
    v = imin_sel(v, dpp_i32<TSVM_DPP_XOR1>(v));
    v = imin_sel(v, dpp_i32<TSVM_DPP_XOR2>(v));
    v = imin_sel(v, dpp_i32<TSVM_DPP_HALF_MIRROR>(v));
    v = imin_sel(v, dpp_i32<TSVM_DPP_MIRROR>(v));
    v = imin_sel(v, dpp_i32<TSVM_DPP_BCAST15, 0xa>(v));
    v = imin_sel(v, dpp_i32<TSVM_DPP_BCAST31, 0xc>(v));
    return __builtin_amdgcn_readlane(v, 63);
}

// As wave_first_argmin (smo_local.h), but among equal values the element that comes first in the working set wins.
// Equal values are rare once the first steps have told the instances apart: they are looked for (scalar work beside the
// reduction) and only then are the positions read.
template <int E>
__device__ __forceinline__ int wave_argmin_by_pos(const double (&x)[E], const unsigned short *pos, int tid, double &value, double &m, int &at) {
    uint64_t twice;
    int win = wave_argmin<E, true>(x, tid * E, value, m, at, twice);
    uint64_t who = __builtin_amdgcn_ballot_w64(m == value);
    if (__builtin_expect(((who & (who - 1)) | (who & twice)) != 0, 0)) {
        int key = 0x7fffffff;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int k = (int) pos[tid * E + e] << 10 | e;
            key = x[e] == value ? imin_sel(key, k) : key;
        }
        const int first = wave_min_i32(key);
        who = __builtin_amdgcn_ballot_w64(key == first && m == value);
        win = __builtin_ctzll(who);
        at = tid * E + (key & (E - 1));
    }
    return win;
}

template <int W>
__device__ __forceinline__ void block_argmin_by_pos(const SvCand *slots, const unsigned short *pos, int lane, double &v, int &at, int &flags) {
    static_assert(W == 2 || W == 4, "quad_perm steps");
    const SvCand c = slots[lane & (W - 1)];
    double m = fmin_f64(c.v, dpp_f64<TSVM_DPP_XOR1>(c.v));
    if (W == 4) m = fmin_f64(m, dpp_f64<TSVM_DPP_XOR2>(m));
    v = m;
    uint64_t who = __builtin_amdgcn_ballot_w64(c.v == m);
    if (__builtin_expect((who & (who - 1) & ((1 << W) - 1)) != 0, 0)) {   // (every quad holds the same W)
        int k = c.v == m ? (int) pos[c.at] : 0x7fffffff;
        const int mine = k;
        k = imin_sel(k, dpp_i32<TSVM_DPP_XOR1>(k));
        k = imin_sel(k, dpp_i32<TSVM_DPP_XOR2>(k));
        who = __builtin_amdgcn_ballot_w64(mine == k && c.v == m);
    }
    at = __builtin_amdgcn_readlane(c.at, __builtin_ctzll(who));
    flags = __builtin_amdgcn_ballot_w64(c.flag != 0) != 0;
}

__device__ __forceinline__ uint64_t ss_key(double f) {   // order-preserving; -0 and +0 compare equal in the reference's sort
    if (f == 0.0) f = 0.0;
    const uint64_t u = (uint64_t) __double_as_longlong(f);
    return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}

template <int E, int W>
struct SmallShared {
    static constexpr int N = 64 * E * W;
    double kd[N];
    double z[W][N];                     // alpha times its label (SvBound): one copy per wavefront (smo_solve.hip)
    double f[N], k[N];                  // local solver: f and the row at the candidates; selection: keys and slots on their way between wavefronts; update: coefficients and rows
    unsigned short pos[N];              // position of a slot in the working set, 0xffff outside it
    unsigned short ws[N];
    unsigned char flags[N];             // selection: the sides an instance is a candidate of
    uint64_t total[2][W];               // per-wavefront counts of a scan
    double red[4][W];
    int event[2], first_x[2], first_y[2], n_list;
    SvCand ci[4 * W], ci2[W], cj[W], cj2[W];
    SvScoreStep score[4 * W];
};

// sort_f + select_working_set (smo_kernel.cpp:321-332, csmosolver.cpp:123-165, nusmosolver.cpp:48-118): writes k picks to
// sh.ws[base ...]; false when there are fewer candidates.
//
// After the sort the alternating scan has a closed form.  Take one pair of sides, `up` reading the order from the low
// end and `low` from the high end, one pick per round each (up first).  Nothing is skipped until the first event: a side
// whose next candidate the other has already taken, or a side that is used up.  At that moment every instance that is
// a candidate of both sides has been taken by one of them (the two ends have met), so from then on each side goes on with
// the candidates that are its own alone.  The event is the minimum of a round number over the instances, and what remains are
// prefix counts.
// The value of lane ^ D.
template <int D>
__device__ __forceinline__ int lane_xor(int v, int lane) {
    if constexpr (D == 1) return dpp_i32<TSVM_DPP_XOR1>(v);
    else if constexpr (D == 2) return dpp_i32<TSVM_DPP_XOR2>(v);
    else if constexpr (D == 4) return dpp_i32<TSVM_DPP_HALF_MIRROR>(dpp_i32<0x1B>(v));   // quad_perm [3,2,1,0]: ^ 3, then ^ 7
    else if constexpr (D == 8) return dpp_i32<0x128>(v);                                 // row_ror:8
    else return __builtin_amdgcn_ds_bpermute((lane ^ D) << 2, v);
}

// One step of the sort at a fixed stride: entry i against entry i ^ STRD, ascending where i & size is zero.
template <int E, int W, int STRD>
__device__ __forceinline__ void ss_sort_step(SmallShared<E, W> &sh, uint64_t (&key)[E], int (&slot)[E], int size) {
    const int tid = threadIdx.x, lane = tid & 63;
    auto less = [](uint64_t ka, int ia, uint64_t kb, int ib) { return (ka < kb) | ((ka == kb) & (ia < ib)); };
    if constexpr (STRD < E) {
#pragma unroll
        for (int e = 0; e < E; ++e) {
            if (e & STRD) continue;
            const int o = e | STRD;
            const bool asc = ((tid * E + e) & size) == 0;
            const bool swap = less(key[o], slot[o], key[e], slot[e]) == asc;
            const uint64_t ke = swap ? key[o] : key[e], ko = swap ? key[e] : key[o];
            const int se = swap ? slot[o] : slot[e], so = swap ? slot[e] : slot[o];
            key[e] = ke; key[o] = ko;
            slot[e] = se; slot[o] = so;
        }
    } else {
        const bool want_less = ((tid * E & STRD) == 0) == ((tid * E & size) == 0);
        uint64_t ok[E];
        int os[E];
        if constexpr (STRD >= 64 * E) {
            uint64_t *const xk = (uint64_t *) sh.f;
            int *const xs = (int *) sh.k;
#pragma unroll
            for (int e = 0; e < E; ++e) { xk[e * 64 * W + tid] = key[e]; xs[e * 64 * W + tid] = slot[e]; }
            __syncthreads();
            const int other = tid ^ (STRD / E);
#pragma unroll
            for (int e = 0; e < E; ++e) { ok[e] = xk[e * 64 * W + other]; os[e] = xs[e * 64 * W + other]; }
            __syncthreads();
        } else {
            constexpr int D = STRD / E;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const unsigned lo = (unsigned) lane_xor<D>((int) (uint32_t) key[e], lane), hi = (unsigned) lane_xor<D>((int) (uint32_t) (key[e] >> 32), lane);
                ok[e] = (uint64_t) hi << 32 | lo;
                os[e] = lane_xor<D>(slot[e], lane);
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const bool take = less(ok[e], os[e], key[e], slot[e]) == want_less;
            key[e] = take ? ok[e] : key[e];
            slot[e] = take ? os[e] : slot[e];
        }
    }
}

// A bitonic sort of E neighbouring entries per thread in registers: strides below E inside a thread, below 64 * E between
// the lanes of a wavefront (below 16 * E without the LDS's crossbar, which four wavefronts would queue for), the others through LDS.
template <int E, int W, int STRD>
__device__ __forceinline__ void ss_merge(SmallShared<E, W> &sh, uint64_t (&key)[E], int (&slot)[E], int size) {
    if constexpr (STRD > 0) {
        if (STRD < size) ss_sort_step<E, W, STRD>(sh, key, slot, size);
        ss_merge<E, W, STRD / 2>(sh, key, slot, size);
    }
}

template <int E, int W, bool NU>
__device__ bool ss_select(SmallShared<E, W> &sh, const double (&f)[E], const bool (&act)[E], int k, int base) {
    constexpr int NP = NU ? 2 : 1;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint64_t key[E];
    int slot[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        key[e] = act[e] ? ss_key(f[e]) : ~0ull;
        slot[e] = tid * E + e;
    }
#pragma unroll 1
    for (int size = 2; size <= 64 * E * W; size <<= 1) ss_merge<E, W, 32 * E * W>(sh, key, slot, size);
    unsigned fl[E];
#pragma unroll
    for (int j = 0; j < E; ++j) fl[j] = sh.flags[slot[j]];
    // counts of up, low, up alone, low alone in 16-bit fields; inclusive scan over the sorted order
    uint64_t incl[NP][E], total[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        uint64_t run = 0;
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const unsigned u = (fl[j] >> q) & 1u, l = (fl[j] >> (q + NP)) & 1u;
            run += (uint64_t) u | (uint64_t) l << 16 | (uint64_t) (u & ~l & 1u) << 32 | (uint64_t) (l & ~u & 1u) << 48;
            incl[q][j] = run;
        }
        uint64_t scan = run;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint64_t o = __shfl_up((unsigned long long) scan, d, 64);
            if (lane >= d) scan += o;
        }
        if (lane == 63) sh.total[q][wave] = scan;
#pragma unroll
        for (int j = 0; j < E; ++j) incl[q][j] += scan - run;
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        uint64_t before = 0;
        total[q] = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const uint64_t t = sh.total[q][w];
            if (w < wave) before += t;
            total[q] += t;
        }
#pragma unroll
        for (int j = 0; j < E; ++j) incl[q][j] += before;
        if (tid == 0) {
            const int n_up = (int) (total[q] & 0xffff), n_low = (int) (total[q] >> 16 & 0xffff);
            const int dry_up = 2 * n_up, dry_low = 2 * n_low + 1;
            sh.event[q] = dry_up < dry_low ? dry_up : dry_low;
            sh.first_x[q] = (int) (total[q] >> 32 & 0xffff);
            sh.first_y[q] = (int) (total[q] >> 48);
        }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
        for (int j = 0; j < E; ++j) {
            if (!((fl[j] >> q) & (fl[j] >> (q + NP)) & 1u)) continue;
            const int ru = (int) (incl[q][j] & 0xffff) - 1, rl = (int) (total[q] >> 16 & 0xffff) - (int) (incl[q][j] >> 16 & 0xffff);
            atomicMin(&sh.event[q], ru <= rl ? 2 * rl + 1 : 2 * ru);   // the round in which the other side finds it taken
        }
    __syncthreads();
    int a0[NP], b0[NP];
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        b0[q] = sh.event[q] >> 1;
        a0[q] = b0[q] + (sh.event[q] & 1);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const unsigned u = (fl[j] >> q) & 1u, l = (fl[j] >> (q + NP)) & 1u;
            const int ru = (int) (incl[q][j] & 0xffff) - 1, rl = (int) (total[q] >> 16 & 0xffff) - (int) (incl[q][j] >> 16 & 0xffff);
            if (u && ru == a0[q]) sh.first_x[q] = (int) (incl[q][j] >> 32 & 0xffff) - (int) (u & ~l & 1u);
            if (l && rl == b0[q]) sh.first_y[q] = (int) (total[q] >> 48) - (int) (incl[q][j] >> 48);
        }
    }
    __syncthreads();
    int len[2 * NP], sum = 0;
#pragma unroll
    for (int q = 0; q < NP; ++q) {
        len[q] = a0[q] + (int) (total[q] >> 32 & 0xffff) - sh.first_x[q];
        len[q + NP] = b0[q] + (int) (total[q] >> 48) - sh.first_y[q];
        sum += len[q] + len[q + NP];
    }
    auto place = [&](int side, int nth, int s) {   // the nth pick of a side: one pick per side and round while the sides last
        int at = 0;
#pragma unroll
        for (int o = 0; o < 2 * NP; ++o) at += (len[o] < nth ? len[o] : nth) + (o < side && len[o] > nth ? 1 : 0);
        if (at < k) sh.ws[base + at] = (unsigned short) s;
    };
#pragma unroll
    for (int q = 0; q < NP; ++q)
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const unsigned u = (fl[j] >> q) & 1u, l = (fl[j] >> (q + NP)) & 1u;
            const int ru = (int) (incl[q][j] & 0xffff) - 1, rl = (int) (total[q] >> 16 & 0xffff) - (int) (incl[q][j] >> 16 & 0xffff);
            if (u) {
                if (ru < a0[q]) place(q, ru, slot[j]);
                else if (!l) place(q, a0[q] + (int) (incl[q][j] >> 32 & 0xffff) - 1 - sh.first_x[q], slot[j]);
            }
            if (l) {
                if (rl < b0[q]) place(q + NP, rl, slot[j]);
                else if (!u) place(q + NP, b0[q] + (int) (total[q] >> 48) - (int) (incl[q][j] >> 48) - sh.first_y[q], slot[j]);
            }
        }
    __syncthreads();
    return sum >= k;
}

// Slot s of a problem: its y > 0 instances first, then from a multiple of four on the others, so that a thread's four
// slots have one label.  In the kernel matrix either group is a run of rows and (the same) columns.
struct SmallMap {
    int n0, n1, n0p, col0, col1, n_rows;
    __device__ __forceinline__ int row(int s) const {
        const int r = s < n0p ? col0 + s : col1 + (s - n0p);
        return r < n_rows ? r : n_rows - 1;   // (an inactive slot's: in range, never used)
    }
    __device__ __forceinline__ bool active(int s) const { return s < n0p ? s < n0 : s - n0p < n1; }
    __device__ __forceinline__ int index(int s) const { return s < n0p ? s : n0 + (s - n0p); }
    __device__ __forceinline__ double label(int s) const { return s < n0p ? 1.0 : -1.0; }
    __device__ __forceinline__ SvBound bound(int s, double Cp, double Cn) const { return s < n0p ? SvBound{Cp, 0.0} : SvBound{0.0, -Cn}; }
};

// A pointer to memory, not to memory or LDS: a problem's pointers come out of memory themselves, so that the compiler would
// read through them by flat loads, and every wait for the LDS would be one for them, too.  Cross-validation of 1203x13 in five
// folds: 2.36 -> 2.31 ms.
#define SS_GLOBAL(T) const T __attribute__((address_space(1)))

template <int E, typename TB>
__device__ __forceinline__ void ss_load(SS_GLOBAL(TB) *row, TB (&out)[E]) {
    if constexpr (E == 1) {
        out[0] = *row;
    } else {
        typedef TB vec_t __attribute__((ext_vector_type(E), aligned(sizeof(TB))));   // (a class's columns start anywhere)
        const vec_t v = *(SS_GLOBAL(vec_t) *) row;
#pragma unroll
        for (int e = 0; e < E; ++e) out[e] = v[e];
    }
}

// The local solver: c_smo_iterate of smo_solve.hip (and nu_smo_solve_kernel) with the instances in place of a gathered
// working set.  Takes up to `left` steps (ALL: as many as there are), counted in n_iter; returns whether the solve has ended.  The new alpha is in sh.z.
// NONE and no_score: as there.
template <int E, int W, bool NU, bool NONE, bool ALL, typename TB>
__device__ __forceinline__ bool ss_local(SmallShared<E, W> &sh, const SmallMap &map, SS_GLOBAL(TB) *K, int64_t ld, int col, const double (&kd)[E], double (&f)[E],
                        unsigned &member, double Cp, double Cn, double local_eps, int max_iter, bool &no_score, int &n_iter, int left) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int NP = NU ? 2 : 1;   // pairs of sides
    SvCand *const ci[2] = {sh.ci, sh.ci2}, *const cj[2] = {sh.cj, sh.cj2};
    const int first_slot = sh.ws[0];
    bool go_on;
    double taken = -__builtin_inf();   // the score of the step
    int worst = 0;
    do {
        if (!NONE) worst = imax_sel(worst, __double2hiint(taken));
        double up[NP], m[NP], v;
        int at[NP], is[NP], go;
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            double fu[E];
#pragma unroll
            for (int e = 0; e < E; ++e) fu[e] = keep_or_none<0>(member << (31 - 2 * NP * e - q), f[e]);
            const int win = wave_argmin_by_pos<E>(fu, sh.pos, tid, up[q], m[q], at[q]);
            if constexpr (W > 1) publish(ci[q] + wave, 1ull << win, m[q], at[q], 0);
            else is[q] = __builtin_amdgcn_readlane(at[q], win);
        }
        if constexpr (W > 1) {
            lds_barrier();
#pragma unroll
            for (int q = 0; q < NP; ++q) block_argmin_by_pos<W>(ci[q], sh.pos, lane, up[q], is[q], go);
        }
        TB kI[NP][E];
        double kd_i[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            is[q] &= 64 * E * W - 1;   // (with only NaN left there is no candidate at all)
            if (NU) is[q] = is_none(up[q]) ? first_slot : is[q];   // (its row enters the other side's scores, smo_kernel.cpp:239)
            ss_load<E, TB>(K + (unsigned) map.row(is[q]) * (unsigned) ld + col, kI[q]);
            kd_i[q] = sh.kd[is[q]];
        }
        SV_PIN_MEMORY;
        double part[E], b[NP][E], b_max = -__builtin_inf();
#pragma unroll
        for (int e = 0; e < E; ++e) {
            part[e] = kd_i[0] + kd[e];
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                b[q][e] = keep_or_none<1>(member << (31 - 2 * NP * e - NP - q), -up[q] + f[e]);
                b_max = fmax_f64(b_max, b[q][e]);
            }
        }
        go = __builtin_amdgcn_ballot_w64(!(b_max < local_eps)) != 0;
        SV_PIN;
        double best[NP];
        int js[NP];
#pragma unroll
        for (int q = 0; q < NP; ++q) {
            double qs[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const double aIJ = __builtin_fma(-2.0, (double) kI[0][e], part[e]);
                const double s = -b[q][e] * b[q][e] / aIJ;
                qs[e] = __hiloint2double(b[q][e] > 0.0 ? __double2hiint(s) : SV_NONE_HI, __double2loint(s));
            }
            const int win = wave_argmin_by_pos<E>(qs, sh.pos, tid, best[q], v, at[q]);
            publish_row<E, TB>(sh.f + tid * E, sh.k + tid * E, 1ull << win, f, kI[q]);
            if constexpr (W > 1) publish(cj[q] + wave, 1ull << win, v, at[q], go);
            else js[q] = __builtin_amdgcn_readlane(at[q], win);
        }
        if constexpr (W > 1) {
            lds_barrier();
#pragma unroll
            for (int q = 0; q < NP; ++q) {
                int g;
                block_argmin_by_pos<W>(cj[q], sh.pos, lane, best[q], js[q], g);
                if (q == 0) go = g;
            }
        }
        const bool second = NU && !__builtin_amdgcn_readfirstlane(best[0] < best[NP - 1] && best[0] < SV_NONE ? 1 : 0);
        const int i = second ? is[NP - 1] : is[0];
        int j2 = (second ? js[NP - 1] : js[0]) & (64 * E * W - 1);
        const double up_value = second ? up[NP - 1] : up[0], kd_i2 = second ? kd_i[NP - 1] : kd_i[0];
        // (two sides' winners may write different rows into one lane's slots when one of them has no candidate, so with
        // two sides K[i, j2] is read from the matrix)
        taken = second ? best[NP - 1] : best[0];
        if (NONE && is_none(taken)) {
            j2 = first_slot;
            __syncthreads();
            if (tid == first_slot / E) {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    sh.f[tid * E + e] = f[e];
                    *(TB *) (sh.k + tid * E + e) = second ? kI[NP - 1][e] : kI[0][e];
                }
            }
            __syncthreads();
        }
        TB kJ[E];
        ss_load<E, TB>(K + (unsigned) map.row(j2) * (unsigned) ld + col, kJ);
        const TB k_ij = NU ? K[(unsigned) map.row(i) * (unsigned) ld + map.row(j2)] : *(const TB *) (sh.k + j2);
        SV_PIN_MEMORY;
        const double kd_j = sh.kd[j2], z_j = sh.z[wave][j2], z_i = sh.z[wave][i], f_j = sh.f[j2];
        const SvBound bound_i = map.bound(i, Cp, Cn), bound_j = map.bound(j2, Cp, Cn);
        SV_PIN;
        go_on = go && !(n_iter > max_iter);
        const double q2 = (-up_value + f_j) / __builtin_fma(-2.0, (double) k_ij, kd_i2 + kd_j);
        const double l = fmin_f64(bound_i.hi - z_i, fmin_f64(z_j - bound_j.lo, q2));
        const double nz_i = z_i + l, nz_j = (j2 == i ? nz_i : z_j) - l;
        // (nu-SVC of 600 rows 1.41 -> 1.37 ms a call, against a shifted field, a comparison and a selection for each)
        const unsigned up_bit_i = own_bit<E, 2 * NP>(tid, i) << (NU && i >= map.n0p ? 1 : 0), up_bit_j = own_bit<E, 2 * NP>(tid, j2) << (NU && j2 >= map.n0p ? 1 : 0);
        const unsigned up_i_on = same_in_all_lanes(nz_i < bound_i.hi), low_i_on = same_in_all_lanes(nz_i > bound_i.lo);
        const unsigned up_j_on = same_in_all_lanes(nz_j < bound_j.hi), low_j_on = same_in_all_lanes(nz_j > bound_j.lo);
        member = put_bits(put_bits(member, up_bit_i, up_i_on), up_bit_i << NP, low_i_on);
        member = put_bits(put_bits(member, up_bit_j, up_j_on), up_bit_j << NP, low_j_on);
        write_by_lane0(go_on, &sh.z[wave][i], nz_i, &sh.z[wave][j2], nz_j);
        SV_PIN;
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = __builtin_fma(-l, (double) kJ[e] - (double) (second ? kI[NP - 1][e] : kI[0][e]), f[e]);
        n_iter += go_on;
    } while (go_on && (ALL || --left > 0));
    if (!NONE) no_score |= __builtin_amdgcn_readfirstlane(go_on ? imax_sel(worst, __double2hiint(taken)) : worst) >= SV_NONE_HI;
    return !go_on;
}

// The C variant's iterations with j2 chosen by b^2/a rounded to float, as long as that decides: c_smo_iterate_rounded of
// smo_solve.hip, with its proof.  What the working set's order would decide, equal values of f included, is left to ss_local.
// 963 instances, 1,000 steps: 2.82 -> 2.72 thousand cycles a step; cross-validation of 1203x13 2.31 -> 2.26 ms.  With that function's
// chains in single blocks, bits by masks and writes in the next step's waits 1.67 -> 1.61.
template <int E, int W, typename TB>
__device__ __forceinline__ bool ss_rounded(SmallShared<E, W> &sh, const SmallMap &map, SS_GLOBAL(TB) *K, int64_t ld, int col, const double (&kd)[E],
                                           double (&f)[E], unsigned &member, double Cp, double Cn, double local_eps, int max_iter, int &n_iter) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    constexpr int R = 4 * W;   // rows of sixteen lanes
    const unsigned my_i = lds_at(sh.ci + (tid >> 4)), my_j = lds_at(sh.score + (tid >> 4));
    unsigned my_z = lds_at(&sh.z[wave][0]);
    asm("" : "+v"(my_z));
    int own[E];
#pragma unroll
    for (int e = 0; e < E; ++e) own[e] = tid * E + e;
    uint64_t go;
    // what a step leaves to the waits of the next: I_low's bits, and the two elements' new z
    unsigned bit_i = 0, bit_j = 0, low_i = 0, low_j = 0, z_at_i = my_z, z_at_j = my_z;
    double nz_i = 0, nz_j = 0;
    int pending = 0;
    for (;;) {
        double fu[E];
#pragma unroll
        for (int e = 0; e < E; ++e) fu[e] = keep_or_none<0>(member << (31 - 2 * e), f[e]);
        SvWords cand;
        uint64_t mine_is, twice;
        row_first_candidate(fu, own, cand, mine_is, twice);
        const uint64_t first = lowest_of_rows(mine_is), equal = mine_is & (twice | ~first);   // a row that has one has its smallest more than once
        cand[3] = (int) ((unsigned) (equal >> (lane & 48)) & 0xffffu);
        publish_words(my_i, first, cand);
        lds_barrier();
        const SvCand c = sh.ci[lane & (R - 1)];
        write_by_lane0(pending, z_at_i, nz_i, z_at_j, nz_j);
        member = put_bits(put_bits(member, bit_i, low_i), bit_j, low_j);
        double up;
        uint64_t has_up;
        row_min_and_who<R>(c.v, up, has_up);
        const uint64_t up_rows = has_up & ((1ull << R) - 1);
        const uint64_t ties = (up_rows & (up_rows - 1)) | (up_rows & __builtin_amdgcn_ballot_w64(c.flag != 0));
        const int i = __builtin_amdgcn_readlane(c.at, __builtin_ctzll(has_up));
        TB kI[E];
        ss_load<E, TB>(K + (unsigned) map.row(i) * (unsigned) ld + col, kI);
        SV_PIN_MEMORY;
        z_at_i = my_z + 8u * (unsigned) i;
        const double kd_i = sh.kd[i], z_i = lds_f64(z_at_i);
        unsigned up_bit_i = own_bit<E, 2>(tid, i);
        asm("" : "+v"(up_bit_i));
        const SvBound bound_i = map.bound(i, Cp, Cn);
        double part[E], b[E], b_max = -__builtin_inf();
        float b32[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            part[e] = kd_i + kd[e];
            b[e] = keep_or_none<1>(member << (30 - 2 * e), -up + f[e]);
            b_max = fmax_f64(b_max, b[e]);
            b32[e] = __builtin_fmaxf((float) b[e], 0.0f);
        }
        const int violates = (__builtin_amdgcn_ballot_w64(!(b_max < local_eps)) != 0) & (n_iter <= max_iter);   // (the way out is one test)
        double up_i = bound_i.hi - z_i;
        asm("" : "+v"(up_i));
        int a_max = __builtin_fabs(up) < SV_UP_LEAST || ties != 0 ? 0x7f800000 : 0;   // (as the bits of a float)
        asm("" : "+v"(a_max));
        SV_PIN;
        double aIJ[E];
        float q[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            aIJ[e] = __builtin_fma(-2.0, (double) kI[e], part[e]);
            const float a32 = (float) aIJ[e];
            a_max = __float_as_int(a32) > a_max ? __float_as_int(a32) : a_max;
            q[e] = __builtin_fmaxf(b32[e] * (b32[e] * __builtin_amdgcn_rcpf(a32)), 0x1p-80f);
        }
        float mine = q[0], second = 0x1p-80f;
#pragma unroll
        for (int e = 1; e < E; ++e) {
            second = __builtin_fmaxf(second, __builtin_fminf(mine, q[e]));
            mine = __builtin_fmaxf(mine, q[e]);
        }
        int at = own[E - 1];
        double b_at = b[E - 1], a_at = aIJ[E - 1];
#pragma unroll
        for (int e = E - 2; e >= 0; --e) {
            const bool is = q[e] == mine;
            at = is ? own[e] : at;
            b_at = is ? b[e] : b_at;
            a_at = is ? aIJ[e] : a_at;
        }
        second = a_max < SV_A_BITS ? second : __builtin_inff();
        float best, next;
        uint64_t who;   // (several only if nothing will be decided)
        row_best_two_and_who(mine, second, best, next, who);
        publish_score(my_j, who, best, next, at, violates, b_at, a_at);
        lds_barrier();
        const SvScoreStep s = sh.score[lane & (R - 1)];
        uint64_t won;
        row_best_two_and_who<R>(s.score.best, s.score.second, best, next, won);
        const int row = __builtin_ctzll(won);
        const int j2 = __builtin_amdgcn_readlane(s.score.at, row);
        TB kJ[E];
        ss_load<E, TB>(K + (unsigned) map.row(j2) * (unsigned) ld + col, kJ);
        SV_PIN_MEMORY;
        z_at_j = my_z + 8u * (unsigned) j2;
        const double z_j = lds_f64(z_at_j);
        const SvBound bound_j = map.bound(j2, Cp, Cn);
        SV_PIN;
        const double steps = s.step.b / s.step.a;   // (every row's)
        const double q2 = readlane_f64(steps, row);
        const unsigned up_bit_j = own_bit<E, 2>(tid, j2);
        go = __builtin_amdgcn_ballot_w64(s.score.go != 0);
        const uint64_t sure = __builtin_amdgcn_ballot_w64(next < best * (1.0f - 0x1p-19f)) & __builtin_amdgcn_ballot_w64(best < 0x1p80f);
        if ((go & sure) == 0) break;
        SV_PIN;
        const double l = fmin_f64(fmin_f64(up_i, z_j - bound_j.lo), q2);
        nz_i = z_i + l;
        nz_j = z_j - l;
        const unsigned up_i_on = same_in_all_lanes(nz_i < bound_i.hi), up_j_on = same_in_all_lanes(nz_j < bound_j.hi);
        low_i = same_in_all_lanes(nz_i > bound_i.lo);
        low_j = same_in_all_lanes(nz_j > bound_j.lo);
        bit_i = up_bit_i << 1;
        bit_j = up_bit_j << 1;
        member = put_bits(put_bits(member, up_bit_i, up_i_on), up_bit_j, up_j_on);
        pending = 1;
        SV_PIN;
#pragma unroll
        for (int e = 0; e < E; ++e) f[e] = __builtin_fma(-l, (double) kJ[e] - (double) kI[e], f[e]);
        ++n_iter;
    }
    return go == 0;
}

// f[j] -= sum over the n_list listed rows (coefficients sh.f, rows in sh.k) in order (smo_kernel.cpp:300-319)
template <int E, int W, typename TB>
__device__ __forceinline__ void ss_update_f(const SmallShared<E, W> &sh, SS_GLOBAL(TB) *K, int64_t ld, int col, int first, int last, double (&f)[E]) {
    const int *rows = (const int *) sh.k;
    double sum[E] = {};
    int t = first;
    constexpr int U = 8;
    for (; t + U <= last; t += U) {
        TB k[U][E];
#pragma unroll
        for (int u = 0; u < U; ++u) ss_load<E, TB>(K + (int64_t) rows[t + u] * ld + col, k[u]);
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int e = 0; e < E; ++e) sum[e] = __builtin_fma(sh.f[t + u], (double) k[u][e], sum[e]);
    }
    for (; t < last; ++t) {
        TB k[E];
        ss_load<E, TB>(K + (int64_t) rows[t] * ld + col, k);
#pragma unroll
        for (int e = 0; e < E; ++e) sum[e] = __builtin_fma(sh.f[t], (double) k[e], sum[e]);
    }
#pragma unroll
    for (int e = 0; e < E; ++e) f[e] -= sum[e];
}

// Reads the kernel matrices of the problems whose workgroups run on this die into its L2, so that a step finds its rows
// there (250 cycles instead of 700 and more; a lone workgroup would need 330,000 cycles for 960 instances).  Workgroups are
// dealt to the eight dies in turn: number x of every eight reads for the problems x, x + 8, ..., up to SS_WARM_BYTES.
// 963 instances, 1,080 steps: 3.74 -> 3.48 million cycles; 360 instances, 348 steps: 1.25 -> 1.18.
#define SS_WARM_GROUPS 32
#define SS_WARM_BYTES (3 << 20)
template <typename TB>
__device__ __forceinline__ void ss_warm(const tsvm_small_problem *__restrict__ problems, int n_problems, int x, int group) {
    typedef uint32_t vec_t __attribute__((ext_vector_type(4), aligned(4)));
    constexpr int V = 16 / (int) sizeof(TB);
    int64_t left = SS_WARM_BYTES;
    for (int p = x; p < n_problems && left > 0; p += 8) {
        const tsvm_small_problem P = problems[p];
        const int n = P.n_pos + P.n_neg;
        left -= (int64_t) n * n * sizeof(TB);
        for (int r = group; r < n; r += SS_WARM_GROUPS) {
            const TB *const row = (const TB *) P.k + (int64_t) (r < P.n_pos ? P.row_pos + r : P.row_neg + (r - P.n_pos)) * P.ld;
#pragma unroll
            for (int side = 0; side < 2; ++side) {
                const int from = side ? P.row_neg : P.row_pos, count = side ? P.n_neg : P.n_pos;
                for (int c = threadIdx.x * V; c < count; c += blockDim.x * V) {
                    const vec_t v = *(const vec_t *) (row + from + c);
                    asm volatile("" ::"v"(v));
                }
            }
        }
    }
}

template <int E, int W, bool NU, typename TB>
__global__ __launch_bounds__(64 * W) void smo_small_kernel(const tsvm_small_problem *__restrict__ problems, int n_problems,
                                                           tsvm_small_state *states, int *ws_all, double *alpha_all, double *f_all, double eps,
                                                           int out_max_iter, int start) {
    constexpr int N = 64 * E * W;
    // (a lone wavefront's second reduction is six steps in registers; by rows and LDS, rounded: 3 pairs of 100 0.37 -> 0.42 ms)
    constexpr bool ROUNDED = !NU && W > 1;
    __shared__ SmallShared<E, W> sh;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if ((int) blockIdx.x >= n_problems) {
        const int warm = (int) blockIdx.x - (n_problems + 7) / 8 * 8;
        if (warm >= 0) ss_warm<TB>(problems, n_problems, warm % 8, warm / 8);
        return;
    }
    __builtin_amdgcn_s_setprio(3);   // (a chain of dependent steps: not to wait behind other kernels' wavefronts)
    const tsvm_small_problem P = problems[blockIdx.x];
    SS_GLOBAL(TB) *const K = (SS_GLOBAL(TB) *) P.k;
    const int64_t ld = P.ld;
    tsvm_small_state *const S = states + blockIdx.x;
    int *const ws_kept = ws_all + (int64_t) blockIdx.x * SS_MAX;
    if (!start && S->status != 0) return;
    SmallMap map;
    map.n0 = P.n_pos;
    map.n1 = P.n_neg;
    map.n0p = (P.n_pos + 3) & ~3;   // (both fit: n0p + n_neg <= N is checked on the host)
    map.col0 = P.row_pos;
    map.col1 = P.row_neg;
    map.n_rows = P.n_rows;
    double *const alpha = alpha_all + P.at, *const f_out = f_all + P.at;
    const int ws = P.ws, q = ws / 2;
    double f[E], kd[E];
    bool act[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int s = tid * E + e;
        act[e] = map.active(s);
        const double z = act[e] ? alpha[map.index(s)] * map.label(s) : 0.0;
        f[e] = act[e] ? f_out[map.index(s)] : 0.0;
        kd[e] = act[e] ? ((SS_GLOBAL(double) *) P.k_diag)[map.row(s)] : 1.0;
        sh.kd[s] = kd[e];
#pragma unroll
        for (int w = 0; w < W; ++w) sh.z[w][s] = z;
    }
    const SvBound bound = map.bound(tid * E, P.Cp, P.Cn);   // (a thread's four slots are of one group)
    // (a vector that starts at an active slot may end in the columns behind the group's, which nothing uses, or up to
    // three elements behind the matrix)
    const int col = act[0] ? map.row(tid * E) : 0;
    double previous_diff = __builtin_inf(), last_diff = __builtin_inf(), second_last_diff = __builtin_inf(), diff = 0.0;
    int same_count = 0, swap_count = 0, iter = 0, status = 0;
    long long local_iter = 0;
    if (!start) {
        previous_diff = S->previous_diff;
        last_diff = S->last_diff;
        second_last_diff = S->second_last_diff;
        same_count = S->same_count;
        swap_count = S->swap_count;
        iter = S->iter;
        local_iter = S->local_iter;
        for (int t = tid; t < ws; t += 64 * W) sh.ws[t] = (unsigned short) ws_kept[t];
    }
    __syncthreads();
    // the list of the instances with `coef` != 0 in slot order, or of the working set's in its order, for ss_update_f
    auto make_list = [&](int count, auto coefficient, auto row_of) {   // entry t < count
        int *rows = (int *) sh.k;
        __syncthreads();
        int filled = 0;
        for (int t0 = 0; t0 < count; t0 += 64 * W) {
            const int t = t0 + tid;
            const double c = t < count ? coefficient(t) : 0.0;
            const uint64_t b = __builtin_amdgcn_ballot_w64(c != 0.0);
            if (lane == 0) sh.red[0][wave] = (double) __popcll(b);
            __syncthreads();
            int before = filled;
            for (int w = 0; w < W; ++w) {
                const int cnt = (int) sh.red[0][w];
                if (w < wave) before += cnt;
                filled += cnt;
            }
            if (c != 0.0) {
                const int at = before + __popcll(b & ((1ull << lane) - 1ull));
                sh.f[at] = c;
                rows[at] = row_of(t);
            }
            __syncthreads();
        }
        return filled;
    };
    if (start) {   // f from a non-zero alpha, in batches of 101 rows (csmosolver.cpp:189-214)
        const int n = make_list(N, [&](int s) { return map.active(s) ? -sh.z[wave][s] : 0.0; }, [&](int s) { return map.row(s); });
        for (int t = 0; t < n; t += 101) ss_update_f<E, W, TB>(sh, K, ld, col, t, t + 101 < n ? t + 101 : n, f);
        __syncthreads();
    }
    const int iter_end = iter + SS_MAX_ITER;
    long long inner_here = 0;
    while (status == 0 && iter < iter_end && inner_here < SS_MAX_INNER) {
        // the working set: its second half moves to the front, q new ones follow (csmosolver.cpp:63-77)
        const int n_new = iter == 0 ? ws : q, first_new = iter == 0 ? 0 : ws - n_new;
#pragma unroll
        for (int e = 0; e < E; ++e) sh.pos[tid * E + e] = 0xffff;
        unsigned short kept[E];
#pragma unroll
        for (int h = 0; h < E; ++h) {
            const int t = h * 64 * W + tid;
            kept[h] = iter > 0 && t < q ? sh.ws[t + q] : 0;
        }
        __syncthreads();
#pragma unroll
        for (int h = 0; h < E; ++h) {
            const int t = h * 64 * W + tid;
            if (iter > 0 && t < q) {
                sh.ws[t] = kept[h];
                sh.pos[kept[h]] = (unsigned short) t;
            }
        }
        __syncthreads();
        unsigned member_all = 0;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int s = tid * E + e;
            const double z = sh.z[wave][s];
            unsigned b = 0;
            if (act[e]) {
                const unsigned u = z < bound.hi ? 1u : 0u, l = z > bound.lo ? 1u : 0u;
                b = NU ? (u | l << 2) << (s < map.n0p ? 0 : 1) : (u | l << 1);
            }
            member_all |= b << ((NU ? 4 : 2) * e);
            sh.flags[s] = (unsigned char) (sh.pos[s] == 0xffff ? b : 0u);
        }
        __syncthreads();
        if (!ss_select<E, W, NU>(sh, f, act, n_new, first_new)) {
            status = 2;
            break;
        }
        for (int t = tid; t < ws; t += 64 * W) sh.pos[sh.ws[t]] = (unsigned short) t;
        __syncthreads();
        unsigned member = 0;
        double fl[E], z_old[E], mn[2] = {__builtin_inf(), __builtin_inf()}, mx[2] = {-__builtin_inf(), -__builtin_inf()};
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int s = tid * E + e, p = sh.pos[s];
            const unsigned b = p != 0xffff ? (member_all >> ((NU ? 4 : 2) * e)) & (NU ? 15u : 3u) : 0u;
            member |= b << ((NU ? 4 : 2) * e);
            fl[e] = f[e];
            z_old[e] = sh.z[wave][s];
#pragma unroll
            for (int r = 0; r < (NU ? 2 : 1); ++r) {
                mn[r] = fmin_f64(mn[r], (b >> r) & 1u ? f[e] : __builtin_inf());
                mx[r] = fmax_f64(mx[r], (b >> (r + (NU ? 2 : 1))) & 1u ? f[e] : -__builtin_inf());
            }
        }
        // the initial gap, and with it the local threshold (smo_kernel.cpp:61-66, 176-183)
#pragma unroll
        for (int r = 0; r < (NU ? 2 : 1); ++r) {
            const double lo = wave_min_f64(mn[r]), hi = wave_max_f64(mx[r]);
            if (lane == 0) { sh.red[2 * r][wave] = lo; sh.red[2 * r + 1][wave] = hi; }
        }
        __syncthreads();
        double gap[2];
#pragma unroll
        for (int r = 0; r < (NU ? 2 : 1); ++r) {
            double lo = sh.red[2 * r][0];
#pragma unroll
            for (int w = 1; w < W; ++w) lo = fmin_f64(lo, sh.red[2 * r][w]);
            gap[r] = block_max<W>(sh.red[2 * r + 1]) - lo;
        }
        diff = NU ? (gap[0] < gap[1] ? gap[1] : gap[0]) : gap[0];
        const double tenth = NU ? 0.1 * diff : 0.1f * diff;   // (a float literal in the C variant, a double in the nu one)
        const double local_eps = tenth > eps ? tenth : eps;
        __syncthreads();
        bool no_score = !__builtin_amdgcn_readfirstlane(local_eps > 0.0 ? 1 : 0);
        int steps = 0;
        if (!no_score) {
            unsigned now = member;
            if constexpr (ROUNDED) {
                bool done;
                int stretch = 4;   // (as in c_smo_solve_kernel)
                do {
                    const int before = steps;
                    done = ss_rounded<E, W, TB>(sh, map, K, ld, col, kd, fl, now, P.Cp, P.Cn, local_eps, P.max_iter, steps);
                    if (done) break;
                    stretch = steps - before > stretch ? 4 : stretch < 1024 ? 8 * stretch : stretch;
                    done = ss_local<E, W, NU, false, false, TB>(sh, map, K, ld, col, kd, fl, now, P.Cp, P.Cn, local_eps, P.max_iter, no_score, steps, stretch);
                } while (!done && !no_score);
            } else {
                ss_local<E, W, NU, false, true, TB>(sh, map, K, ld, col, kd, fl, now, P.Cp, P.Cn, local_eps, P.max_iter, no_score, steps, 0);
            }
            if (no_score) {   // once more from the start
                __syncthreads();
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    fl[e] = f[e];
#pragma unroll
                    for (int w = 0; w < W; ++w) sh.z[w][tid * E + e] = z_old[e];
                }
                __syncthreads();
            }
        }
        if (no_score) {
            steps = 0;
            ss_local<E, W, NU, true, true, TB>(sh, map, K, ld, col, kd, fl, member, P.Cp, P.Cn, local_eps, P.max_iter, no_score, steps, 0);
        }
        inner_here += steps;
        if (!NU) local_iter += steps;   // (the nu variant reports none, smo_kernel.cpp:283)
        // alpha_diff of the working set, in its order: -(new - old) * y
        __syncthreads();
        double *const old = sh.k;   // (free between the local solver and the list)
#pragma unroll
        for (int e = 0; e < E; ++e) old[tid * E + e] = z_old[e];
        __syncthreads();
        double ad[E];
        int rr[E], cnt = 0;
#pragma unroll
        for (int h = 0; h < E; ++h) {   // thread t owns entries E t .. E t + E - 1
            const int t = tid * E + h;
            const int s = t < ws ? sh.ws[t] : 0;
            ad[h] = t < ws ? -(sh.z[wave][s] - old[s]) : 0.0;
            rr[h] = map.row(s);
            cnt += ad[h] != 0.0;
        }
        int incl = cnt;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(incl, d, 64);
            if (lane >= d) incl += o;
        }
        if (lane == 63) sh.red[0][wave] = (double) incl;
        __syncthreads();
        int at = incl - cnt, n_list = 0;
#pragma unroll
        for (int w = 0; w < W; ++w) {
            const int c = (int) sh.red[0][w];
            if (w < wave) at += c;
            n_list += c;
        }
        int *const rows = (int *) sh.k;
#pragma unroll
        for (int h = 0; h < E; ++h)
            if (ad[h] != 0.0) {
                sh.f[at] = ad[h];
                rows[at] = rr[h];
                ++at;
            }
        __syncthreads();
        ss_update_f<E, W, TB>(sh, K, ld, col, 0, n_list, f);
        __syncthreads();
        // stall guards and stopping rule (csmosolver.cpp:86-111)
        if (__builtin_fabs(diff - previous_diff) < eps * 0.001) {
            same_count++;
        } else {
            same_count = 0;
            previous_diff = diff;
        }
        if (__builtin_fabs(diff - second_last_diff) < eps * 0.001) swap_count++;
        else swap_count = 0;
        second_last_diff = last_diff;
        last_diff = diff;
        const bool stalled = (same_count >= 10 || swap_count >= 10) && __builtin_fabs(diff - 2.0) > eps;
        if (stalled || diff < eps || (out_max_iter != -1 && iter == out_max_iter)) status = 1;
        ++iter;
    }
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const int s = tid * E + e;
        if (act[e]) {
            alpha[map.index(s)] = sh.z[wave][s] * map.label(s) + 0.0;   // (+ 0.0: a zero comes out as +0, as from alpha +- l)
            f_out[map.index(s)] = f[e];
        }
    }
    for (int t = tid; t < ws; t += 64 * W) ws_kept[t] = sh.ws[t];
    if (tid == 0) {
        S->previous_diff = previous_diff;
        S->last_diff = last_diff;
        S->second_last_diff = second_last_diff;
        S->same_count = same_count;
        S->swap_count = swap_count;
        S->iter = iter;
        S->local_iter = local_iter;
        S->diff = diff;
        S->status = status;
        S->xcd = (int) __builtin_amdgcn_s_getreg(20 | (0 << 6) | (3 << 11));   // XCC_ID
    }
}

template <int E, int W, typename TB>
static void launch_small(const tsvm_small_problem *problems, int n_problems, tsvm_small_state *states, int *ws, double *alpha, double *f, int nu,
                         double eps, int out_max_iter, int start, hipStream_t stream) {
    const int grid = start ? (n_problems + 7) / 8 * 8 + 8 * SS_WARM_GROUPS : n_problems;
    if (nu)
        smo_small_kernel<E, W, true, TB><<<grid, 64 * W, 0, stream>>>(problems, n_problems, states, ws, alpha, f, eps, out_max_iter, start);
    else
        smo_small_kernel<E, W, false, TB><<<grid, 64 * W, 0, stream>>>(problems, n_problems, states, ws, alpha, f, eps, out_max_iter, start);
}

extern "C" {

int tsvm_smo_small_max(void) { return SS_MAX; }

int tsvm_smo_solve_small(int row_type, const tsvm_small_problem *problems, int n_problems, int max_slots, tsvm_small_state *states, int *ws,
                         double *alpha, double *f, int nu, double eps, int out_max_iter, int start, tsvm_stream stream) {
    TSVM_REQUIRE(row_type == TSVM_ROW_F32 || row_type == TSVM_ROW_F64, "tsvm_smo_solve_small: row type %d", row_type);
    TSVM_REQUIRE(n_problems >= 0, "tsvm_smo_solve_small: %d problems", n_problems);
    TSVM_REQUIRE(max_slots >= 1 && max_slots <= SS_MAX, "tsvm_smo_solve_small: %d slots (1 .. %d)", max_slots, SS_MAX);
    if (n_problems == 0) return 0;
    TSVM_REQUIRE(problems && states && ws && alpha && f, "tsvm_smo_solve_small: null argument");
#define TSVM_SMALL(E, W, TB) launch_small<E, W, TB>(problems, n_problems, states, ws, alpha, f, nu, eps, out_max_iter, start, tsvm_s(stream))
    // (the shapes of the local solvers, smo_solve.hip, for the same reasons)
#define TSVM_SMALL_T(TB)                                  \
    do {                                                  \
        if (max_slots <= 64) TSVM_SMALL(1, 1, TB);        \
        else if (max_slots <= 128) TSVM_SMALL(2, 1, TB);  \
        else if (max_slots <= 256) TSVM_SMALL(4, 1, TB);  \
        else if (max_slots <= 512) TSVM_SMALL(4, 2, TB);  \
        else TSVM_SMALL(4, 4, TB);                        \
    } while (0)
    if (row_type == TSVM_ROW_F32) TSVM_SMALL_T(float);
    else TSVM_SMALL_T(double);
#undef TSVM_SMALL_T
#undef TSVM_SMALL
    TSVM_LAUNCH_CHECK();
    return 0;
}

}  // extern "C"
