// What the local SMO solvers share (smo_solve.hip: one call per working set; smo_small.hip: whole solves of small
// problems): masked extrema over a working set that is spread over the registers of one, two or four wavefronts, and LDS writes by
// single lanes.  See smo_solve.hip for what bounds these kernels and why they are written this way.
#pragma once
#include "tsvm_device.h"

// What a masked-out element or score is replaced by.  Only the high word is replaced (one instruction), so every value from
// SV_NONE on means "not a candidate": the last 2^32 finite doubles and infinity, which is no candidate for the reference either.
// (The high word of infinity itself would make NaNs of the low words.  A lower one is not enough: a solve on a kernel that is
// not positive definite may run away, and its scores b^2/a pass 2^1023 before they overflow.)
#define SV_NONE_HI 0x7fefffff
#define SV_NONE 0x1.fffffp+1023

// x when the sign bit of `bit_at_top` is set, otherwise a value >= SV_NONE (SIGN = 0) or <= -SV_NONE (SIGN = 1).
template <int SIGN>
__device__ __forceinline__ double keep_or_none(unsigned bit_at_top, double x) {
    const int m = (int) bit_at_top >> 31;
    return __hiloint2double((m & __double2hiint(x)) | (~m & (int) (SV_NONE_HI | (SIGN ? 0x80000000u : 0u))), __double2loint(x));
}

// The scalar test for such a value.
__device__ __forceinline__ bool is_none(double v) { return __builtin_amdgcn_readfirstlane(__double2hiint(v)) >= SV_NONE_HI; }

// The smallest of a wavefront's E * 64 values (x[e] of a lane is element base + e) and the first element that has it:
// `value` is the minimum; m and at are every lane's own smallest value and its first element; the lane returned is the
// lowest one whose m is the minimum, so its `at` is the lowest element among equals.
// With one wavefront per SIMD an instruction costs its four cycles whatever it does, a DPP operand has to be two wait
// states old, and a value that crosses to the scalar unit and back costs about forty cycles, as much as a branch around
// a few instructions (all measured on this part).  Hence one chain of six DPP steps on doubles with the instructions
// that find the thread's own element in its gaps, and the winner by ballot instead of a second chain over the indices.
#define SV_PIN __builtin_amdgcn_sched_barrier(0)
// (the same for memory accesses: a row's load stays in front of the work that is to pass while it is on its way, and
// in front of the exit test; the block is not declared restrict, or the load could be moved all the same)
#define SV_PIN_MEMORY asm volatile("" ::: "memory")
// TWICE: `twice` is the lanes of which several elements hold the lane's smallest value.
template <int E, bool TWICE>
__device__ __forceinline__ int wave_argmin(const double (&x)[E], int base, double &value, double &m, int &at, uint64_t &twice) {
    m = x[0];
#pragma unroll
    for (int e = 1; e < E; ++e) m = fmin_f64(m, x[e]);
    SV_PIN;
    uint64_t has[E];   // which lanes' element e is their minimum
#pragma unroll
    for (int e = 0; e < (TWICE ? E : E - 1); ++e) asm volatile("v_cmp_eq_f64_e64 %0, %1, %2" : "=s"(has[e]) : "v"(x[e]), "v"(m));
    SV_PIN;
    int tl = dpp_i32<TSVM_DPP_XOR1>(__double2loint(m)), th = dpp_i32<TSVM_DPP_XOR1>(__double2hiint(m));
    double r = fmin_f64(m, __hiloint2double(th, tl));
    SV_PIN;
    at = base + E - 1;
#pragma unroll
    for (int e = E - 2; e >= 0 && e >= E - 3; --e) asm volatile("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(at) : "v"(at), "v"(base + e), "s"(has[e]));
    SV_PIN;
    tl = dpp_i32<TSVM_DPP_XOR2>(__double2loint(r));
    th = dpp_i32<TSVM_DPP_XOR2>(__double2hiint(r));
    r = fmin_f64(r, __hiloint2double(th, tl));
    SV_PIN;
#pragma unroll
    for (int e = E - 4; e >= 0; --e) asm volatile("v_cndmask_b32_e64 %0, %1, %2, %3" : "=v"(at) : "v"(at), "v"(base + e), "s"(has[e]));
    SV_PIN;
    if constexpr (TWICE) {   // (scalar work in the gaps of the chain)
        twice = 0;
        uint64_t one = E > 1 ? has[0] : 0;
#pragma unroll
        for (int e = 1; e < E; ++e) {
            twice |= one & has[e];
            one |= has[e];
        }
    }
    tl = dpp_i32<TSVM_DPP_HALF_MIRROR>(__double2loint(r));
    th = dpp_i32<TSVM_DPP_HALF_MIRROR>(__double2hiint(r));
    r = fmin_f64(r, __hiloint2double(th, tl));
    tl = dpp_i32<TSVM_DPP_MIRROR>(__double2loint(r));
    th = dpp_i32<TSVM_DPP_MIRROR>(__double2hiint(r));
    r = fmin_f64(r, __hiloint2double(th, tl));
    // (lanes outside the row mask keep what the step before moved there, which is no smaller than their own r)
    tl = __builtin_amdgcn_update_dpp(tl, __double2loint(r), TSVM_DPP_BCAST15, 0xa, 0xf, false);
    th = __builtin_amdgcn_update_dpp(th, __double2hiint(r), TSVM_DPP_BCAST15, 0xa, 0xf, false);
    r = fmin_f64(r, __hiloint2double(th, tl));
    tl = __builtin_amdgcn_update_dpp(tl, __double2loint(r), TSVM_DPP_BCAST31, 0xc, 0xf, false);
    th = __builtin_amdgcn_update_dpp(th, __double2hiint(r), TSVM_DPP_BCAST31, 0xc, 0xf, false);
    r = fmin_f64(r, __hiloint2double(th, tl));
    value = readlane_f64(r, 63);
    return __builtin_ctzll(__builtin_amdgcn_ballot_w64(m == value));
}
template <int E>
__device__ __forceinline__ int wave_first_argmin(const double (&x)[E], int base, double &value, double &m, int &at) {
    uint64_t twice;
    return wave_argmin<E, false>(x, base, value, m, at, twice);
}

// One wavefront's best candidate for the others: the workgroup's minimum is taken over W of these.
struct __align__(16) SvCand {
    double v;
    int at;
    int flag;
};

// Writes by one lane (or by one of each row), without the branch that an if around them costs (all 64 lanes are active
// before and after).  Four wavefronts share the LDS, so a write or a broadcast read by 64 lanes is paid four times over:
// what one lane knows is written by that lane alone.
#define SV_EXEC_ON "s_mov_b64 exec, %0\n\t"
#define SV_EXEC_OFF "s_mov_b64 exec, -1"
__device__ __forceinline__ void publish_words(unsigned slot, uint64_t lanes, int a, int b, int c, int d) {
    typedef int v4i __attribute__((ext_vector_type(4)));
    const v4i v = {a, b, c, d};
    asm volatile(SV_EXEC_ON "ds_write_b128 %1, %2\n\t" SV_EXEC_OFF :: "s"(lanes), "v"(slot), "v"(v) : "memory");
}
__device__ __forceinline__ void publish(SvCand *slot, uint64_t lanes, double m, int at, int flag) {
    publish_words(lds_at(slot), lanes, __double2loint(m), __double2hiint(m), at, flag);
}
// The same with the lane's E values of f and of the block row for the step (the row's values in slots of eight bytes).
// (One asm statement each: nothing else may come between the two writes of exec.)
// `only`: the lanes that write, each to slots of its own.  S: doubles from one slot for f to the next.
template <int E, typename TB, int S = 1>
__device__ __forceinline__ void publish_row(double *f_slot, double *k_slot, uint64_t only, const double (&f)[E], const TB (&k)[E]) {
    const unsigned fa = lds_at(f_slot), ka = lds_at(k_slot);
    static_assert(E == 1 || E == 2 || E == 4, "elements per thread");
    if constexpr (E == 1 && sizeof(TB) == 4)
        asm volatile(SV_EXEC_ON "ds_write_b64 %1, %3\n\tds_write_b32 %2, %4\n\t" SV_EXEC_OFF
                     :: "s"(only), "v"(fa), "v"(ka), "v"(f[0]), "v"(k[0]) : "memory");
    else if constexpr (E == 1)
        asm volatile(SV_EXEC_ON "ds_write_b64 %1, %3\n\tds_write_b64 %2, %4\n\t" SV_EXEC_OFF
                     :: "s"(only), "v"(fa), "v"(ka), "v"(f[0]), "v"(k[0]) : "memory");
    else if constexpr (E == 2 && sizeof(TB) == 4)
        asm volatile(SV_EXEC_ON "ds_write2_b64 %1, %3, %4 offset1:%7\n\tds_write2_b32 %2, %5, %6 offset1:2\n\t" SV_EXEC_OFF
                     :: "s"(only), "v"(fa), "v"(ka), "v"(f[0]), "v"(f[1]), "v"(k[0]), "v"(k[1]), "n"(S) : "memory");
    else if constexpr (E == 2)
        asm volatile(SV_EXEC_ON "ds_write2_b64 %1, %3, %4 offset1:%7\n\tds_write2_b64 %2, %5, %6 offset1:1\n\t" SV_EXEC_OFF
                     :: "s"(only), "v"(fa), "v"(ka), "v"(f[0]), "v"(f[1]), "v"(k[0]), "v"(k[1]), "n"(S) : "memory");
    else if constexpr (sizeof(TB) == 4)
        asm volatile(SV_EXEC_ON "ds_write2_b64 %1, %3, %4 offset1:%11\n\tds_write2_b64 %1, %5, %6 offset0:%12 offset1:%13\n\t"
                     "ds_write2_b32 %2, %7, %8 offset1:2\n\tds_write2_b32 %2, %9, %10 offset0:4 offset1:6\n\t" SV_EXEC_OFF
                     :: "s"(only), "v"(fa), "v"(ka), "v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(f[3]), "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]), "n"(S), "n"(2 * S), "n"(3 * S) : "memory");
    else
        asm volatile(SV_EXEC_ON "ds_write2_b64 %1, %3, %4 offset1:%11\n\tds_write2_b64 %1, %5, %6 offset0:%12 offset1:%13\n\t"
                     "ds_write2_b64 %2, %7, %8 offset1:1\n\tds_write2_b64 %2, %9, %10 offset0:2 offset1:3\n\t" SV_EXEC_OFF
                     :: "s"(only), "v"(fa), "v"(ka), "v"(f[0]), "v"(f[1]), "v"(f[2]), "v"(f[3]), "v"(k[0]), "v"(k[1]), "v"(k[2]), "v"(k[3]), "n"(S), "n"(2 * S), "n"(3 * S) : "memory");
}
// The same for a record that is already a run of four registers, and for a score with its step.
typedef int SvWords __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void publish_words(unsigned slot, uint64_t lanes, const SvWords &v) {
    asm volatile(SV_EXEC_ON "ds_write_b128 %1, %2\n\t" SV_EXEC_OFF :: "s"(lanes), "v"(slot), "v"(v) : "memory");
}
__device__ __forceinline__ void publish_score(unsigned slot, uint64_t lanes, float best, float second, int at, int go, double b, double a) {
    const SvWords v = {__float_as_int(best), __float_as_int(second), at, go};
    asm volatile(SV_EXEC_ON "ds_write_b128 %1, %2\n\tds_write2_b64 %1, %3, %4 offset0:2 offset1:3\n\t" SV_EXEC_OFF
                 :: "s"(lanes), "v"(slot), "v"(v), "v"(b), "v"(a) : "memory");
}
__device__ __forceinline__ double lds_f64(unsigned at) { return *(const __attribute__((address_space(3))) double *) (uintptr_t) at; }
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }
// (p, then q: if both name one element the second value is the final one; `on` = 0: nothing is written)
__device__ __forceinline__ void write_by_lane0(int on, double *p, double v, double *q, double w) {
    asm volatile(SV_EXEC_ON "ds_write_b64 %1, %2\n\tds_write_b64 %3, %4\n\t" SV_EXEC_OFF
                 :: "s"((uint64_t) (uint32_t) __builtin_amdgcn_readfirstlane(on)), "v"(lds_at(p)), "v"(v), "v"(lds_at(q)), "v"(w) : "memory");
}

// (the same by LDS addresses)
__device__ __forceinline__ void write_by_lane0(int on, unsigned p, double v, unsigned q, double w) {
    asm volatile(SV_EXEC_ON "ds_write_b64 %1, %2\n\tds_write_b64 %3, %4\n\t" SV_EXEC_OFF :: "s"((uint64_t) (uint32_t) on), "v"(p), "v"(v), "v"(q), "v"(w) : "memory");
}

template <int W>
__device__ __forceinline__ double block_max(const double *s_v) {
    double v = s_v[0];
#pragma unroll
    for (int w = 1; w < W; ++w) v = fmax_f64(v, s_v[w]);
    return v;
}

// Membership bits in three instructions a change.  own_bit: element t's first bit (of EACH) in the thread that owns it; in another
// one it is a bit beyond the elements', which nobody reads.  A decision that all lanes have come to alike is a mask of
// ones or zeros in a scalar register.
template <int E, int EACH = 1>
__device__ __forceinline__ unsigned own_bit(int tid, int t) {
    const unsigned at = (unsigned) (t - tid * E) * EACH;
    return 1u << (at < 31u ? at : 31u);
}
__device__ __forceinline__ unsigned same_in_all_lanes(bool x) { return (unsigned) __builtin_amdgcn_ballot_w64(x); }
__device__ __forceinline__ unsigned put_bits(unsigned m, unsigned bits, unsigned on) { return (m & ~bits) | (bits & on); }

// The local solvers hold alpha times its label, z = y * alpha in [lo, hi] with lo = 0, hi = Cp for y > 0 and lo = -Cn,
// hi = 0 for y < 0: an element is in I_up while z < hi and in I_low while z > lo, a step is bounded by hi - z_i and z_j - lo
// (smo_kernel.h:13-23, smo_kernel.cpp:94-99), and it moves z_i up and z_j down by the same l.  All of it rounds as the
// reference's expressions in alpha do (they differ in the sign of both operands), and an infinite C (a hard margin) is a bound like
// any other.  (The bounds are selected by the label: computed from it, as y * C/2 + C/2, one of them would be inf - inf.)
struct __align__(16) SvBound {
    double hi, lo;
};

struct __align__(16) SvStep {   // f_t - up and K_ii + K_tt - 2 K_it of a candidate for j2
    double b, a;
};

// One row's (sixteen lanes') best and second-best score, rounded to float.
struct __align__(16) SvScore {
    float best, second;
    int at, go;
};
struct SvScoreStep {
    SvScore score;
    SvStep step;
};

// What follows are whole chains in one asm block each, with registers of their own from v144 on (the halves of a register pair
// cannot be named otherwise): between the builtins and one-instruction blocks that they replace the compiler puts
// wait states, as it does not know what such a block holds.  A DPP operand is two wait states old everywhere, a mask
// that a comparison wrote is read three instructions later.
#define SV_DPP_MOV(TO, FROM, CTRL) "v_mov_b32_dpp " TO ", " FROM " " CTRL " row_mask:0xf bank_mask:0xf\n\t"
#define SV_MIN_STEP(CTRL) SV_DPP_MOV("v148", "v150", CTRL) SV_DPP_MOV("v149", "v151", CTRL) "v_min_f64 v[150:151], v[150:151], v[148:149]\n\t"
// The smallest of a row's E * 16 values: every lane's own smallest and its first element as the record that the lane publishes (its last word is
// anything); `has`: the lanes whose own is the row's.  (The first four steps of wave_argmin.)
template <int E>
__device__ __forceinline__ void row_first_candidate(const double (&x)[E], const int (&at)[E], SvWords &rec, uint64_t &has) {
    uint64_t h0, h1, h2;
    if constexpr (E == 4) {
        asm("v_min_f64 v[144:145], %5, %6\n\t"
            "v_min_f64 v[148:149], %7, %8\n\t"
            "v_min_f64 v[144:145], v[144:145], v[148:149]\n\t"
            "v_cmp_eq_f64_e64 %2, %5, v[144:145]\n\t"
            "v_cmp_eq_f64_e64 %3, %6, v[144:145]\n\t"
            "v_cmp_eq_f64_e64 %4, %7, v[144:145]\n\t"
            SV_DPP_MOV("v148", "v144", "quad_perm:[1,0,3,2]") SV_DPP_MOV("v149", "v145", "quad_perm:[1,0,3,2]")
            "v_min_f64 v[150:151], v[144:145], v[148:149]\n\t"
            "v_cndmask_b32_e64 v146, %12, %11, %4\n\t"
            "v_cndmask_b32_e64 v146, v146, %10, %3\n\t"
            SV_MIN_STEP("quad_perm:[2,3,0,1]")
            "v_cndmask_b32_e64 v146, v146, %9, %2\n\t"
            "s_nop 0\n\t" SV_MIN_STEP("row_half_mirror")
            "s_nop 1\n\t" SV_MIN_STEP("row_mirror")
            "v_cmp_eq_f64_e64 %1, v[144:145], v[150:151]"
            : "=&{v[144:147]}"(rec), "=&s"(has), "=&s"(h0), "=&s"(h1), "=&s"(h2)
            : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
            : "v148", "v149", "v150", "v151");
    } else {
        static_assert(E == 2, "elements per thread");
        asm("v_min_f64 v[144:145], %3, %4\n\t"
            "v_cmp_eq_f64_e64 %2, %3, v[144:145]\n\t"
            "s_nop 0\n\t"
            SV_DPP_MOV("v148", "v144", "quad_perm:[1,0,3,2]") SV_DPP_MOV("v149", "v145", "quad_perm:[1,0,3,2]")
            "v_min_f64 v[150:151], v[144:145], v[148:149]\n\t"
            "v_cndmask_b32_e64 v146, %6, %5, %2\n\t"
            "s_nop 0\n\t" SV_MIN_STEP("quad_perm:[2,3,0,1]")
            "s_nop 1\n\t" SV_MIN_STEP("row_half_mirror")
            "s_nop 1\n\t" SV_MIN_STEP("row_mirror")
            "v_cmp_eq_f64_e64 %1, v[144:145], v[150:151]"
            : "=&{v[144:147]}"(rec), "=&s"(has), "=&s"(h0)
            : "v"(x[0]), "v"(x[1]), "v"(at[0]), "v"(at[1])
            : "v148", "v149", "v150", "v151");
    }
}
// The same for four elements per thread with `twice`, the lanes whose own smallest occurs more than once.
__device__ __forceinline__ void row_first_candidate(const double (&x)[4], const int (&at)[4], SvWords &rec, uint64_t &has, uint64_t &twice) {
    uint64_t h0, h1, h2, h3;
    asm("v_min_f64 v[144:145], %6, %7\n\t"
        "v_min_f64 v[148:149], %8, %9\n\t"
        "v_min_f64 v[144:145], v[144:145], v[148:149]\n\t"
        "v_cmp_eq_f64_e64 %2, %6, v[144:145]\n\t"
        "v_cmp_eq_f64_e64 %3, %7, v[144:145]\n\t"
        "v_cmp_eq_f64_e64 %4, %8, v[144:145]\n\t"
        SV_DPP_MOV("v148", "v144", "quad_perm:[1,0,3,2]") SV_DPP_MOV("v149", "v145", "quad_perm:[1,0,3,2]")
        "v_min_f64 v[150:151], v[144:145], v[148:149]\n\t"
        "v_cndmask_b32_e64 v146, %13, %12, %4\n\t"
        "v_cndmask_b32_e64 v146, v146, %11, %3\n\t"
        SV_MIN_STEP("quad_perm:[2,3,0,1]")
        "v_cndmask_b32_e64 v146, v146, %10, %2\n\t"
        "v_cmp_eq_f64_e64 %5, %9, v[144:145]\n\t"
        SV_MIN_STEP("row_half_mirror")
        "s_nop 1\n\t" SV_MIN_STEP("row_mirror")
        "v_cmp_eq_f64_e64 %1, v[144:145], v[150:151]"
        : "=&{v[144:147]}"(rec), "=&s"(has), "=&s"(h0), "=&s"(h1), "=&s"(h2), "=&s"(h3)
        : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
        : "v148", "v149", "v150", "v151");
    twice = (h0 & h1) | ((h0 | h1) & h2) | ((h0 | h1 | h2) & h3);
}
// Two of them, for the nu variant's sides: each chain fills the other's wait states.
#define SV_MOVS(CTRL) SV_DPP_MOV("v148", "v150", CTRL) SV_DPP_MOV("v149", "v151", CTRL) SV_DPP_MOV("v156", "v158", CTRL) SV_DPP_MOV("v157", "v159", CTRL)
#define SV_MINS "v_min_f64 v[150:151], v[150:151], v[148:149]\n\tv_min_f64 v[158:159], v[158:159], v[156:157]\n\t"
#define SV_FIRST_MOVS(CTRL) SV_DPP_MOV("v148", "v144", CTRL) SV_DPP_MOV("v149", "v145", CTRL) SV_DPP_MOV("v156", "v152", CTRL) SV_DPP_MOV("v157", "v153", CTRL) \
    "v_min_f64 v[150:151], v[144:145], v[148:149]\n\tv_min_f64 v[158:159], v[152:153], v[156:157]\n\t"
template <int E>
__device__ __forceinline__ void row_first_candidates(const double (&x)[E], const double (&y)[E], const int (&at)[E], SvWords &rec_x, SvWords &rec_y,
                                                     uint64_t &has_x, uint64_t &has_y) {
    uint64_t x0, x1, x2, y0, y1, y2;
    if constexpr (E == 4) {
        asm("v_min_f64 v[144:145], %10, %11\n\t"
            "v_min_f64 v[152:153], %14, %15\n\t"
            "v_min_f64 v[148:149], %12, %13\n\t"
            "v_min_f64 v[156:157], %16, %17\n\t"
            "v_min_f64 v[144:145], v[144:145], v[148:149]\n\t"
            "v_min_f64 v[152:153], v[152:153], v[156:157]\n\t"
            "v_cmp_eq_f64_e64 %4, %10, v[144:145]\n\t"
            "v_cmp_eq_f64_e64 %5, %11, v[144:145]\n\t"
            "v_cmp_eq_f64_e64 %6, %12, v[144:145]\n\t"
            "v_cmp_eq_f64_e64 %7, %14, v[152:153]\n\t"
            "v_cmp_eq_f64_e64 %8, %15, v[152:153]\n\t"
            "v_cmp_eq_f64_e64 %9, %16, v[152:153]\n\t"
            SV_FIRST_MOVS("quad_perm:[1,0,3,2]")
            "v_cndmask_b32_e64 v146, %21, %20, %6\n\t"
            "v_cndmask_b32_e64 v154, %21, %20, %9\n\t"
            SV_MOVS("quad_perm:[2,3,0,1]") SV_MINS
            "v_cndmask_b32_e64 v146, v146, %19, %5\n\t"
            "v_cndmask_b32_e64 v154, v154, %19, %8\n\t"
            SV_MOVS("row_half_mirror") SV_MINS
            "v_cndmask_b32_e64 v146, v146, %18, %4\n\t"
            "v_cndmask_b32_e64 v154, v154, %18, %7\n\t"
            SV_MOVS("row_mirror") SV_MINS
            "v_cmp_eq_f64_e64 %2, v[144:145], v[150:151]\n\t"
            "v_cmp_eq_f64_e64 %3, v[152:153], v[158:159]"
            : "=&{v[144:147]}"(rec_x), "=&{v[152:155]}"(rec_y), "=&s"(has_x), "=&s"(has_y), "=&s"(x0), "=&s"(x1), "=&s"(x2), "=&s"(y0), "=&s"(y1), "=&s"(y2)
            : "v"(x[0]), "v"(x[1]), "v"(x[2]), "v"(x[3]), "v"(y[0]), "v"(y[1]), "v"(y[2]), "v"(y[3]), "v"(at[0]), "v"(at[1]), "v"(at[2]), "v"(at[3])
            : "v148", "v149", "v150", "v151", "v156", "v157", "v158", "v159");
    } else {
        static_assert(E == 2, "elements per thread");
        asm("v_min_f64 v[144:145], %6, %7\n\t"
            "v_min_f64 v[152:153], %8, %9\n\t"
            "v_cmp_eq_f64_e64 %4, %6, v[144:145]\n\t"
            "v_cmp_eq_f64_e64 %5, %8, v[152:153]\n\t"
            SV_FIRST_MOVS("quad_perm:[1,0,3,2]")
            "v_cndmask_b32_e64 v146, %11, %10, %4\n\t"
            SV_MOVS("quad_perm:[2,3,0,1]") SV_MINS
            "v_cndmask_b32_e64 v154, %11, %10, %5\n\t"
            SV_MOVS("row_half_mirror") SV_MINS
            "s_nop 0\n\t" SV_MOVS("row_mirror") SV_MINS
            "v_cmp_eq_f64_e64 %2, v[144:145], v[150:151]\n\t"
            "v_cmp_eq_f64_e64 %3, v[152:153], v[158:159]"
            : "=&{v[144:147]}"(rec_x), "=&{v[152:155]}"(rec_y), "=&s"(has_x), "=&s"(has_y), "=&s"(x0), "=&s"(y0)
            : "v"(x[0]), "v"(x[1]), "v"(y[0]), "v"(y[1]), "v"(at[0]), "v"(at[1])
            : "v148", "v149", "v150", "v151", "v156", "v157", "v158", "v159");
    }
}
__device__ __forceinline__ void row_mins_and_who(double x, double y, double &min_x, double &min_y, uint64_t &who_x, uint64_t &who_y) {
    const double s = dpp_f64<TSVM_DPP_XOR1>(x), t = dpp_f64<TSVM_DPP_XOR1>(y);
    asm("v_min_f64 v[150:151], %4, %5\n\t"
        "v_min_f64 v[158:159], %6, %7\n\t"
        "s_nop 0\n\t" SV_MOVS("quad_perm:[2,3,0,1]") SV_MINS
        "s_nop 0\n\t" SV_MOVS("row_half_mirror") SV_MINS
        "s_nop 0\n\t" SV_MOVS("row_mirror")
        "v_min_f64 %0, v[150:151], v[148:149]\n\t"
        "v_min_f64 %1, v[158:159], v[156:157]\n\t"
        "v_cmp_eq_f64_e64 %2, %4, %0\n\t"
        "v_cmp_eq_f64_e64 %3, %6, %1"
        : "=&v"(min_x), "=&v"(min_y), "=&s"(who_x), "=&s"(who_y) : "v"(x), "v"(s), "v"(y), "v"(t)
        : "v148", "v149", "v150", "v151", "v156", "v157", "v158", "v159");
}
// The smallest of a row's x in all its lanes, and the lanes that have it.  LANES: of so many lanes that hold different ones.
template <int LANES = 16>
__device__ __forceinline__ void row_min_and_who(double x, double &value, uint64_t &who) {
    const double t = dpp_f64<TSVM_DPP_XOR1>(x);
    static_assert(LANES == 8 || LANES == 16, "half a row, a row");
    if constexpr (LANES == 8)
        asm("v_min_f64 v[150:151], %2, %3\n\t"
            "s_nop 1\n\t" SV_MIN_STEP("quad_perm:[2,3,0,1]")
            "s_nop 1\n\t" SV_DPP_MOV("v148", "v150", "row_half_mirror") SV_DPP_MOV("v149", "v151", "row_half_mirror")
            "v_min_f64 %0, v[150:151], v[148:149]\n\t"
            "v_cmp_eq_f64_e64 %1, %2, %0"
            : "=&v"(value), "=s"(who) : "v"(x), "v"(t) : "v148", "v149", "v150", "v151");
    else asm("v_min_f64 v[150:151], %2, %3\n\t"
        "s_nop 1\n\t" SV_MIN_STEP("quad_perm:[2,3,0,1]")
        "s_nop 1\n\t" SV_MIN_STEP("row_half_mirror")
        "s_nop 1\n\t" SV_DPP_MOV("v148", "v150", "row_mirror") SV_DPP_MOV("v149", "v151", "row_mirror")
        "v_min_f64 %0, v[150:151], v[148:149]\n\t"
        "v_cmp_eq_f64_e64 %1, %2, %0"
        : "=&v"(value), "=s"(who) : "v"(x), "v"(t) : "v148", "v149", "v150", "v151");
}
// The lowest lane of every row among those that are set; the last one where none is (whatever is NaN).
__device__ __forceinline__ uint64_t lowest_of_rows(uint64_t lanes) {
    lanes |= 0x8000800080008000ull;
    return lanes & ~(lanes - 0x0001000100010001ull);
}
// The smallest of four wavefronts' E * 256 values and the number of the first element that has it, over sixteen rows of lanes; `flag`
// comes back as whether any row's was set.  also: writes by the rows' candidates, by their lanes, in front of the barrier.
template <int E, typename F>
__device__ __forceinline__ void block_first_min(SvCand *slots, const double (&x)[E], const int (&at)[E], int flag, F also, double &value, int &first, int &any) {
    SvWords rec;
    uint64_t has, who;
    row_first_candidate<E>(x, at, rec, has);
    const uint64_t lanes = lowest_of_rows(has);
    also(lanes);
    rec[3] = flag;
    publish_words(lds_at(slots + (threadIdx.x >> 4)), lanes, rec);
    lds_barrier();
    const SvCand c = slots[threadIdx.x & 15];
    row_min_and_who(c.v, value, who);
    first = __builtin_amdgcn_readlane(c.at, __builtin_ctzll(who));
    any = __builtin_amdgcn_ballot_w64(c.flag != 0) != 0;
}
template <int E, typename F>
__device__ __forceinline__ void block_first_mins(SvCand *slots_x, SvCand *slots_y, const double (&x)[E], const double (&y)[E], const int (&at)[E], int flag, F also,
                                                 double &min_x, double &min_y, int &first_x, int &first_y, int &any) {
    SvWords rec_x, rec_y;
    uint64_t has_x, has_y, who_x, who_y;
    row_first_candidates<E>(x, y, at, rec_x, rec_y, has_x, has_y);
    const uint64_t lanes_x = lowest_of_rows(has_x), lanes_y = lowest_of_rows(has_y);
    also(lanes_x, lanes_y);
    rec_x[3] = flag;
    publish_words(lds_at(slots_x + (threadIdx.x >> 4)), lanes_x, rec_x);
    publish_words(lds_at(slots_y + (threadIdx.x >> 4)), lanes_y, rec_y);
    lds_barrier();
    const SvCand cx = slots_x[threadIdx.x & 15], cy = slots_y[threadIdx.x & 15];
    row_mins_and_who(cx.v, cy.v, min_x, min_y, who_x, who_y);
    first_x = __builtin_amdgcn_readlane(cx.at, __builtin_ctzll(who_x));
    first_y = __builtin_amdgcn_readlane(cy.at, __builtin_ctzll(who_y));
    any = __builtin_amdgcn_ballot_w64(cx.flag != 0) != 0;
}
// Best and second of a row in all its lanes, and the lanes that have the best.  Four instructions per step, ordered so that none of the
// DPP operands is younger than two instructions: no wait states between the steps, so the second-best costs hardly more than the
// waits would.
template <int LANES = 16>
__device__ __forceinline__ void row_best_two_and_who(float mine, float second_in, float &best, float &second, uint64_t &who) {
    float t;
#define SV_BEST_STEP(CTRL, B, S)                                          \
    "v_min_f32_dpp %2, " B ", " B " " CTRL " row_mask:0xf bank_mask:0xf\n\t" \
    "v_max_f32_dpp %0, " B ", " B " " CTRL " row_mask:0xf bank_mask:0xf\n\t" \
    "v_max_f32_dpp %1, " S ", " S " " CTRL " row_mask:0xf bank_mask:0xf\n\t" \
    "v_max_f32 %1, %1, %2\n\t"
    static_assert(LANES == 8 || LANES == 16, "half a row, a row");
    if constexpr (LANES == 8)
        asm("s_nop 1\n\t" SV_BEST_STEP("quad_perm:[1,0,3,2]", "%4", "%5") SV_BEST_STEP("quad_perm:[2,3,0,1]", "%0", "%1")
                SV_BEST_STEP("row_half_mirror", "%0", "%1")
            "v_cmp_eq_f32_e64 %3, %4, %0"
            : "=&v"(best), "=&v"(second), "=&v"(t), "=s"(who) : "v"(mine), "v"(second_in));
    else asm("s_nop 1\n\t" SV_BEST_STEP("quad_perm:[1,0,3,2]", "%4", "%5") SV_BEST_STEP("quad_perm:[2,3,0,1]", "%0", "%1")
            SV_BEST_STEP("row_half_mirror", "%0", "%1") SV_BEST_STEP("row_mirror", "%0", "%1")
        "v_cmp_eq_f32_e64 %3, %4, %0"
        : "=&v"(best), "=&v"(second), "=&v"(t), "=s"(who) : "v"(mine), "v"(second_in));
#undef SV_BEST_STEP
}
// Bounds of what c_smo_iterate_rounded (smo_solve.hip) decides: the least |up|, and from where on an a is too large (as float bits).
#define SV_UP_LEAST_HI 0x3b600000   // 2^-73
#define SV_UP_LEAST 0x1p-73
#define SV_A_BITS 0x7e800000         // 2^126
