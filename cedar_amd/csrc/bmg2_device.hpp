// Device functions shared by the 2D kernels: point formulas, wavefront scans of the line solves,
// transfers of one point and the coarsest band solve.  Layout and numerics as described in
// bmg2_kernels.hip; every file that includes this is built with -ffp-contract=off, so a formula
// rounds the same wherever it is used.
#pragma once

#include "band_chol.hpp"
#include "bmg2_launch.hpp"

#include <hip/hip_runtime.h>

#include <cstddef>

namespace cdr {
namespace k2 {

constexpr int WAVE = 64;

__host__ __device__ inline std::size_t pidx(int i, int j, int ii) {
    return (std::size_t)j * (std::size_t)ii + (std::size_t)i;
}

// ------------------------------------------------------------------------------------------
// deterministic block reduction of one double per thread (256 threads = 4 waves)
// ------------------------------------------------------------------------------------------
__device__ inline double wave_sum(double v) {
#pragma unroll
    for (int off = WAVE / 2; off > 0; off >>= 1) v += __shfl_xor(v, off, WAVE);
    return v;
}

// barrier that orders LDS only: prefetched global loads stay in flight across it
__device__ inline void lds_barrier() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// LDS_ONLY: the barrier orders LDS alone (global loads issued before it stay in flight)
template <int NWAVES = 4, bool LDS_ONLY = false>
__device__ inline void block_sum_store(double v, double *dst) {
    __shared__ double part[NWAVES];
    v = wave_sum(v);
    int lane = threadIdx.x % WAVE, wid = threadIdx.x / WAVE;
    if (lane == 0) part[wid] = v;
    if (LDS_ONLY)
        lds_barrier();
    else
        __syncthreads();
    if (threadIdx.x == 0) {
        double t = part[0];
        for (int w = 1; w < NWAVES; ++w) t += part[w];
        *dst = t;
    }
}

// Left to itself the compiler issues the operands of a long sum a few at a time and waits in
// between.  Where a launch is short (every level of at most 512 points a side) those waits are its
// whole time, so the point functions below issue all loads before the first product
// (loads_issued): a 511^2 Poisson solve 1.91 -> 1.84 ms, the 27-point FP32 residual at
// 127 x 127 x 95 15.2 -> 8.2 us.
__device__ inline void loads_issued() { __builtin_amdgcn_sched_barrier(0); }

// f + the couplings of point p to its neighbours, in the reference's order
// (src/2d/ftn/BMG2_SymStd_residual.f90:85-119)
template <typename T, bool NINE>
__device__ inline T apply_offdiag(const T *__restrict__ so, std::size_t P, const T *__restrict__ q,
                                  std::size_t p, int ii, T acc) {
    const T w0 = so[P * KW + p], w1 = so[P * KW + p + 1];
    const T s0 = so[P * KS + p], s1 = so[P * KS + p + ii];
    const T qw = q[p - 1], qe = q[p + 1], qs = q[p - ii], qn = q[p + ii];
    if constexpr (NINE) {
        const T sw0 = so[P * KSW + p], nw0 = so[P * KNW + p + 1];
        const T nw1 = so[P * KNW + p + ii], sw1 = so[P * KSW + p + ii + 1];
        const T qsw = q[p - ii - 1], qse = q[p - ii + 1], qnw = q[p + ii - 1], qne = q[p + ii + 1];
        loads_issued();
        acc = acc + w0 * qw;
        acc = acc + w1 * qe;
        acc = acc + s0 * qs;
        acc = acc + s1 * qn;
        acc = acc + sw0 * qsw;
        acc = acc + nw0 * qse;
        acc = acc + nw1 * qnw;
        acc = acc + sw1 * qne;
    } else {
        loads_issued();
        acc = acc + w0 * qw;
        acc = acc + w1 * qe;
        acc = acc + s0 * qs;
        acc = acc + s1 * qn;
    }
    return acc;
}

// Inclusive scans of affine maps y -> a*y + b across the 64 lanes of a wavefront.
// up:   lane l gets F_l o F_{l-1} o ... o F_0        (forward substitution)
// down: lane l gets G_l o G_{l+1} o ... o G_63       (backward substitution)
template <typename T>
__device__ inline void scan_affine_up(T &a, T &b, int lane) {
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const T ap = __shfl_up(a, d, WAVE);
        const T bp = __shfl_up(b, d, WAVE);
        if (lane >= d) {
            b = a * bp + b;
            a = a * ap;
        }
    }
}

template <typename T>
__device__ inline void scan_affine_down(T &a, T &b, int lane) {
#pragma unroll
    for (int d = 1; d < WAVE; d <<= 1) {
        const T an = __shfl_down(a, d, WAVE);
        const T bn = __shfl_down(b, d, WAVE);
        if (lane + d < WAVE) {
            b = a * bn + b;
            a = a * an;
        }
    }
}

// Same inclusive scan with DPP lane moves (row_shr 1/2/4/8 inside 16-lane rows, then
// row_bcast 15 and 31 across rows) instead of LDS permutes: a few cycles per step, which keeps
// the carry chain of a line short.  Lanes whose source is out of range keep the identity (1, 0).
template <int CTRL, int RMASK>
__device__ inline float dpp_move(float v, float ident) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, ident),
                                                                 __builtin_bit_cast(int, v), CTRL,
                                                                 RMASK, 0xF, false));
}

template <int CTRL, int RMASK>
__device__ inline double dpp_move(double v, double ident) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned long long o = __builtin_bit_cast(unsigned long long, ident);
    const int lo = __builtin_amdgcn_update_dpp((int)(unsigned)o, (int)(unsigned)u, CTRL, RMASK, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(unsigned)(o >> 32), (int)(unsigned)(u >> 32), CTRL,
                                               RMASK, 0xF, false);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// The affine step a * c + b of the line recurrences: a fused multiply-add in FP32 (the
// preconditioning V-cycle of the mixed solver), separate rounding in FP64.  Every line kernel
// evaluates its recurrences through this one function, so all of them (every launch shape, the
// direct and the transposed y sweeps, the fused coarse cycle) still round identically.
__device__ inline float affine(float a, float c, float b) { return __builtin_fmaf(a, c, b); }
__device__ inline double affine(double a, double c, double b) { return a * c + b; }
// y / d for a line pivot d: FP32 multiplies by the hardware reciprocal (about 1 ulp), FP64
// divides (correctly rounded, as the sequential substitution does).
__device__ inline float div_pivot(float y, float d) { return y * __builtin_amdgcn_rcpf(d); }
__device__ inline double div_pivot(double y, double d) { return y / d; }

// the source lane's value, 0 where the source lane is out of range or the row is masked off
template <int CTRL, int RMASK>
__device__ inline float dpp_zero(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v),
                                                                 CTRL, RMASK, 0xF, true));
}
template <int CTRL, int RMASK>
__device__ inline double dpp_zero(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)u, CTRL, RMASK, 0xF, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(u >> 32), CTRL, RMASK, 0xF, true);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

// lanes that receive a value in each step of the scan (row_shr:1/2/4/8 within 16-lane rows,
// row_bcast:15 into rows 1 and 3, row_bcast:31 into rows 2 and 3); the others keep (a, b)
__device__ inline int lane_id() { return __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u)); }
template <int STEP>
__device__ inline bool dpp_valid(int lane) {
    return STEP == 0 ? (lane & 15) >= 1 : STEP == 1 ? (lane & 15) >= 2 : STEP == 2 ? (lane & 15) >= 4
         : STEP == 3 ? (lane & 15) >= 8 : STEP == 4 ? ((lane >> 4) & 1) != 0 : lane >= 32;
}

// One step: (a, b) <- (a * a', a * b' + b) with (a', b') from the source lane.  Where no value
// arrives, b' reads 0 (a * 0 + b = b exactly) and a is kept: the identity map.  The product
// a * b' is rounded on its own in both precisions (a multiply that takes its lane move for free
// is cheaper here than a fused multiply-add, which cannot).
// The broadcast steps move data into every row (row 0 reads 0); the lanes outside the rows the
// step feeds are then restored by the select, as the row_shr steps restore a.
template <int CTRL, int STEP, typename T>
__device__ inline void dpp_scan_step(T &a, T &b, int lane) {
    const T ap = dpp_zero<CTRL, 0xF>(a);
    const T bp = dpp_zero<CTRL, 0xF>(b);
    const bool v = dpp_valid<STEP>(lane);
    const T bn = a * bp + b;
    b = (STEP < 4 || v) ? bn : b;
    a = v ? a * ap : a;
}

template <typename T>
__device__ inline void scan_affine_dpp(T &a, T &b) {
    const int lane = lane_id();
    dpp_scan_step<0x111, 0>(a, b, lane);  // row_shr:1
    dpp_scan_step<0x112, 1>(a, b, lane);  // row_shr:2
    dpp_scan_step<0x114, 2>(a, b, lane);  // row_shr:4
    dpp_scan_step<0x118, 3>(a, b, lane);  // row_shr:8
    dpp_scan_step<0x142, 4>(a, b, lane);  // row_bcast:15, kept in rows 1 and 3
    dpp_scan_step<0x143, 5>(a, b, lane);  // row_bcast:31, kept in rows 2 and 3
}

// scan_affine_dpp over each group of w = 16, 32 or 64 lanes (w is the same in every lane)
template <typename T>
__device__ inline void scan_affine_rows(T &a, T &b, int w) {
    const int lane = lane_id();
    dpp_scan_step<0x111, 0>(a, b, lane);
    dpp_scan_step<0x112, 1>(a, b, lane);
    dpp_scan_step<0x114, 2>(a, b, lane);
    dpp_scan_step<0x118, 3>(a, b, lane);
    if (w > 16) dpp_scan_step<0x142, 4>(a, b, lane);
    if (w > 32) dpp_scan_step<0x143, 5>(a, b, lane);
}

// the multiplier part of scan_affine_dpp alone (the same products in the same order)
template <int CTRL, int STEP, typename T>
__device__ inline void dpp_prod_step(T &a, int lane) {
    const T ap = dpp_zero<CTRL, 0xF>(a);
    a = dpp_valid<STEP>(lane) ? a * ap : a;
}

template <typename T>
__device__ inline void scan_prod_dpp(T &a) {
    const int lane = lane_id();
    dpp_prod_step<0x111, 0>(a, lane);
    dpp_prod_step<0x112, 1>(a, lane);
    dpp_prod_step<0x114, 2>(a, lane);
    dpp_prod_step<0x118, 3>(a, lane);
    dpp_prod_step<0x142, 4>(a, lane);
    dpp_prod_step<0x143, 5>(a, lane);
}

// value of lane 63, broadcast (v_readlane: no LDS round trip)
__device__ inline float last_lane(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), WAVE - 1));
}
__device__ inline double last_lane(double v) {
    const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)u, WAVE - 1);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(u >> 32), WAVE - 1);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// raw operands of the right-hand side of one point of a line
template <typename T>
struct line_raw {
    T qf, s0, q0, s1, q1, sw0, q0m, nw0, q0p, nw1, q1m, sw1, q1p;
};

// Right-hand side of one point in the reference's order.  X-lines: s0/q0 = coupling to the row
// below, s1/q1 = to the row above; y-lines: the column to the left / right.
// SWAP adds the two NW terms in the opposite order: an x-line of the transposed grid then sums
// its terms in exactly the order of the corresponding y-line of the original grid.
template <typename T, bool NINE, bool SWAP = false>
__device__ inline T line_rhs(const line_raw<T> &r) {
    T rhs = r.qf;
    rhs = affine(r.s0, r.q0, rhs);
    rhs = affine(r.s1, r.q1, rhs);
    if (NINE) {
        rhs = affine(r.sw0, r.q0m, rhs);
        if (SWAP) {
            rhs = affine(r.nw1, r.q1m, rhs);
            rhs = affine(r.nw0, r.q0p, rhs);
        } else {
            rhs = affine(r.nw0, r.q0p, rhs);
            rhs = affine(r.nw1, r.q1m, rhs);
        }
        rhs = affine(r.sw1, r.q1p, rhs);
    }
    return rhs;
}

// loads the operands of point p (array index) of an x-line (DIR 0) or y-line (DIR 1)
template <typename T, bool NINE, int DIR>
__device__ inline void line_load(line_raw<T> &r, const T *__restrict__ so, const T *__restrict__ qf,
                                 const T *__restrict__ q, std::size_t P, int ii, std::size_t p,
                                 bool zq = false) {
    r.qf = qf[p];
    if (DIR == 0) {
        r.s0 = so[P * KS + p];
        r.q0 = zq ? T(0) : q[p - ii];
        r.s1 = so[P * KS + p + ii];
        r.q1 = zq ? T(0) : q[p + ii];
    } else {
        r.s0 = so[P * KW + p];
        r.q0 = zq ? T(0) : q[p - 1];
        r.s1 = so[P * KW + p + 1];
        r.q1 = zq ? T(0) : q[p + 1];
    }
    if (NINE) {
        r.sw0 = so[P * KSW + p];
        r.q0m = zq ? T(0) : q[p - ii - 1];
        r.nw0 = so[P * KNW + p + 1];
        r.q0p = zq ? T(0) : q[p - ii + 1];
        r.nw1 = so[P * KNW + p + ii];
        r.q1m = zq ? T(0) : q[p + ii - 1];
        r.sw1 = so[P * KSW + p + ii + 1];
        r.q1p = zq ? T(0) : q[p + ii + 1];
    }
}

// coarse point (ic, jc) of qc = P^T q (the reference's operation order); ci, q, qc of one problem
template <typename T>
struct restrict_ops {
    T w[8], q[9];
};
template <typename T>
__device__ inline void load_restrict(restrict_ops<T> &o, const T *__restrict__ ci,
                                     const T *__restrict__ q, int iif, int iic, std::size_t Pc,
                                     int ic, int jc) {
    const int i = 2 * ic - 1, j = 2 * jc - 1;
    auto CI = [&](int a, int b, int k) { return ci[Pc * k + pidx(a, b, iic)]; };
    auto Q = [&](int a, int b) { return q[pidx(a, b, iif)]; };
    o.w[0] = CI(ic, jc, LNE), o.q[0] = Q(i - 1, j - 1);
    o.w[1] = CI(ic, jc, LA), o.q[1] = Q(i, j - 1);
    o.w[2] = CI(ic + 1, jc, LNW), o.q[2] = Q(i + 1, j - 1);
    o.w[3] = CI(ic, jc, LR), o.q[3] = Q(i - 1, j);
    o.q[8] = Q(i, j);
    o.w[4] = CI(ic + 1, jc, LL), o.q[4] = Q(i + 1, j);
    o.w[5] = CI(ic, jc + 1, LSE), o.q[5] = Q(i - 1, j + 1);
    o.w[6] = CI(ic, jc + 1, LB), o.q[6] = Q(i, j + 1);
    o.w[7] = CI(ic + 1, jc + 1, LSW), o.q[7] = Q(i + 1, j + 1);
}
template <typename T>
__device__ inline T sum_restrict(const restrict_ops<T> &o) {
    T v = o.w[0] * o.q[0];
    v = v + o.w[1] * o.q[1];
    v = v + o.w[2] * o.q[2];
    v = v + o.w[3] * o.q[3];
    v = v + o.q[8];
    v = v + o.w[4] * o.q[4];
    v = v + o.w[5] * o.q[5];
    v = v + o.w[6] * o.q[6];
    v = v + o.w[7] * o.q[7];
    return v;
}
template <typename T>
__device__ inline T restrict_point(const T *__restrict__ ci, const T *__restrict__ q, int iif,
                                   int iic, std::size_t Pc, int ic, int jc) {
    restrict_ops<T> o;
    load_restrict(o, ci, q, iif, iic, Pc, ic, jc);
    loads_issued();
    return sum_restrict(o);
}

// One 2 x 2 block of fine points (2m-1 .. 2m, 2n-1 .. 2n) of interp_add: the coarse point
// (m, n), the x-edge point (2m, 2n-1), the y-edge point (2m-1, 2n) and the cell point (2m, 2n),
// sharing the four coarse values around the cell.  Arrays of one problem.
// Two adjacent floats moved by one 8-byte access.  On this GPU an 8-byte global access needs only
// 4-byte alignment, so a pair may start at any float (rows of odd length included).
struct __attribute__((aligned(4))) float_pair {
    float a, b;
};
__device__ inline void load_pair(const float *p, float &a, float &b) {
    float_pair v;
    __builtin_memcpy(&v, p, sizeof(v));
    a = v.a;
    b = v.b;
}
__device__ inline void store_pair(float *p, float a, float b) {
    const float_pair v{a, b};
    __builtin_memcpy(p, &v, sizeof(v));
}

// PAIRS: in FP32, blocks inside the grid move horizontally adjacent values as pairs.
template <typename T, bool PAIRS = true>
__device__ inline void interp_block(T *__restrict__ q, const T *__restrict__ qc,
                                    const T *__restrict__ res, const T *__restrict__ so,
                                    const T *__restrict__ ci, int iic, int jjc, int iif, int jjf,
                                    int m, int n) {
    const int imax = iif - 2 + ((iif - 2) % 2 == 0 ? 1 : 0);
    const int jmax = jjf - 2 + ((jjf - 2) % 2 == 0 ? 1 : 0);
    const int i0 = 2 * m - 1, j0 = 2 * n - 1;
    if (i0 > imax || j0 > jmax) return;
    const bool xe = i0 + 1 <= imax, ye = j0 + 1 <= jmax;  // the even fine points exist
    const std::size_t Pc = (std::size_t)iic * jjc;
    auto CI = [&](int a, int b, int k) { return ci[Pc * k + pidx(a, b, iic)]; };
    auto QC = [&](int a, int b) { return qc[pidx(a, b, iic)]; };
    if constexpr (PAIRS && sizeof(T) == 4) {
        if (xe && ye && i0 + 1 <= iif - 2 && j0 + 1 <= jjf - 2) {
            const std::size_t p = pidx(i0, j0, iif), p2 = p + iif;
            T q0, q1, q2, q3, c00, c10, c01, c11, r2, r3, s2, s3;
            load_pair(qc + pidx(m, n, iic), c00, c10);
            load_pair(qc + pidx(m, n + 1, iic), c01, c11);
            load_pair(q + p, q0, q1);
            load_pair(q + p2, q2, q3);
            load_pair(res + p2, r2, r3);
            load_pair(so + p2, s2, s3);
            const T r1 = res[p + 1], s1 = so[p + 1];
            const T wr = CI(m + 1, n, LR), wl = CI(m + 1, n, LL);
            const T wa = CI(m, n + 1, LA), wb = CI(m, n + 1, LB);
            const T wsw = CI(m + 1, n + 1, LSW), wnw = CI(m + 1, n + 1, LNW);
            const T wne = CI(m + 1, n + 1, LNE), wse = CI(m + 1, n + 1, LSE);
            loads_issued();
            q0 = q0 + c00;
            const T a = wr * c10 + wl * c00;
            q1 = q1 + a + r1 / s1;
            const T b = wa * c01 + wb * c00;
            q2 = q2 + b + r2 / s2;
            T c = wsw * c00;
            c = c + wnw * c01;
            c = c + wne * c11;
            c = c + wse * c10;
            q3 = q3 + c + r3 / s3;
            store_pair(q + p, q0, q1);
            store_pair(q + p2, q2, q3);
            return;
        }
    }
    // where a point does not exist, its operands are those of its neighbour in the block and its
    // result is dropped, so that all loads come before the first branch
    const int mx = m + (xe ? 1 : 0), ny = n + (ye ? 1 : 0);
    const std::size_t p0 = pidx(i0, j0, iif), p1 = p0 + (xe ? 1 : 0);
    const std::size_t p2 = p0 + (ye ? iif : 0), p3 = p2 + (xe ? 1 : 0);
    const T c00 = QC(m, n), c10 = QC(mx, n), c01 = QC(m, ny), c11 = QC(mx, ny);
    T q0 = q[p0], q1 = q[p1], q2 = q[p2], q3 = q[p3];
    const T r2 = res[p2], r3 = res[p3], s2 = so[p2], s3 = so[p3];
    const T r1 = res[p1], s1 = so[p1];
    const T wr = CI(mx, n, LR), wl = CI(mx, n, LL);
    const T wa = CI(m, ny, LA), wb = CI(m, ny, LB);
    const T wsw = CI(mx, ny, LSW), wnw = CI(mx, ny, LNW);
    const T wne = CI(mx, ny, LNE), wse = CI(mx, ny, LSE);
    loads_issued();
    // a ghost point reached by an even extent takes the raw res
    auto R = [&](int i, int j, T r, T s) { return (i > iif - 2 || j > jjf - 2) ? r : r / s; };
    q0 = q0 + c00;  // coarse point
    const T a = wr * c10 + wl * c00;  // (2m, 2n-1): between coarse (m, n) and (m+1, n)
    q1 = q1 + a + R(i0 + 1, j0, r1, s1);
    const T b = wa * c01 + wb * c00;  // (2m-1, 2n): between coarse (m, n) and (m, n+1)
    q2 = q2 + b + R(i0, j0 + 1, r2, s2);
    T c = wsw * c00;  // (2m, 2n): the cell of coarse (m..m+1, n..n+1)
    c = c + wnw * c01;
    c = c + wne * c11;
    c = c + wse * c10;
    q3 = q3 + c + R(i0 + 1, j0 + 1, r3, s3);
    q[p0] = q0;
    if (xe) q[p1] = q1;
    if (ye) q[p2] = q2;
    if (xe && ye) q[p3] = q3;
}

// The coarsest level's band solve, q = A^-1 qf, by the threads tid < nt of one workgroup.  Where
// the factor (ld * n) and the iterate (n) fit in CG_LDS doubles (sh), both are staged into LDS and
// one wavefront runs the two triangular sweeps (4x4 coarsest grid of the 4095^2 hierarchy: 25 us
// per solve through memory); otherwise one thread runs them with the iterate in the global scratch
// x.  Same operations either way.  staged: coarse_band_stage has filled sh, and a barrier has
// passed since.
constexpr int CG_LDS = 1024;
__device__ inline bool coarse_band_fits(int ii, int n) {
    return (std::size_t)n * (ii + 1) <= (std::size_t)CG_LDS;
}
__device__ inline void coarse_band_stage(const double *abd, int ii, int jj, int tid, int nt, double *sh) {
    const int n = (ii - 2) * (jj - 2);
    if (coarse_band_fits(ii, n))
        for (int k = tid; k < ii * n; k += nt) sh[n + k] = abd[k];
}
template <typename T>
__device__ inline void coarse_band_solve(T *q, const T *qf, const double *abd, double *x, int ii,
                                         int jj, int tid, int nt, double *sh, bool staged = false) {
    const int nx = ii - 2, ny = jj - 2, n = nx * ny, kd = ii - 1, ld = ii;
    const bool lds = coarse_band_fits(ii, n);
    if (lds && !staged) coarse_band_stage(abd, ii, jj, tid, nt, sh);
    if (lds && n <= WAVE && kd < WAVE && nt >= WAVE) {
        if (!staged) __syncthreads();
        if (tid < WAVE) {
            const bool own = tid < n;
            const std::size_t p = own ? pidx(tid % nx + 1, tid / nx + 1, ii) : 0;
            const double v = band_solve_upper_regs(sh + n, n, kd, ld, own ? (double)qf[p] : 0.0, tid);
            if (own) q[p] = (T)v;
        }
        return;
    }
    double *xx = lds ? sh : x;
    const double *ab = lds ? sh + n : abd;
    for (int kk = tid; kk < n; kk += nt) xx[kk] = (double)qf[pidx(kk % nx + 1, kk / nx + 1, ii)];
    __syncthreads();
    if (lds && kd < WAVE && nt >= WAVE) {  // bitwise the same sweeps, one wavefront
        if (tid < WAVE) band_solve_upper_wave(ab, n, kd, ld, xx, tid);
    } else if (tid == 0) {
        band_solve_upper(ab, n, kd, ld, xx);
    }
    __syncthreads();
    for (int kk = tid; kk < n; kk += nt) q[pidx(kk % nx + 1, kk / nx + 1, ii)] = (T)xx[kk];
}

}  // namespace k2
}  // namespace cdr
