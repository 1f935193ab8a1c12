// Line relaxation of the 2D path (src/2d/ftn/BMG2_SymStd_relax_lines_{x,y}.f90): segmented scan
// kernels, the autotuner of their launch shapes, and y sweeps through the transposed grid.  Layout
// and batching as in bmg2_kernels.hip.
#include "../../include/cedar_hip.h"
#include "bmg2_device.hpp"
#include "bmg2_launch.hpp"
#include "tile_order.hpp"

#include <hip/hip_runtime.h>

#include <array>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

namespace cdr {
namespace k2 {

namespace {

// One wavefront solves one line: L D L^T x = rhs with the stored factors.  Forward pass in
// 64-element chunks: y_k = rhs_k - E_{k-1} y_{k-1}, stores c_k = y_k / D_k in place of q;
// backward pass: x_k = c_k - E_k x_{k+1}.  A line of one colour only reads lines of the other
// colour, so the in-place staging is race free.
//
// DIR 0: x-lines (row j = first + 2*line, elements along i, unit stride)
// DIR 1: y-lines (column i = first + 2*line, elements along j, stride ii; factors transposed)
template <typename T, bool NINE, int DIR>
__global__ __launch_bounds__(256) void relax_lines_k(const T *__restrict__ so, const T *__restrict__ qf,
                                                     T *__restrict__ q, const T *__restrict__ sor,
                                                     int ii, int jj, int first, int nlines, int rep) {
    const int lane = threadIdx.x % WAVE;
    int bx = (int)blockIdx.x, prob = (int)blockIdx.y;
    shared_op_order((int)gridDim.x, rep, bx, prob);
    const int line = bx * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (line >= nlines) return;  // whole wavefront leaves together; no block barrier below
    const std::size_t P = (std::size_t)ii * jj, bz = prob, bo = operator_of(bz, rep);
    so += bo * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    sor += bo * 2 * P;
    const int fixed = first + 2 * line;
    const int n = (DIR == 0) ? ii - 2 : jj - 2;
    const std::size_t stride = (DIR == 0) ? 1 : (std::size_t)ii;
    const std::size_t base = (DIR == 0) ? pidx(1, fixed, ii) : pidx(fixed, 1, ii);  // element 0
    const T *D = (DIR == 0) ? sor + pidx(1, fixed, ii) : sor + (std::size_t)fixed * jj + 1;
    const T *E = (DIR == 0) ? sor + P + pidx(2, fixed, ii) : sor + P + (std::size_t)fixed * jj + 2;
    const int nch = (n + WAVE - 1) / WAVE;

    T carry = T(0);
    for (int c = 0; c < nch; ++c) {
        const int k = c * WAVE + lane;
        const bool act = k < n;
        T a = T(0), b = T(0);
        if (act) {
            const std::size_t p = base + (std::size_t)k * stride;
            T rhs = qf[p];
            if (DIR == 0) {
                rhs = rhs + so[P * KS + p] * q[p - ii];
                rhs = rhs + so[P * KS + p + ii] * q[p + ii];
            } else {
                rhs = rhs + so[P * KW + p] * q[p - 1];
                rhs = rhs + so[P * KW + p + 1] * q[p + 1];
            }
            if (NINE) {
                rhs = rhs + so[P * KSW + p] * q[p - ii - 1];
                rhs = rhs + so[P * KNW + p + 1] * q[p - ii + 1];
                rhs = rhs + so[P * KNW + p + ii] * q[p + ii - 1];
                rhs = rhs + so[P * KSW + p + ii + 1] * q[p + ii + 1];
            }
            b = rhs;
            a = (k > 0) ? -E[k - 1] : T(0);
        }
        scan_affine_up(a, b, lane);
        const T y = affine(a, carry, b);
        carry = __shfl(y, WAVE - 1, WAVE);
        if (act) q[base + (std::size_t)k * stride] = div_pivot(y, D[k]);
    }
    carry = T(0);
    for (int c = nch - 1; c >= 0; --c) {
        const int k = c * WAVE + lane;
        const bool act = k < n;
        T a = T(1), b = T(0);
        if (act) {
            b = q[base + (std::size_t)k * stride];
            a = (k < n - 1) ? -E[k] : T(0);
        }
        scan_affine_down(a, b, lane);
        const T x = affine(a, carry, b);
        carry = __shfl(x, 0, WAVE);
        if (act) q[base + (std::size_t)k * stride] = x;
    }
}

// Workgroup index remapped so that consecutive logical tiles run on the same XCD (workgroups
// are dealt round-robin over the 8 XCDs): neighbouring lines share rows of q and of the
// operator, which then stay in one XCD's L2.  Launch 8 * ceil(ntiles / 8) workgroups.
// rev: each XCD walks its range of tiles from the end, so that a launch starts on the lines the
// previous launch touched last (still in the memory-side cache); the work is unchanged.
__device__ inline int xcd_tile(int bx, int ntiles, int rev = 0) {
    const int per = (ntiles + 7) / 8;
    const int k = bx / 8;
    return (bx % 8) * per + (rev ? per - 1 - k : k);
}

// ------------------------------------------------------------------------------------------
// Segmented line solves.  W wavefronts share a line: wavefront w owns the CPW chunks
// [w*CPW, (w+1)*CPW) of 64 elements.  Every operand of a wavefront's chunks is loaded before the
// first scan, so no load latency sits inside the carry chain, and at most CPW chunks live in
// registers; W wavefronts per line put W times as many wavefronts in flight as there are lines.
//
// The carries between chunks are evaluated in exactly the single-wavefront order: chunk m's
// scanned map (a_m, b_m) at its last element goes to LDS, and the carry into chunk m is
// c_m = a_{m-1} c_{m-1} + b_{m-1} from c_0 = 0, the same operations the one-wavefront loop
// performs.  Results are therefore bitwise identical for every (CPW, W) and workgroup shape, so
// the shape can be picked by timing alone.
// ------------------------------------------------------------------------------------------
template <typename T>
struct seg_map {
    T a, b;  // carry_out = a * carry_in + b
};

// Forward recurrence y_k = a_k y_{k-1} + b_k over the wavefront's chunks.  On entry b[u] holds
// chunk u's right-hand sides; afun(u) returns its multipliers a_k (reloaded when needed, so that
// only b stays in registers) and dval(u) its pivots.  On exit b[u] = y_k / d_k.  xch: this
// line's LDS slots, one per chunk of the line.
// AHEAD > 1 (W == 1): the multipliers and pivots of AHEAD chunks are loaded at a time.
template <typename T, int CPW, int W, int AHEAD = 1, typename AF, typename DF>
__device__ inline void seg_forward(T (&b)[CPW], AF afun, DF dval, seg_map<T> *xch, int w) {
    if constexpr (AHEAD > 1) {
        static_assert(W == 1 && CPW % AHEAD == 0, "whole groups of a line's one segment");
        T carry = T(0);
#pragma unroll
        for (int g = 0; g < CPW; g += AHEAD) {
            T a[AHEAD], d[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                a[u] = afun(g + u);
                d[u] = dval(g + u);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) {
                scan_affine_dpp(a[u], b[g + u]);
                const T y = affine(a[u], carry, b[g + u]);
                carry = last_lane(y);
                b[g + u] = div_pivot(y, d[u]);
            }
        }
        return;
    }
    if (W > 1) {
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            T a = afun(u);
            scan_affine_dpp(a, b[u]);
            const seg_map<T> m{last_lane(a), last_lane(b[u])};
            if (w < W - 1 && threadIdx.x % WAVE == 0) xch[w * CPW + u] = m;
        }
        lds_barrier();
        // the multipliers are reloaded below rather than kept live across the exchange
        asm volatile("" ::: "memory");
    }
    T carry = T(0);
    for (int m = 0; m < w * CPW; ++m) carry = affine(xch[m].a, carry, xch[m].b);
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
        T a = afun(u);
        if (W > 1)
            scan_prod_dpp(a);
        else
            scan_affine_dpp(a, b[u]);
        const T y = affine(a, carry, b[u]);
        carry = last_lane(y);
        b[u] = div_pivot(y, dval(u));
    }
}

// Backward recurrence x_k = a_k x_{k+1} + b_k, lanes in reversed element order (lane l of chunk
// c holds element 64c + 63 - l); the carry runs from the line's last chunk to its first.
// coef(u, a, b[u]) turns b[u] (the forward results) into the chunk's coefficients and returns
// the multipliers in a; afun(u) returns the multipliers alone.  On exit b[u] = x.
template <typename T, int CPW, int W, int AHEAD = 1, typename CF, typename AF>
__device__ inline void seg_backward(T (&b)[CPW], CF coef, AF afun, seg_map<T> *xch, int w) {
    if constexpr (AHEAD > 1) {
        static_assert(W == 1 && CPW % AHEAD == 0, "whole groups of a line's one segment");
        T carry = T(0);
#pragma unroll
        for (int g = CPW - AHEAD; g >= 0; g -= AHEAD) {
            T a[AHEAD];
#pragma unroll
            for (int u = 0; u < AHEAD; ++u) coef(g + u, a[u], b[g + u]);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = AHEAD - 1; u >= 0; --u) {
                scan_affine_dpp(a[u], b[g + u]);
                const T x = affine(a[u], carry, b[g + u]);
                carry = last_lane(x);
                b[g + u] = x;
            }
        }
        return;
    }
    if (W > 1) {
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            T a;
            coef(u, a, b[u]);
            scan_affine_dpp(a, b[u]);
            const seg_map<T> m{last_lane(a), last_lane(b[u])};
            if (w > 0 && threadIdx.x % WAVE == 0) xch[w * CPW + u] = m;
        }
        lds_barrier();
        // the multipliers are reloaded below rather than kept live across the exchange
        asm volatile("" ::: "memory");
    }
    T carry = T(0);
    for (int m = W * CPW - 1; m >= (w + 1) * CPW; --m) carry = affine(xch[m].a, carry, xch[m].b);
#pragma unroll
    for (int u = CPW - 1; u >= 0; --u) {
        T a;
        if (W > 1) {
            a = afun(u);
            scan_prod_dpp(a);
        } else {
            coef(u, a, b[u]);
            scan_affine_dpp(a, b[u]);
        }
        const T x = affine(a, carry, b[u]);
        carry = last_lane(x);
        b[u] = x;
    }
}

// Register-rich forms of the two recurrences (scanned multipliers kept in a[]), used by the
// x-line kernel: forward recurrence y_k = a_k y_{k-1} + b_k over the wavefront's chunks; on exit
// b[u] = y_k / D(u) with D(u) the pivots of chunk u (a functor, loaded after the scans).
// xch: this line's LDS slots, one per chunk of the line.
template <typename T, int CPW, int W, typename DF>
__device__ inline void seg_forward_ab(T (&a)[CPW], T (&b)[CPW], DF dval, seg_map<T> *xch, int w) {
#pragma unroll
    for (int u = 0; u < CPW; ++u) scan_affine_dpp(a[u], b[u]);
    T carry = T(0);
    if (W > 1) {
        if (w < W - 1) {  // chunk-end maps of all but the last segment
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                const seg_map<T> m{last_lane(a[u]), last_lane(b[u])};
                if (threadIdx.x % WAVE == 0) xch[w * CPW + u] = m;
            }
        }
        lds_barrier();
        for (int m = 0; m < w * CPW; ++m) carry = affine(xch[m].a, carry, xch[m].b);
    }
#pragma unroll
    for (int u = 0; u < CPW; ++u) {
        const T y = affine(a[u], carry, b[u]);
        carry = last_lane(y);
        b[u] = div_pivot(y, dval(u));
    }
}

// Backward recurrence x_k = a_k x_{k+1} + b_k, lanes in reversed element order (lane l of chunk
// c holds element 64c + 63 - l); the carry runs from the line's last chunk to its first.  On
// exit b[u] = x.
template <typename T, int CPW, int W>
__device__ inline void seg_backward_ab(T (&a)[CPW], T (&b)[CPW], seg_map<T> *xch, int w) {
#pragma unroll
    for (int u = 0; u < CPW; ++u) scan_affine_dpp(a[u], b[u]);
    T carry = T(0);
    if (W > 1) {
        if (w > 0) {
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                const seg_map<T> m{last_lane(a[u]), last_lane(b[u])};
                if (threadIdx.x % WAVE == 0) xch[w * CPW + u] = m;
            }
        }
        lds_barrier();
        for (int m = W * CPW - 1; m >= (w + 1) * CPW; --m) carry = affine(xch[m].a, carry, xch[m].b);
    }
#pragma unroll
    for (int u = CPW - 1; u >= 0; --u) {
        const T x = affine(a[u], carry, b[u]);
        carry = last_lane(x);
        b[u] = x;
    }
}

// x-lines of one colour, in place: L lines per workgroup, W wavefronts per line.  TR: the grid
// is the transpose of a y-line problem (right-hand side terms in the y-line order).
// rev: the tile walk of xcd_tile.  ZQ (zero start): q holds zeros outside the lines of this
// colour (a sweep that starts from a zero iterate), so the neighbour rows are not read and
// literal zeros enter the same arithmetic (a compile-time switch: a run-time select in front of
// the loads slowed the kernel by a quarter).
template <typename T, bool NINE, int CPW, int W, int L, bool TR = false, bool ZQ = false>
__global__ __launch_bounds__(L *W * 64) void relax_xlines_seg_k(const T *__restrict__ so,
                                                               const T *__restrict__ qf,
                                                               T *__restrict__ q,
                                                               const T *__restrict__ sor, int ii,
                                                               int jj, int first, int nlines,
                                                               int ntiles, int rev, int rep) {
    __shared__ seg_map<T> xch[2][L][W > 1 ? W * CPW : 1];
    int bx = (int)blockIdx.x, prob = (int)blockIdx.y;
    shared_op_order((int)gridDim.x, rep, bx, prob);  // gridDim.x is a multiple of 8
    const int tile = xcd_tile(bx, ntiles, rev);
    if (tile >= ntiles) return;  // uniform over the workgroup
    const int wl = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int slot = wl / W, w = wl % W;
    const int line = tile * L + slot;
    const bool valid = line < nlines;  // invalid wavefronts solve a copy of the last line
    const int j = first + 2 * min(line, nlines - 1);
    const std::size_t P = (std::size_t)ii * jj, bz = prob, bo = operator_of(bz, rep);
    so += bo * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    sor += bo * 2 * P;
    const int n = ii - 2;
    const std::size_t row = (std::size_t)j * ii;
    const T *D = sor + row + 1;      // D[k]
    const T *E = sor + P + row + 2;  // E[k], k < n-1
    const int rl = WAVE - 1 - lane;
    // Short segments (PRE): every operand, pivots and multipliers of both passes included, is in
    // flight before the first product.  Longer ones have no registers for that; theirs (MID) load
    // the pivots and the backward multipliers when the right-hand sides are formed, so that they
    // arrive during the forward scans and the exchange.  FP32, per colour: 77.5 -> 74.4 us at 4095^2,
    // 21.8 -> 19.1 at 2048^2, about 5 % on the levels below.
    constexpr bool PRE = CPW * sizeof(T) <= 16, MID = !PRE && W > 1 && CPW * sizeof(T) <= 64;
    // FP32 lines of one wavefront and 8 to 17 chunks load a chunk ahead of the one they scan: left to the
    // compiler the loads came late, 24.3 us per nine-point sweep at 1080^2 (20.9 before its registers
    // were dealt anew for PRE and MID), 26.6 at 1000 x 2048; 16.0 and 19.8.
    constexpr bool PIPE = W == 1 && !PRE && sizeof(T) == 4 && CPW >= 8 && CPW <= 17;
    line_raw<T> raw[PRE ? CPW : 1];
    T pe[PRE ? CPW : 1], pd[PRE || MID ? CPW : 1], pb[PRE || MID ? CPW : 1];
    if constexpr (PRE) {
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            const int k0 = (w * CPW + u) * WAVE, kc = min(k0 + lane, n - 1);
            line_load<T, NINE, 0>(raw[u], so, qf, q, P, ii, row + kc + 1, ZQ);
            pe[u] = E[max(kc - 1, 0)];
            pd[u] = D[kc];
            pb[u] = E[min(k0 + rl, max(n - 2, 0))];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    // right-hand side and multiplier of chunk u of the forward pass
    auto fwd_coef = [&](int u, T &au, T &bu) {
        const int k = (w * CPW + u) * WAVE + lane, kc = min(k, n - 1);
        T e;
        if constexpr (PRE) {
            bu = line_rhs<T, NINE, TR>(raw[u]);
            e = pe[u];
        } else {
            line_raw<T> r;
            line_load<T, NINE, 0>(r, so, qf, q, P, ii, row + kc + 1, ZQ);
            bu = line_rhs<T, NINE, TR>(r);
            e = E[max(kc - 1, 0)];
        }
        au = (k > 0) ? -e : T(0);
    };
    auto pivot = [&](int u) {
        if constexpr (PRE || MID)
            return pd[u];
        else
            return D[min((w * CPW + u) * WAVE + lane, n - 1)];
    };
    auto bwd_coef = [&](int u, T &au, T &bu) {  // chunk u of the backward pass, reversed lanes
        const int k = (w * CPW + u) * WAVE + rl;
        const T c = __shfl(bu, rl, WAVE);
        T e;
        if constexpr (PRE || MID)
            e = pb[u];
        else
            e = E[min(k, max(n - 2, 0))];
        au = (k < n - 1) ? -e : T(0);
        au = (k < n) ? au : T(1);
        bu = (k < n) ? c : T(0);
    };
    T b[CPW];
    if constexpr (W == 1) {
        // one wavefront per line: scan and carry chunk by chunk, only the results kept
        T carry = T(0);
        if constexpr (PIPE) {
            line_raw<T> r[2];
            T e[2], d[2];
            auto load = [&](int u) {
                const int kc = min(u * WAVE + lane, n - 1);
                line_load<T, NINE, 0>(r[u % 2], so, qf, q, P, ii, row + kc + 1, ZQ);
                e[u % 2] = E[max(kc - 1, 0)];
                d[u % 2] = D[kc];
            };
            load(0);
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                if (u + 1 < CPW) load(u + 1);
                __builtin_amdgcn_sched_barrier(0);
                T bu = line_rhs<T, NINE, TR>(r[u % 2]);
                T au = u * WAVE + lane > 0 ? -e[u % 2] : T(0);
                scan_affine_dpp(au, bu);
                const T y = affine(au, carry, bu);
                carry = last_lane(y);
                b[u] = div_pivot(y, d[u % 2]);
            }
        } else {
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                T au, bu;
                fwd_coef(u, au, bu);
                scan_affine_dpp(au, bu);
                const T y = affine(au, carry, bu);
                carry = last_lane(y);
                b[u] = div_pivot(y, pivot(u));
            }
        }
        carry = T(0);
#pragma unroll
        for (int u = CPW - 1; u >= 0; --u) {
            T au;
            bwd_coef(u, au, b[u]);
            scan_affine_dpp(au, b[u]);
            const T x = affine(au, carry, b[u]);
            carry = last_lane(x);
            b[u] = x;
        }
    } else {
        T a[CPW];
#pragma unroll
        for (int u = 0; u < CPW; ++u) fwd_coef(u, a[u], b[u]);
        if constexpr (MID) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < CPW; ++u) {
                const int k0 = (w * CPW + u) * WAVE;
                pd[u] = D[min(k0 + lane, n - 1)];
                pb[u] = E[min(k0 + rl, max(n - 2, 0))];
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        seg_forward_ab<T, CPW, W>(a, b, pivot, xch[0][slot], w);
#pragma unroll
        for (int u = 0; u < CPW; ++u) bwd_coef(u, a[u], b[u]);
        seg_backward_ab<T, CPW, W>(a, b, xch[1][slot], w);
    }
    if (valid) {
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            const int k = (w * CPW + u) * WAVE + rl;
            if (k < n) q[row + k + 1] = b[u];
        }
    }
}

// y-lines of one colour, in place: NC columns per workgroup, W wavefronts per column.  The
// right-hand sides of G chunk rows at a time are formed by the whole workgroup with
// row-contiguous loads (thread t: column t % NC, row t / NC of the W*64 rows) and handed to the
// column owners through LDS; results return through LDS for row-contiguous stores.
template <typename T, bool NINE, int CPW, int W, int NC, int G>
__global__ __launch_bounds__(NC *W * 64) void relax_ylines_seg_k(const T *__restrict__ so,
                                                                const T *__restrict__ qf,
                                                                T *__restrict__ q,
                                                                const T *__restrict__ sor,
                                                                int ii, int jj, int first,
                                                                int ncols, int ntiles, int rev,
                                                                int rep) {
    static_assert(CPW % G == 0, "G must divide CPW");
    __shared__ T tile_s[G][W][NC][WAVE + 1];
    __shared__ seg_map<T> xch[2][NC][W > 1 ? W * CPW : 1];
    int bx = (int)blockIdx.x, prob = (int)blockIdx.y;
    shared_op_order((int)gridDim.x, rep, bx, prob);  // gridDim.x is a multiple of 8
    const int tile = xcd_tile(bx, ntiles, rev);
    if (tile >= ntiles) return;  // uniform over the workgroup
    const int wl = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const int cs = wl / W, w = wl % W;
    const std::size_t P = (std::size_t)ii * jj, bz = prob, bo = operator_of(bz, rep);
    so += bo * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    sor += bo * 2 * P;
    const int n = jj - 2;
    const int col0 = tile * NC;
    const int nc = min(NC, ncols - col0);
    const int cb = first + 2 * col0;
    // the wavefront's own column (factors contiguous in j)
    const int ime = cb + 2 * min(cs, nc - 1);
    const T *D = sor + (std::size_t)ime * jj + 1;
    const T *E = sor + P + (std::size_t)ime * jj + 2;
    // this thread's tile position for the right-hand sides and the stores
    const int tc = threadIdx.x % NC, tr = threadIdx.x / NC;
    const int tseg = tr / WAVE, trow = tr % WAVE;
    const bool tok = tc < nc;
    const int ti = cb + 2 * min(tc, nc - 1);
    const int rl = WAVE - 1 - lane;
    // the factors of segments that have registers for them (PRE) are loaded with the first operands,
    // not when the scans reach them: per colour, 10.2 -> 8.5 us at 511^2 in FP32, 9.9 -> 8.2 at
    // 750 x 550 in FP64
    constexpr bool PRE = CPW * sizeof(T) <= 64;
    // The longest FP32 segments have no registers for that; left to itself the compiler loaded their
    // factors one at a time (five-point, per sweep: 4090^2 295 us, in groups of 8 149, of 4 159; 3000^2
    // 177 and 107).
    constexpr int AHEAD = W == 1 && CPW == 64 && sizeof(T) == 4 ? 8 : 1;
    T pe[PRE ? CPW : 1], pd[PRE ? CPW : 1], pb[PRE ? CPW : 1];
    auto fwd_a = [&](int u) {  // forward coefficient of chunk u
        const int k = (w * CPW + u) * WAVE + lane;
        T e;
        if constexpr (PRE)
            e = pe[u];
        else
            e = E[max(min(k, n - 1) - 1, 0)];
        return (k > 0) ? -e : T(0);
    };
    auto pivot = [&](int u) {
        if constexpr (PRE)
            return pd[u];
        else
            return D[min((w * CPW + u) * WAVE + lane, n - 1)];
    };
    // Right-hand sides of chunk rows g .. g+G-1 go through the tile.  The raw operands of the
    // next group are loaded before the current group's barrier (software pipelining), so one
    // group of loads is always in flight across the LDS exchange.
    line_raw<T> raw[G];
    auto load_group = [&](int g) {
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int k = min((tseg * CPW + g + u) * WAVE + trow, n - 1);
            line_load<T, NINE, 1>(raw[u], so, qf, q, P, ii, pidx(ti, k + 1, ii));
        }
    };
    auto form_tile = [&](int g) {
#pragma unroll
        for (int u = 0; u < G; ++u) tile_s[u][tseg][tc][trow] = line_rhs<T, NINE>(raw[u]);
        if (g + G < CPW) load_group(g + G);
    };
    load_group(0);
    if constexpr (PRE) {
#pragma unroll
        for (int u = 0; u < CPW; ++u) {
            const int k0 = (w * CPW + u) * WAVE, kc = min(k0 + lane, n - 1);
            pe[u] = E[max(kc - 1, 0)];
            pd[u] = D[kc];
            pb[u] = E[min(k0 + rl, max(n - 2, 0))];
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    auto bwd_a = [&](int u) {  // backward multipliers of chunk u, reversed lanes
        const int k = (w * CPW + u) * WAVE + rl;
        T e;
        if constexpr (PRE)
            e = pb[u];
        else
            e = E[min(k, max(n - 2, 0))];
        const T a = (k < n - 1) ? -e : T(0);
        return (k < n) ? a : T(1);
    };
    auto bwd_coef = [&](int u, T &au, T &bu) {
        const int k = (w * CPW + u) * WAVE + rl;
        const T c = __shfl(bu, rl, WAVE);
        au = bwd_a(u);
        bu = (k < n) ? c : T(0);
    };
    // all right-hand sides first (memory streaming only), then the scans
    T b[CPW];
#pragma unroll
    for (int g = 0; g < CPW; g += G) {
        form_tile(g);
        lds_barrier();
#pragma unroll
        for (int u = 0; u < G; ++u) b[g + u] = tile_s[u][w][cs][lane];
        lds_barrier();
    }
    if constexpr (PRE && W > 1) {
        T a[CPW];
#pragma unroll
        for (int u = 0; u < CPW; ++u) a[u] = fwd_a(u);
        seg_forward_ab<T, CPW, W>(a, b, pivot, xch[0][cs], w);
#pragma unroll
        for (int u = 0; u < CPW; ++u) bwd_coef(u, a[u], b[u]);
        seg_backward_ab<T, CPW, W>(a, b, xch[1][cs], w);
    } else {
        seg_forward<T, CPW, W, AHEAD>(b, fwd_a, pivot, xch[0][cs], w);
        seg_backward<T, CPW, W, AHEAD>(b, bwd_coef, bwd_a, xch[1][cs], w);
    }
#pragma unroll
    for (int g = 0; g < CPW; g += G) {
#pragma unroll
        for (int u = 0; u < G; ++u) tile_s[u][w][cs][rl] = b[g + u];
        lds_barrier();
#pragma unroll
        for (int u = 0; u < G; ++u) {
            const int k = (tseg * CPW + g + u) * WAVE + trow;
            if (tok && k < n) q[pidx(ti, k + 1, ii)] = tile_s[u][tseg][tc][trow];
        }
        lds_barrier();
    }
}

}  // namespace

// ---- line kernel shapes and their autotuner ---------------------------------------------------
// A shape is (CPW, W, L) for x-lines (chunks per wavefront, wavefronts per line, lines per
// workgroup) and (CPW, W, NC, G) for y-lines (..., columns per workgroup, chunk rows per LDS
// round).  All shapes of a chunk class give bitwise identical results (see the segmented
// kernels), so the shape of each (precision, stencil, direction, extents, batch) is picked by
// timing: tune_lines() times every candidate once on the caller's data and records the fastest in
// a process-wide table that the launchers consult; without an entry, candidate 0 runs.

template <typename T, bool NINE, int CPW, int W, int L, bool TR>
static void launch_x(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int first,
                     int nlines, hipStream_t s, int nb, int rev, int rep) {
    const int ntiles = (nlines + L - 1) / L;
    const dim3 blocks((unsigned)(8 * ((ntiles + 7) / 8)), (unsigned)nb);
    // rev bit 1: zero start (x-lines of the grid itself only)
    if (!TR && (rev & 2))
        relax_xlines_seg_k<T, NINE, CPW, W, L, TR, !TR><<<blocks, L * W * 64, 0, s>>>(
            so, qf, q, sor, ii, jj, first, nlines, ntiles, rev & 1, rep);
    else
        relax_xlines_seg_k<T, NINE, CPW, W, L, TR, false><<<blocks, L * W * 64, 0, s>>>(
            so, qf, q, sor, ii, jj, first, nlines, ntiles, rev & 1, rep);
}

template <typename T, bool NINE, int CPW, int W, int NC, int G>
static void launch_y(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int first,
                     int nlines, hipStream_t s, int nb, int rev, int rep) {
    const int ntiles = (nlines + NC - 1) / NC;
    const dim3 blocks((unsigned)(8 * ((ntiles + 7) / 8)), (unsigned)nb);
    relax_ylines_seg_k<T, NINE, CPW, W, NC, G><<<blocks, NC * W * 64, 0, s>>>(
        so, qf, q, sor, ii, jj, first, nlines, ntiles, rev, rep);
}

// Launches candidate c of chunk class NCH (lines of at most 64*NCH points); returns the number
// of candidates of the class (c outside [0, count) launches nothing).
static std::string shape_text(const char *k, int cpw, int w, const char *tn, int t, int g) {
    char buf[96];
    if (g > 0)
        std::snprintf(buf, sizeof(buf), "%s<CPW=%d,W=%d,%s=%d,G=%d>", k, cpw, w, tn, t, g);
    else
        std::snprintf(buf, sizeof(buf), "%s<CPW=%d,W=%d,%s=%d>", k, cpw, w, tn, t);
    return buf;
}

// With `name` non-null nothing is launched and *name receives candidate c's description.
// DIR 0: x-lines, 1: y-lines, 2: x-lines of a transposed y-line problem.
template <typename T, bool NINE, int DIR, int NCH>
static int launch_shape(int c, const T *so, const T *qf, T *q, const T *sor, int ii, int jj,
                        int first, int nlines, hipStream_t s, int nb, std::string *name = nullptr,
                        int rev = 0, int rep = 1) {
    constexpr bool TR = DIR == 2;
    constexpr bool F64 = sizeof(T) == 8;
#define CDR_X(k, C, W, L)                                                                       \
    if (c == k) {                                                                               \
        if (name)                                                                               \
            *name = shape_text("relax_xlines_seg_k", C, W, "L", L, 0);                          \
        else                                                                                    \
            launch_x<T, NINE, C, W, L, TR>(so, qf, q, sor, ii, jj, first, nlines, s, nb, rev,   \
                                           rep);                                                \
    }
#define CDR_Y(k, C, W, NC, G)                                                                   \
    if (c == k) {                                                                               \
        if (name)                                                                               \
            *name = shape_text("relax_ylines_seg_k", C, W, "NC", NC, G);                        \
        else                                                                                    \
            launch_y<T, NINE, C, W, NC, G>(so, qf, q, sor, ii, jj, first, nlines, s, nb, rev,   \
                                           rep);                                                \
    }
    // x: (CPW, W, L); y: (CPW, W, NC, G).  At most 16 wavefronts per workgroup.
    if constexpr (DIR != 1) {
        if constexpr (NCH <= 2) {
            CDR_X(0, NCH, 1, 4);
            return 1;
        } else if constexpr (NCH == 4) {
            CDR_X(0, 4, 1, 4);
            CDR_X(1, 1, 4, 1);
            return 2;
        } else if constexpr (NCH == 8) {
            CDR_X(0, 8, 1, 4);
            CDR_X(1, 4, 2, 2);
            CDR_X(2, 2, 4, 1);
            CDR_X(3, 1, 8, 1);  // one chunk per wavefront: the shortest chain per line
            return 4;
        } else if constexpr (NCH == 16) {
            CDR_X(0, 16, 1, 4);
            CDR_X(1, 8, 2, 2);
            CDR_X(2, 4, 4, 1);
            CDR_X(3, 2, 8, 1);
            CDR_X(4, 1, 16, 1);
            return 5;
        } else if constexpr (NCH == 32) {
            CDR_X(0, 16, 2, 2);
            CDR_X(1, 8, 4, 1);
            CDR_X(2, 4, 8, 1);
            CDR_X(3, F64 ? 2 : 32, F64 ? 16 : 1, F64 ? 1 : 4);
            // two neighbouring lines of a colour per workgroup share the row of q between them
            CDR_X(4, 8, 4, 2);
            CDR_X(5, 4, 8, 2);
            return 6;
        } else if constexpr (NCH == 3) {  // classes of 2^k + 1 chunks: W * CPW >= NCH
            CDR_X(0, 3, 1, 4);
            CDR_X(1, 1, 3, 2);
            return 2;
        } else if constexpr (NCH == 5) {
            CDR_X(0, 5, 1, 4);
            CDR_X(1, 3, 2, 2);
            CDR_X(2, 1, 5, 2);
            return 3;
        } else if constexpr (NCH == 9) {
            CDR_X(0, 9, 1, 4);
            CDR_X(1, 5, 2, 2);
            CDR_X(2, 3, 3, 2);
            CDR_X(3, 1, 9, 1);
            return 4;
        } else if constexpr (NCH == 17) {
            CDR_X(0, 17, 1, 4);
            CDR_X(1, 9, 2, 2);
            CDR_X(2, 6, 3, 1);
            CDR_X(3, 6, 3, 2);
            CDR_X(4, 3, 6, 1);
            return 5;
        } else if constexpr (NCH == 33) {
            CDR_X(0, 11, 3, 1);
            CDR_X(1, 11, 3, 2);
            CDR_X(2, 6, 6, 1);
            CDR_X(3, 3, 11, 1);
            CDR_X(4, 17, 2, 2);
            return 5;
        } else {
            CDR_X(0, 16, 4, 1);
            CDR_X(1, 8, 8, 1);
            CDR_X(2, 4, 16, 1);
            CDR_X(3, 64, 1, 4);
            CDR_X(4, 8, 8, 2);
            CDR_X(5, 16, 4, 2);
            return 6;
        }
    } else {
        // columns per workgroup for 64-byte (N1) and 128-byte (2 N1) row segments
        constexpr int N1 = F64 ? 4 : 8;
        // small levels: fewer columns per workgroup put more workgroups on the GPU (their rows
        // come from the caches at these sizes)
        if constexpr (NCH <= 2) {
            CDR_Y(0, NCH, 1, N1, NCH);
            CDR_Y(1, NCH, 1, 2 * N1, NCH);
            CDR_Y(2, NCH, 1, N1 / 4, NCH);
            return 3;
        } else if constexpr (NCH == 4) {
            CDR_Y(0, 4, 1, N1, 4);
            CDR_Y(1, 4, 1, 2 * N1, 2);
            CDR_Y(2, 1, 4, N1 / 2, 1);
            CDR_Y(3, 4, 1, N1 / 4, 4);
            CDR_Y(4, 2, 2, N1 / 4, 2);
            // FP32: one column per workgroup as well (FP64 has it as N1 / 4): the levels of a few
            // hundred columns are latency-bound, where more, smaller workgroups fill more CUs
            if constexpr (!F64) {
                CDR_Y(5, 2, 2, 1, 2);
                CDR_Y(6, 1, 4, 1, 1);
                return 7;
            }
            return 5;
        } else if constexpr (NCH == 8) {
            CDR_Y(0, 8, 1, N1, 4);
            CDR_Y(1, 8, 1, 2 * N1, 2);
            CDR_Y(2, 4, 2, N1, 4);
            CDR_Y(3, 2, 4, N1 / 2, 2);
            CDR_Y(4, 8, 1, N1 / 4, 4);
            CDR_Y(5, 4, 2, N1 / 4, 4);
            if constexpr (!F64) {
                CDR_Y(6, 4, 2, 1, 4);
                CDR_Y(7, 2, 4, 1, 2);
                return 8;
            }
            return 6;
        } else if constexpr (NCH == 16) {
            CDR_Y(0, 16, 1, N1, 4);
            CDR_Y(1, 8, 2, N1, 4);
            CDR_Y(2, 16, 1, 2 * N1, 2);
            CDR_Y(3, 4, 4, N1 / 2, 4);
            if constexpr (!F64) {
                CDR_Y(4, 4, 4, 1, 4);
                CDR_Y(5, 8, 2, 1, 4);
                return 6;
            }
            return 4;
        } else if constexpr (NCH == 32) {
            CDR_Y(0, 16, 2, N1, 2);
            CDR_Y(1, 32, 1, N1, 4);
            CDR_Y(2, 8, 4, N1 / 2, 2);
            CDR_Y(3, 4, 8, N1 / 4, 4);
            return 4;
        } else {  // 16-wavefront workgroups get 128 VGPRs: narrower tiles for long segments
            CDR_Y(0, 64, 1, N1, 2);
            CDR_Y(1, 16, 4, N1 / 2, 2);
            CDR_Y(2, 32, 2, N1 / 2, 2);
            CDR_Y(3, 64, 1, 2 * N1, 2);
            return 4;
        }
    }
#undef CDR_X
#undef CDR_Y
}

// chunk class of a line of n points: 1, 2, 4, ..., 64, or 0 beyond 4096 points.  With odd set
// (x-line shapes), lines of 3, 5, 9, 17 or 33 chunks get a class of their own: the lines of the
// 2^k + 1 grids (129 ... 2049 points) would otherwise leave almost half of the lanes of a
// power-of-two class idle.
static int chunk_class(int n, bool odd) {
    const int nch = (n + WAVE - 1) / WAVE;
    if (odd && (nch == 3 || nch == 5 || nch == 9 || nch == 17 || nch == 33)) return nch;
    int c = 1;
    while (c < nch && c < 64) c *= 2;
    return nch > 64 ? 0 : c;
}

template <typename T, bool NINE, int DIR>
static int launch_class(int c, const T *so, const T *qf, T *q, const T *sor, int ii, int jj,
                        int first, int nlines, hipStream_t s, int nb, std::string *name = nullptr,
                        int rev = 0, int rep = 1) {
    const int n = (DIR != 1) ? ii - 2 : jj - 2;
#define CDR_C(K)                                                                                  \
    case K:                                                                                       \
        return launch_shape<T, NINE, DIR, K>(c, so, qf, q, sor, ii, jj, first, nlines, s, nb, name, \
                                             rev, rep)
#define CDR_O(K)                                                                                  \
    case K:                                                                                       \
        if constexpr (DIR != 1)                                                                   \
            return launch_shape<T, NINE, DIR, K>(c, so, qf, q, sor, ii, jj, first, nlines, s, nb,  \
                                                 name, rev, rep);                                 \
        else                                                                                      \
            return 0;  /* not reached: y-lines use the power-of-two classes */
    switch (chunk_class(n, DIR != 1)) {
        CDR_C(1);
        CDR_C(2);
        CDR_O(3);
        CDR_C(4);
        CDR_O(5);
        CDR_C(8);
        CDR_O(9);
        CDR_C(16);
        CDR_O(17);
        CDR_C(32);
        CDR_O(33);
        CDR_C(64);
    default:  // lines longer than 4096: stage the forward results in q itself
        if constexpr (DIR == 2) {
            return 0;  // no transposed path for such lines
        } else {
            if (c == 0 && name) *name = "relax_lines_k";
            if (c == 0 && !name)
                relax_lines_k<T, NINE, DIR><<<dim3((unsigned)((nlines + 3) / 4), (unsigned)nb), 256,
                                              0, s>>>(so, qf, q, sor, ii, jj, first, nlines, rep);
            return 1;
        }
    }
#undef CDR_C
#undef CDR_O
}

namespace {
using tune_key = std::array<int, 6>;  // direction, word size, 9-point, ii, jj, batch
std::mutex g_tune_mu;
std::map<tune_key, int> g_tune;
std::atomic<int> g_autotune{1};
}  // namespace

template <typename T>
static tune_key key_of(int dir, int nstncl, int ii, int jj, int nb) {
    return tune_key{dir, (int)sizeof(T), nstncl == 5 ? 1 : 0, ii, jj, nb};
}

static int tuned_shape(const tune_key &k) {
    std::lock_guard<std::mutex> g(g_tune_mu);
    const auto it = g_tune.find(k);
    return it == g_tune.end() ? 0 : it->second;
}

template <typename T, int DIR>
static int launch_colour(int c, const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii,
                         int jj, int first, int nlines, hipStream_t s, int nb,
                         std::string *name = nullptr, int rev = 0, int rep = 1) {
    if (nstncl == 5)
        return launch_class<T, true, DIR>(c, so, qf, q, sor, ii, jj, first, nlines, s, nb, name, rev,
                                          rep);
    return launch_class<T, false, DIR>(c, so, qf, q, sor, ii, jj, first, nlines, s, nb, name, rev,
                                       rep);
}

static std::string shape_name(const std::array<int, 6> &k, int c) {
    std::string name;
    const int ns = k[2] ? 5 : 3;
    // direction 2 (y-lines through the transposed grid): an x-line shape on the swapped extents
    if (k[0] == 2 && c < 0) return "direct y-lines";
    const int dir = k[0] == 1 ? 1 : 0;
    const int ii = k[0] == 2 ? k[4] : k[3], jj = k[0] == 2 ? k[3] : k[4];
    if (k[1] == 8)
        (void)(dir == 0 ? launch_colour<double, 0>(c, nullptr, ns, nullptr, nullptr, nullptr, ii,
                                                   jj, 1, 1, nullptr, 1, &name)
                        : launch_colour<double, 1>(c, nullptr, ns, nullptr, nullptr, nullptr, ii,
                                                   jj, 1, 1, nullptr, 1, &name));
    else
        (void)(dir == 0 ? launch_colour<float, 0>(c, nullptr, ns, nullptr, nullptr, nullptr, ii,
                                                  jj, 1, 1, nullptr, 1, &name)
                        : launch_colour<float, 1>(c, nullptr, ns, nullptr, nullptr, nullptr, ii,
                                                  jj, 1, 1, nullptr, 1, &name));
    return k[0] == 2 ? "transposed, " + name : name;
}

// zq (x-lines of at most 4096 points only): the sweep starts from q = 0 (see relax_xlines_seg_k)
template <typename T, int DIR>
static void relax_lines(const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii, int jj,
                        int updown, hipStream_t s, int nb, int rep = 1, int zq = 0) {
    const int c = tuned_shape(key_of<T>(DIR, nstncl, ii, jj, nb));
    // lines of one colour: DOWN relaxes the lines at even array index (odd Cedar index) first,
    // UP the odd ones first (src/2d/ftn/BMG2_SymStd_relax_lines_x.f90:82-97)
    const int nfix = (DIR == 0) ? jj - 2 : ii - 2;
    for (int t = 0; t < 2; ++t) {
        const int first = (updown == 0) ? (t == 0 ? 2 : 1) : (t == 0 ? 1 : 2);
        if (first > nfix) continue;
        const int nlines = (nfix - first) / 2 + 1;
        // the second colour walks the lines in the opposite order (see xcd_tile)
        const int z = (DIR == 0 && zq && t == 0) ? 2 : 0;
        launch_colour<T, DIR>(c, so, nstncl, qf, q, sor, ii, jj, first, nlines, s, nb, nullptr,
                              t | z, rep);
    }
}

template <typename T>
void relax_lines_x(const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii, int jj,
                   int updown, hipStream_t s, int nb, int rep, int zero_start) {
    relax_lines<T, 0>(so, nstncl, qf, q, sor, ii, jj, updown, s, nb, rep,
                      zero_start && chunk_class(ii - 2, true) != 0);
}

bool lines_zero_start(int ii) { return chunk_class(ii - 2, true) != 0; }

template <typename T>
void relax_lines_y(const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii, int jj,
                   int updown, hipStream_t s, int nb, int rep) {
    relax_lines<T, 1>(so, nstncl, qf, q, sor, ii, jj, updown, s, nb, rep);
}

int set_autotune(int on) { return g_autotune.exchange(on ? 1 : 0); }
bool autotune_enabled() { return g_autotune.load() != 0; }

int line_shape_count(int dir, int wbytes, int nstncl, int ii, int jj) {
    const hipStream_t s = nullptr;  // counting launches nothing
    if (dir == 2) {  // x-line shapes of the transposed grid; none for lines over 4096 points
        if (jj - 2 > 64 * WAVE) return 0;
        dir = 0;
        std::swap(ii, jj);
    }
    if (wbytes == 8)
        return dir == 0 ? launch_colour<double, 0>(-1, nullptr, nstncl, nullptr, nullptr, nullptr,
                                                   ii, jj, 1, 1, s, 1)
                        : launch_colour<double, 1>(-1, nullptr, nstncl, nullptr, nullptr, nullptr,
                                                   ii, jj, 1, 1, s, 1);
    return dir == 0 ? launch_colour<float, 0>(-1, nullptr, nstncl, nullptr, nullptr, nullptr, ii,
                                              jj, 1, 1, s, 1)
                    : launch_colour<float, 1>(-1, nullptr, nstncl, nullptr, nullptr, nullptr, ii,
                                              jj, 1, 1, s, 1);
}

void set_line_shape(int dir, int wbytes, int nstncl, int ii, int jj, int nb, int shape) {
    const tune_key k{dir, wbytes, nstncl == 5 ? 1 : 0, ii, jj, nb};
    std::lock_guard<std::mutex> g(g_tune_mu);
    if (shape < 0)
        g_tune.erase(k);
    else
        g_tune[k] = shape;
}

template <typename T>
int tune_lines(int dir, const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii, int jj,
               hipStream_t s, int nb, int rep) {
    const tune_key k = key_of<T>(dir, nstncl, ii, jj, nb);
    {
        std::lock_guard<std::mutex> g(g_tune_mu);
        if (g_tune.count(k)) return g_tune[k];
    }
    auto run = [&](int c) {
        return dir == 0 ? launch_colour<T, 0>(c, so, nstncl, qf, q, sor, ii, jj, 1,
                                              (jj - 2 + 1) / 2, s, nb, nullptr, 0, rep)
                        : launch_colour<T, 1>(c, so, nstncl, qf, q, sor, ii, jj, 1,
                                              (ii - 2 + 1) / 2, s, nb, nullptr, 0, rep);
    };
    const int ncand = run(-1);  // count only
    if (!g_autotune.load() || ncand < 2) return 0;
    int best = 0;
    {
        hipEvent_t e0, e1;
        if (hipEventCreate(&e0) != hipSuccess) return -1;
        if (hipEventCreate(&e1) != hipSuccess) {
            (void)hipEventDestroy(e0);
            return -1;
        }
        // two rounds over the candidates, each candidate's time the smaller of its two: shapes
        // within a few percent of each other were otherwise picked by the noise of one timing
        std::vector<float> tmin(ncand, -1.f);
        for (int round = 0; round < 2; ++round)
            for (int c = 0; c < ncand; ++c) {
                run(c);  // warm-up
                (void)hipEventRecord(e0, s);
                for (int r = 0; r < 3; ++r) run(c);
                (void)hipEventRecord(e1, s);
                if (hipEventSynchronize(e1) != hipSuccess) break;
                float ms = 0.f;
                (void)hipEventElapsedTime(&ms, e0, e1);
                if (tmin[c] < 0.f || ms < tmin[c]) tmin[c] = ms;
            }
        for (int c = 1; c < ncand; ++c)
            if (tmin[c] >= 0.f && tmin[c] < tmin[best]) best = c;
        (void)hipEventDestroy(e0);
        (void)hipEventDestroy(e1);
        if (hipGetLastError() != hipSuccess) return -1;
    }
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune[k] = best;
    return best;
}

// ---- y-lines through the transposed grid ------------------------------------------------------
// With the operator transposed once at setup (soT: c, w, s, sw, nw of the transposed grid, i.e.
// the transposes of c, s, w, sw, nw), a y-line sweep is an x-line sweep of the transposed grid:
// q and f are transposed, both colours are relaxed with the x-line kernel (right-hand side terms in
// the y-line order, the y-line factors are already stored column-contiguous), and q is transposed
// back.  The result is bitwise that of relax_lines_y.

template <typename T>
static void relax_lines_ytr(const T *soT, int nstncl, const T *qf, T *q, const T *sory, T *qT,
                            T *qfT, int ii, int jj, int updown, int shape, hipStream_t s, int nb,
                            bool qfT_ready = false, bool q_in_T = false, bool keep_T = false,
                            int rep = 1) {
    if (!q_in_T) transpose<T>(q, qT, jj, ii, s, nb);
    if (!qfT_ready) transpose<T>(qf, qfT, jj, ii, s, nb);
    const int nfix = ii - 2;  // columns of the original grid = rows of the transposed one
    for (int t = 0; t < 2; ++t) {
        const int first = (updown == 0) ? (t == 0 ? 2 : 1) : (t == 0 ? 1 : 2);
        if (first > nfix) continue;
        const int nlines = (nfix - first) / 2 + 1;
        if (nstncl == 5)
            launch_class<T, true, 2>(shape, soT, qfT, qT, sory, jj, ii, first, nlines, s, nb,
                                     nullptr, t, rep);
        else
            launch_class<T, false, 2>(shape, soT, qfT, qT, sory, jj, ii, first, nlines, s, nb,
                                      nullptr, t, rep);
    }
    if (!keep_T) transpose<T>(qT, q, ii, jj, s, nb);
}

static int tuned_transposed(const tune_key &k) {
    std::lock_guard<std::mutex> g(g_tune_mu);
    const auto it = g_tune.find(k);
    return it == g_tune.end() ? -1 : it->second;
}

template <typename T>
bool relax_lines_y_auto(const T *so, const T *soT, int nstncl, const T *qf, T *q, const T *sory,
                        T *qT, T *qfT, int ii, int jj, int updown, hipStream_t s, int nb,
                        bool qfT_ready, bool q_in_T, bool keep_T, int rep) {
    const int c = uses_transposed_y<T>(soT, nstncl, ii, jj, nb);
    if (c < 0) {
        if (q_in_T) transpose<T>(qT, q, ii, jj, s, nb);
        relax_lines<T, 1>(so, nstncl, qf, q, sory, ii, jj, updown, s, nb, rep);
        return false;
    }
    relax_lines_ytr<T>(soT, nstncl, qf, q, sory, qT, qfT, ii, jj, updown, c, s, nb, qfT_ready,
                       q_in_T, keep_T, rep);
    return true;
}

template <typename T>
int uses_transposed_y(const T *soT, int nstncl, int ii, int jj, int nb) {
    return soT ? tuned_transposed(key_of<T>(2, nstncl, ii, jj, nb)) : -1;
}

// Milliseconds for 3 replays of what run(cs) launches, captured as a graph on the capture stream
// cs and replayed on s, the way the solvers execute their cycles (eager back-to-back launches
// would leave gaps that favour the variant with fewer launches); -1 if capture fails.
template <typename F>
static float time_captured(hipStream_t cs, hipStream_t s, hipEvent_t e0, hipEvent_t e1, F &&run) {
    if (!cs || hipStreamSynchronize(s) != hipSuccess) return -1.f;
    if (hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal) != hipSuccess) return -1.f;
    run(cs);
    hipGraph_t g = nullptr;
    if (hipStreamEndCapture(cs, &g) != hipSuccess || !g) {
        if (g) (void)hipGraphDestroy(g);
        return -1.f;
    }
    hipGraphExec_t ge = nullptr;
    float ms = -1.f;
    if (hipGraphInstantiate(&ge, g, nullptr, nullptr, 0) == hipSuccess) {
        (void)hipGraphLaunch(ge, s);  // warm-up
        (void)hipEventRecord(e0, s);
        for (int r = 0; r < 3; ++r) (void)hipGraphLaunch(ge, s);
        (void)hipEventRecord(e1, s);
        if (hipEventSynchronize(e1) == hipSuccess) (void)hipEventElapsedTime(&ms, e0, e1);
        (void)hipGraphExecDestroy(ge);
    }
    (void)hipGraphDestroy(g);
    return ms;
}

template <typename T>
int tune_lines_ytr(const T *so, const T *soT, int nstncl, const T *qf, T *q, const T *sory,
                   T *qT, T *qfT, int ii, int jj, hipStream_t s, int nb, int sweeps, int rep) {
    sweeps = sweeps < 1 ? 1 : sweeps;
    const tune_key k = key_of<T>(2, nstncl, ii, jj, nb);
    {
        std::lock_guard<std::mutex> g(g_tune_mu);
        if (g_tune.count(k)) return g_tune[k];
    }
    if (!g_autotune.load()) return -1;
    if (tune_lines<T>(1, so, nstncl, qf, q, sory, ii, jj, s, nb, rep) < 0) return -2;
    const int ncand = nstncl == 5 ? launch_class<T, true, 2>(-1, soT, qf, q, sory, jj, ii, 1, 1, s, nb)
                                  : launch_class<T, false, 2>(-1, soT, qf, q, sory, jj, ii, 1, 1, s, nb);
    hipEvent_t e0, e1;
    if (hipEventCreate(&e0) != hipSuccess) return -2;
    if (hipEventCreate(&e1) != hipSuccess) {
        (void)hipEventDestroy(e0);
        return -2;
    }
    hipStream_t cs = nullptr;
    if (hipStreamCreateWithFlags(&cs, hipStreamNonBlocking) != hipSuccess) cs = nullptr;
    auto timed1 = [&](auto &&run) {  // run(stream) launches one timed unit on that stream
        const float tc = time_captured(cs, s, e0, e1, run);
        if (tc >= 0.f) return tc;
        (void)hipGetLastError();  // eager timing when capture is not available
        run(s);  // warm-up
        (void)hipEventRecord(e0, s);
        for (int r = 0; r < 3; ++r) run(s);
        (void)hipEventRecord(e1, s);
        float ms = -1.f;
        if (hipEventSynchronize(e1) == hipSuccess) (void)hipEventElapsedTime(&ms, e0, e1);
        return ms;
    };
    auto timed = [&](auto &&run) {  // the faster of two timings
        const float a = timed1(run), b = timed1(run);
        return a < 0.f ? b : (b < 0.f ? a : (b < a ? b : a));
    };
    // `sweeps` y sweeps share one right-hand side (one transpose of qf)
    const float tdirect = timed([&](hipStream_t st) {
        for (int k = 0; k < sweeps; ++k)
            relax_lines<T, 1>(so, nstncl, qf, q, sory, ii, jj, 0, st, nb, rep);
    });
    int best = -1;
    float tbest = tdirect;
    for (int c = 0; c < ncand; ++c) {
        const float t = timed([&](hipStream_t st) {
            for (int k = 0; k < sweeps; ++k)
                relax_lines_ytr<T>(soT, nstncl, qf, q, sory, qT, qfT, ii, jj, 0, c, st, nb, k > 0,
                                   k > 0, k < sweeps - 1, rep);
        });
        if (t >= 0.f && t < tbest) {
            tbest = t;
            best = c;
        }
    }
    if (cs) (void)hipStreamDestroy(cs);
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    if (hipGetLastError() != hipSuccess) return -2;
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune[k] = best;
    return best;
}

void tune_clear() {
    std::lock_guard<std::mutex> g(g_tune_mu);
    g_tune.clear();
}

std::string tune_report() {
    std::lock_guard<std::mutex> g(g_tune_mu);
    std::string out = "[";
    for (const auto &kv : g_tune) {
        const tune_key &k = kv.first;
        char buf[160];
        std::snprintf(buf, sizeof(buf),
                      "%s{\"dir\":\"%c\",\"fp\":%d,\"stencil\":%d,\"ii\":%d,\"jj\":%d,\"nb\":%d,"
                      "\"shape\":%d,\"kernel\":\"",
                      out.size() > 1 ? "," : "", k[0] == 0 ? 'x' : (k[0] == 1 ? 'y' : 't'),
                      8 * k[1], k[2] ? 9 : 5,
                      k[3], k[4], k[5], kv.second);
        out += buf;
        out += shape_name(k, kv.second) + "\"}";
    }
    return out + "]";
}

template <typename T>
void relax_lines_xy(const T *so, int nstncl, const T *qf, T *q, const T *sorx, const T *sory,
                    T *work, int ii, int jj, int updown, hipStream_t s, int nb, int rep) {
    (void)work;
    if (updown == 0) {
        relax_lines<T, 0>(so, nstncl, qf, q, sorx, ii, jj, updown, s, nb, rep);
        relax_lines<T, 1>(so, nstncl, qf, q, sory, ii, jj, updown, s, nb, rep);
    } else {
        relax_lines<T, 1>(so, nstncl, qf, q, sory, ii, jj, updown, s, nb, rep);
        relax_lines<T, 0>(so, nstncl, qf, q, sorx, ii, jj, updown, s, nb, rep);
    }
}

#define CDR_INST(T)                                                                               \
    template void relax_lines_x<T>(const T *, int, const T *, T *, const T *, int, int, int,      \
        hipStream_t, int, int, int);                                                              \
    template void relax_lines_y<T>(const T *, int, const T *, T *, const T *, int, int, int,      \
        hipStream_t, int, int);                                                                   \
    template void relax_lines_xy<T>(const T *, int, const T *, T *, const T *, const T *, T *,    \
        int, int, int, hipStream_t, int, int);                                                    \
    template int tune_lines<T>(int, const T *, int, const T *, T *, const T *, int, int,          \
        hipStream_t, int, int);                                                                   \
    template bool relax_lines_y_auto<T>(const T *, const T *, int, const T *, T *, const T *,     \
        T *, T *, int, int, int, hipStream_t, int, bool, bool, bool, int);                        \
    template int uses_transposed_y<T>(const T *, int, int, int, int);                             \
    template int tune_lines_ytr<T>(const T *, const T *, int, const T *, T *, const T *, T *,     \
        T *, int, int, hipStream_t, int, int, int);
CDR_INST(double)
CDR_INST(float)
#undef CDR_INST

}  // namespace k2
}  // namespace cdr
