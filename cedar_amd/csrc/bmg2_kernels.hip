// 2D BoxMG kernels for CDNA4 (gfx950).
//
// Layout: Fortran order with one ghost layer; array index (i, j) with 0 <= i < ii, 0 <= j < jj,
// interior 1..ii-2 x 1..jj-2, point p = j*ii + i.  Stencil plane k of a level lives at
// so[k*ii*jj + p].  The off-diagonal couplings are stored negated; so[KNW] at (a, b) couples
// (a-1, b) with (a, b-1) and so[KSW] at (a, b) couples (a, b) with (a-1, b-1).
//
// Numerics: the FP64 kernels for residual, Gauss-Seidel, restriction, interpolation and
// operator-induced interpolation evaluate every point with the same operation order as Cedar's
// serial kernels and are compiled with -ffp-contract=off, so they reproduce them bit for bit.
// Line relaxation replaces the sequential LDL^T sweeps by a wavefront-wide affine scan and the
// Galerkin product is formed generically as P^T A P, so those two round differently (ulp level).
//
// All kernels are stencils on HBM-resident arrays (~0.2-0.3 flop/byte): no MFMA, coalesced
// accesses along i, 64-wide wavefronts, deterministic fixed-order reductions.
#include "../../include/cedar_hip.h"
#include "band_chol.hpp"
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
#include <vector>
#include <string>
#include <utility>

namespace cdr {
namespace k2 {

namespace {

inline dim3 grid2(int nx, int ny, int bx, int by) {
    return dim3((unsigned)((nx + bx - 1) / bx), (unsigned)((ny + by - 1) / by), 1);
}

// Batched problems: every kernel below takes the problem index from the last grid dimension
// (blockIdx.z for tiled kernels, blockIdx.y for line kernels, blockIdx.x for one-workgroup
// kernels); the problems of a batch are stored back to back, each with the layout above.
//  Shared
// operators: tile_order.hpp.

// one block of 1024 threads: sum of n partials in a fixed order -> *out.  Thread t adds
// partials t, t+1024, t+2048, ... in that order; loads are batched so they overlap.
__global__ __launch_bounds__(1024) void finalize_sum_k(const double *__restrict__ partials,
                                                       std::size_t n, double *__restrict__ out) {
    constexpr int T = 1024, U = 8;
    partials += (std::size_t)blockIdx.x * n;  // one workgroup per problem of a batch
    out += blockIdx.x;
    double v = 0.0;
    std::size_t k = threadIdx.x;
    for (; k + (U - 1) * T < n; k += U * T) {
        double t[U];
#pragma unroll
        for (int u = 0; u < U; ++u) t[u] = partials[k + (std::size_t)u * T];
#pragma unroll
        for (int u = 0; u < U; ++u) v += t[u];
    }
    for (; k < n; k += T) v += partials[k];
    block_sum_store<16>(v, out);
}

// ------------------------------------------------------------------------------------------
// residual  r = f + sum(couplings * q) - c q   (src/2d/ftn/BMG2_SymStd_residual.f90:85-119)
// block: 64 (i) x 4 (j)
// ------------------------------------------------------------------------------------------
template <typename T, bool NINE, bool NORM>
__global__ __launch_bounds__(256) void residual_k(const T *__restrict__ so, const T *__restrict__ qf,
                                                  const T *__restrict__ q, T *__restrict__ res,
                                                  int ii, int jj, double *__restrict__ partials,
                                                  int rep) {
    const wg_pos g = tiled_wg(rep);
    const int i = g.x * 64 + (threadIdx.x % 64) + 1;
    const int j = g.y * 4 + (threadIdx.x / 64) + 1;
    const std::size_t P = (std::size_t)ii * jj, bz = g.z;
    so += operator_of(bz, rep) * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    res += bz * P;
    if (NORM) partials += bz * gridDim.x * gridDim.y;
    double sq = 0.0;
    if (i <= ii - 2 && j <= jj - 2) {
        const std::size_t p = pidx(i, j, ii);
        const T c = so[p], x = q[p];
        T r = apply_offdiag<T, NINE>(so, P, q, p, ii, qf[p]);
        r = r - c * x;
        res[p] = r;
        if (NORM) sq = (double)r * (double)r;
    }
    if (NORM) block_sum_store(sq, &partials[g.y * gridDim.x + g.x]);
}

template <typename T>
__global__ __launch_bounds__(256) void sumsq_k(const T *__restrict__ x, int ii, int jj,
                                               double *__restrict__ partials) {
    const int i = blockIdx.x * 64 + (threadIdx.x % 64) + 1;
    const int j = blockIdx.y * 4 + (threadIdx.x / 64) + 1;
    const std::size_t bz = blockIdx.z;
    x += bz * (std::size_t)ii * jj;
    partials += bz * gridDim.x * gridDim.y;
    double sq = 0.0;
    if (i <= ii - 2 && j <= jj - 2) {
        double v = (double)x[pidx(i, j, ii)];
        sq = v * v;
    }
    block_sum_store(sq, &partials[blockIdx.y * gridDim.x + blockIdx.x]);
}

// mixed precision outer step: xnew = x + e, r = f - A xnew (FP64), r32 = (float) r; blocks of
// 64 (i) x IR_ROWS (j) points, 64 * IR_ROWS threads.  One workgroup per tile of one operator
// (blockIdx.z) does the rep right-hand sides of that operator (problems z * rep .. z * rep +
// rep - 1) one after another: the operator's couplings of a point are loaded once into
// registers for all of them (with one workgroup per problem, each re-read the 40 bytes per point
// of the operator).  f is loaded with the staged iterate, and the barriers order LDS only, so
// that stores of one right-hand side do not hold up the next.  Measured on the mixed solve of 29
// operators of 2049^2 with 4 right-hand sides each: 658 ms, against 686 ms with one workgroup
// per problem and 702 ms with the next right-hand side's loads software-pipelined.
constexpr int IR_ROWS = 8;
template <bool NINE, bool HAS_E>
__global__ __launch_bounds__(64 * IR_ROWS) void residual_ir_k(const double *__restrict__ so,
                                                     const double *__restrict__ qf,
                                                     const double *__restrict__ x,
                                                     const float *__restrict__ e,
                                                     double *__restrict__ xnew,
                                                     float *__restrict__ r32, int ii, int jj,
                                                     double *__restrict__ partials,
                                                     const int *__restrict__ active, int rep,
                                                     float *__restrict__ r32T) {
    // the updated iterate of the block and its one-point halo, formed once per point
    __shared__ double xs[IR_ROWS + 2][66];
    __shared__ float rt[IR_ROWS][65];  // r32 of the block, for the transposed copy
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    const int i0 = blockIdx.x * 64, j0 = blockIdx.y * IR_ROWS;  // halo corner of the block
    const int i = i0 + tx + 1, j = j0 + ty + 1;
    const std::size_t P = (std::size_t)ii * jj;
    const bool in = i <= ii - 2 && j <= jj - 2;
    const std::size_t p = in ? pidx(i, j, ii) : 0;
    so += (std::size_t)blockIdx.z * (NINE ? 5 : 3) * P;
    double cw0 = 0.0, cw1 = 0.0, cs0 = 0.0, cs1 = 0.0, co = 0.0;
    double csw0 = 0.0, cnw0 = 0.0, cnw1 = 0.0, csw1 = 0.0;
    if (in) {
        cw0 = so[P * KW + p];
        cw1 = so[P * KW + p + 1];
        cs0 = so[P * KS + p];
        cs1 = so[P * KS + p + ii];
        if (NINE) {
            csw0 = so[P * KSW + p];
            cnw0 = so[P * KNW + p + 1];
            cnw1 = so[P * KNW + p + ii];
            csw1 = so[P * KSW + p + ii + 1];
        }
        co = so[p];
    }
    auto X = [&](int di, int dj) { return xs[ty + 1 + dj][tx + 1 + di]; };
    for (int rh = 0; rh < rep; ++rh) {
        // xs, rt and the block sum's slots of the previous right-hand side are free: every
        // thread has passed the barrier of its block_sum_store (and, with r32T, the one before
        // its transposed copy), and thread 0 the staging barrier below
        const std::size_t bz = (std::size_t)blockIdx.z * rep + rh, off = bz * P;
        // a problem of a batch that has already converged keeps its iterate (active[b] == 0)
        const bool upd = HAS_E && (active == nullptr || active[bz] != 0);
        const double f = in ? qf[off + p] : 0.0;
        for (int t = threadIdx.x; t < (IR_ROWS + 2) * 66; t += 64 * IR_ROWS) {
            const int ti = i0 + t % 66, tj = j0 + t / 66;
            double v = 0.0;
            if (ti < ii && tj < jj) {
                const std::size_t k = off + pidx(ti, tj, ii);
                v = upd ? x[k] + (double)e[k] : x[k];
            }
            xs[t / 66][t % 66] = v;
        }
        lds_barrier();
        double sq = 0.0;
        if (in) {
            double r = f;
            r = r + cw0 * X(-1, 0);
            r = r + cw1 * X(1, 0);
            r = r + cs0 * X(0, -1);
            r = r + cs1 * X(0, 1);
            if (NINE) {
                r = r + csw0 * X(-1, -1);
                r = r + cnw0 * X(1, -1);
                r = r + cnw1 * X(-1, 1);
                r = r + csw1 * X(1, 1);
            }
            const double xc = X(0, 0);
            r = r - co * xc;
            xnew[off + p] = xc;
            r32[off + p] = (float)r;
            rt[ty][tx] = (float)r;
            sq = r * r;
        }
        block_sum_store<IR_ROWS, true>(
            sq, &partials[bz * gridDim.x * gridDim.y + blockIdx.y * gridDim.x + blockIdx.x]);
        if (r32T) {  // uniform over the launch
            lds_barrier();
            // consecutive threads write consecutive j of one row of the transposed grid
            const int a = threadIdx.x / IR_ROWS, c = threadIdx.x % IR_ROWS;
            const int i2 = i0 + a + 1, j2 = j0 + c + 1;
            if (i2 <= ii - 2 && j2 <= jj - 2) r32T[off + (std::size_t)i2 * jj + j2] = rt[c][a];
        }
    }
}

// ------------------------------------------------------------------------------------------
// point Gauss-Seidel, one launch per colour (src/2d/ftn/BMG2_SymStd_relax_GS.f90:78-137)
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void recip_k(const double *__restrict__ so,
                                               double *__restrict__ sor, int ii, int jj, int ns) {
    const int i = blockIdx.x * 64 + (threadIdx.x % 64) + 1;
    const int j = blockIdx.y * 4 + (threadIdx.x / 64) + 1;
    const std::size_t P = (std::size_t)ii * jj, bz = blockIdx.z;
    so += bz * ns * P;
    sor += bz * 2 * P;
    if (i <= ii - 2 && j <= jj - 2) {
        const std::size_t p = pidx(i, j, ii);
        sor[P + p] = 1.0 / so[p];
    }
}

// 5-point: colour = parity of (i + j); 9-point: colour = (i parity pi, j parity pj)
template <typename T, bool NINE>
// rev: the tiles are visited in reverse (a colour then starts where the previous one ended, in
// the memory-side cache); points of one colour are independent, so the result is unchanged
__global__ __launch_bounds__(256) void gs_colour_k(const T *__restrict__ so, const T *__restrict__ qf,
                                                   T *__restrict__ q, const T *__restrict__ sor,
                                                   int ii, int jj, int pi, int pj, int rep,
                                                   int rev = 0) {
    const wg_pos g = tiled_wg(rep);
    const int bx = rev ? (int)gridDim.x - 1 - g.x : g.x;
    const int by = rev ? (int)gridDim.y - 1 - g.y : g.y;
    const int k = bx * 64 + (threadIdx.x % 64);
    const int m = by * 4 + (threadIdx.x / 64);
    int i, j;
    if (NINE) {
        i = 2 * k + pi;
        j = 2 * m + pj;
    } else {
        j = m + 1;
        i = 2 * k + ((pi + j) & 1);  // (i + j) % 2 == pi
    }
    if (i < 1 || i > ii - 2 || j < 1 || j > jj - 2) return;
    const std::size_t P = (std::size_t)ii * jj, bz = g.z, bo = operator_of(bz, rep);
    so += bo * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    sor += bo * 2 * P;
    const std::size_t p = pidx(i, j, ii);
    const T rec = sor[P + p];
    const T v = apply_offdiag<T, NINE>(so, P, q, p, ii, qf[p]);
    q[p] = v * rec;
}

// ------------------------------------------------------------------------------------------
// restriction qc = P^T q (src/2d/ftn/BMG2_SymStd_restrict.f90:76-92); coarse (ic, jc) sits on
// fine (2ic-1, 2jc-1)
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void restrict_k(const T *__restrict__ ci, const T *__restrict__ q,
                                                  T *__restrict__ qc, int iif, int jjf, int iic,
                                                  int jjc, int rep) {
    const wg_pos g = tiled_wg(rep);
    const int ic = g.x * 64 + (threadIdx.x % 64) + 1;
    const int jc = g.y * 4 + (threadIdx.x / 64) + 1;
    if (ic > iic - 2 || jc > jjc - 2) return;
    const std::size_t Pc = (std::size_t)iic * jjc, bz = g.z;
    ci += operator_of(bz, rep) * 8 * Pc;
    q += bz * iif * (std::size_t)jjf;
    qc += bz * Pc;
    qc[pidx(ic, jc, iic)] = restrict_point<T>(ci, q, iif, iic, Pc, ic, jc);
}

// Restriction for a V-cycle step: qc = P^T q as restrict_k (same operations), and in the same
// launch the coarse iterate xc is zeroed (ghosts included: the coarse cycle starts from 0) and,
// where qcT is given, qc is also written transposed (qcT[ic * jjc + jc], for a coarse level whose
// y sweeps run through the transposed grid).  Tiles of 64 (ic) x 16 (jc) coarse points over the
// ghost-inclusive coarse grid, 64 * rc_rows<T> threads.
// FP64: one thread per coarse point of the tile, so that every point's loads are in flight at
// once (with a loop over rows the FP64 build kept one row's loads in flight at a time).  FP32: 4
// rows per thread (one point per thread was 3.8x slower over the levels of a batch of 116
// problems of 2049^2, and no faster on 4095^2).
template <typename T>
constexpr int rc_rows = sizeof(T) == 8 ? 16 : 4;
template <typename T>
__global__ __launch_bounds__(64 * rc_rows<T>) void restrict_cycle_k(const T *__restrict__ ci,
                                                                    const T *__restrict__ q,
                                                                    T *__restrict__ qc,
                                                                    T *__restrict__ xc,
                                                                    T *__restrict__ qcT, int iif,
                                                                    int jjf, int iic, int jjc,
                                                                    int rep) {
    constexpr int NT = 64 * rc_rows<T>;
    __shared__ T tile[16][65];
    const wg_pos g = tiled_wg(rep);
    const int ic0 = g.x * 64, jc0 = g.y * 16;
    const std::size_t Pc = (std::size_t)iic * jjc, bz = g.z;
    ci += operator_of(bz, rep) * 8 * Pc;
    q += bz * iif * (std::size_t)jjf;
    qc += bz * Pc;
    xc += bz * Pc;
    const int tx = threadIdx.x % 64, ic = ic0 + tx;
    constexpr int U = 16 / rc_rows<T>;
    restrict_ops<T> o[U];  // of the thread's rows, clamped into the interior
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int jc = jc0 + threadIdx.x / 64 + u * rc_rows<T>;
        load_restrict(o[u], ci, q, iif, iic, Pc, min(max(ic, 1), iic - 2), min(max(jc, 1), jjc - 2));
    }
    loads_issued();
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int k = threadIdx.x / 64 + u * rc_rows<T>;
        const int jc = jc0 + k;
        if (ic >= iic || jc >= jjc) continue;
        const std::size_t pc = pidx(ic, jc, iic);
        xc[pc] = T(0);
        if (ic >= 1 && ic <= iic - 2 && jc >= 1 && jc <= jjc - 2) {
            const T v = sum_restrict(o[u]);
            qc[pc] = v;
            tile[k][tx] = v;
        }
    }
    if (!qcT) return;  // uniform over the launch
    qcT += bz * Pc;
    __syncthreads();
    for (int e = threadIdx.x; e < 64 * 16; e += NT) {
        const int a = e / 16, c = e % 16;  // a: ic offset, c: jc offset (contiguous in qcT)
        const int i2 = ic0 + a, j2 = jc0 + c;
        if (i2 >= 1 && i2 <= iic - 2 && j2 >= 1 && j2 <= jjc - 2)
            qcT[(std::size_t)i2 * jjc + j2] = tile[c][a];
    }
}

// ------------------------------------------------------------------------------------------
// interp_add q += P qc + res / c at F-points (src/2d/ftn/BMG2_SymStd_interp_add.f90:101-137);
// one thread per 2 x 2 block of fine points.  res is only read (the reference divides it in place; nothing
// reads it afterwards).  For an even fine extent the reference's loops also reach the last
// fine ghost column / row (coarse index IICF1 = IIC); those points are updated the same way,
// with the raw res value there since the reference divides res only in the interior.
// ------------------------------------------------------------------------------------------
template <typename T>
__global__ __launch_bounds__(256) void interp_add_k(T *__restrict__ q, const T *__restrict__ qc,
                                                    const T *__restrict__ res,
                                                    const T *__restrict__ so,
                                                    const T *__restrict__ ci, int iic, int jjc,
                                                    int iif, int jjf, int ns, int rep) {
    const wg_pos g = tiled_wg(rep);
    const int m = g.x * 64 + (threadIdx.x % 64) + 1;
    const int n = g.y * 4 + (threadIdx.x / 64) + 1;
    const std::size_t Pc = (std::size_t)iic * jjc, Pf = (std::size_t)iif * jjf, bz = g.z;
    const std::size_t bo = operator_of(bz, rep);
    interp_block<T>(q + bz * Pf, qc + bz * Pc, res + bz * Pf, so + bo * ns * Pf, ci + bo * 8 * Pc,
                    iic, jjc, iif, jjf, m, n);
}

// ------------------------------------------------------------------------------------------
// operator-induced interpolation (src/2d/ftn/BMG2_SymStd_SETUP_interp_OI.f90:109-257)
// ------------------------------------------------------------------------------------------
__device__ inline double lumped(double c, double sum, double ep) {
    const double emach = 0x1.0p-53;  // D1MACH(3)
    return (c - sum) * fmax(c - (1.0 + ep) * sum, 0.0) / (fabs(c - (1.0 + ep) * sum) + emach);
}

// edge weights: x-edges (LR, LL) for ic in [2, nxf/2+1], jc in [1, ncy]; y-edges (LA, LB) for
// ic in [1, ncx], jc in [2, nyf/2+1].  Threads cover the union of both ranges.
template <bool NINE>
__global__ __launch_bounds__(256) void oi_edges_k(const double *__restrict__ so, double *__restrict__ ci,
                                                  int iif, int jjf, int iic, int jjc) {
    const int ic = blockIdx.x * 64 + (threadIdx.x % 64) + 1;
    const int jc = blockIdx.y * 4 + (threadIdx.x / 64) + 1;
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc, bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * P;
    ci += bz * 8 * Pc;
    auto S = [&](int a, int b, int k) { return so[P * k + pidx(a, b, iif)]; };
    const int icmax = (iif - 2) / 2 + 1, jcmax = (jjf - 2) / 2 + 1;
    const int i = 2 * ic - 1, j = 2 * jc - 1;
    const std::size_t pc = pidx(ic, jc, iic);
    if (ic >= 2 && ic <= icmax && jc <= jjc - 2) {
        double a, b;
        if (NINE) {
            a = S(i, j, KW) + S(i, j, KNW) + S(i, j + 1, KSW);
            b = S(i - 1, j, KW) + S(i - 1, j, KSW) + S(i - 1, j + 1, KNW);
        } else {
            a = S(i, j, KW);
            b = S(i - 1, j, KW);
        }
        const double c = S(i - 1, j, KO);
        const double ep = fmin(fabs(a / c), fabs(b / c));
        double sum = a + b + S(i - 1, j, KS) + S(i - 1, j + 1, KS);
        sum = a + b + lumped(c, sum, ep);
        sum = 1.0 / sum;
        ci[Pc * LR + pc] = a * sum;
        ci[Pc * LL + pc] = b * sum;
    }
    if (jc >= 2 && jc <= jcmax && ic <= iic - 2) {
        double a, b;
        if (NINE) {
            a = S(i, j, KS) + S(i, j, KNW) + S(i + 1, j, KSW);
            b = S(i, j - 1, KS) + S(i, j - 1, KSW) + S(i + 1, j - 1, KNW);
        } else {
            a = S(i, j, KS);
            b = S(i, j - 1, KS);
        }
        const double c = S(i, j - 1, KO);
        const double ep = fmin(fabs(a / c), fabs(b / c));
        double sum = a + b + S(i, j - 1, KW) + S(i + 1, j - 1, KW);
        sum = a + b + lumped(c, sum, ep);
        sum = 1.0 / sum;
        ci[Pc * LA + pc] = a * sum;
        ci[Pc * LB + pc] = b * sum;
    }
}

// corner weights for ic in [2, nxf/2+1], jc in [2, nyf/2+1], from the edge weights
template <bool NINE>
__global__ __launch_bounds__(256) void oi_corners_k(const double *__restrict__ so, double *__restrict__ ci,
                                                    int iif, int jjf, int iic, int jjc) {
    const int ic = blockIdx.x * 64 + (threadIdx.x % 64) + 2;
    const int jc = blockIdx.y * 4 + (threadIdx.x / 64) + 2;
    const int icmax = (iif - 2) / 2 + 1, jcmax = (jjf - 2) / 2 + 1;
    if (ic > icmax || jc > jcmax) return;
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc, bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * P;
    ci += bz * 8 * Pc;
    auto S = [&](int a, int b, int k) { return so[P * k + pidx(a, b, iif)]; };
    auto CI = [&](int a, int b, int k) { return ci[Pc * k + pidx(a, b, iic)]; };
    const int i = 2 * ic - 1, j = 2 * jc - 1;
    const double c = S(i - 1, j - 1, KO);
    double sum, ep;
    if (NINE) {
        sum = S(i - 1, j - 1, KW) + S(i - 1, j, KNW) + S(i - 1, j, KS) + S(i, j, KSW)
            + S(i, j - 1, KW) + S(i, j - 1, KNW) + S(i - 1, j - 1, KS) + S(i - 1, j - 1, KSW);
        const double e1 = fabs((S(i - 1, j - 1, KSW) + S(i - 1, j - 1, KW) + S(i - 1, j, KNW)) / c);
        const double e2 = fabs((S(i - 1, j, KNW) + S(i - 1, j, KS) + S(i, j, KSW)) / c);
        const double e3 = fabs((S(i, j, KSW) + S(i, j - 1, KW) + S(i, j - 1, KNW)) / c);
        const double e4 = fabs((S(i, j - 1, KNW) + S(i - 1, j - 1, KS) + S(i - 1, j - 1, KSW)) / c);
        ep = fmin(fmin(fmin(e1, e2), e3), e4);
    } else {
        sum = S(i - 1, j - 1, KW) + S(i - 1, j, KS) + S(i, j - 1, KW) + S(i - 1, j - 1, KS);
        ep = fmin(fmin(fmin(fabs(S(i - 1, j - 1, KW) / c), fabs(S(i - 1, j, KS) / c)),
                       fabs(S(i, j - 1, KW) / c)),
                  fabs(S(i - 1, j - 1, KS) / c));
    }
    sum = sum + lumped(c, sum, ep);
    const double s = 1.0 / sum;
    const std::size_t pc = pidx(ic, jc, iic);
    double sw = S(i - 1, j - 1, KS) * CI(ic, jc - 1, LL) + S(i - 1, j - 1, KW) * CI(ic - 1, jc, LB);
    double se = S(i - 1, j - 1, KS) * CI(ic, jc - 1, LR) + S(i, j - 1, KW) * CI(ic, jc, LB);
    double nw = S(i - 1, j - 1, KW) * CI(ic - 1, jc, LA) + S(i - 1, j, KS) * CI(ic, jc, LL);
    double ne = S(i - 1, j, KS) * CI(ic, jc, LR) + S(i, j - 1, KW) * CI(ic, jc, LA);
    if (NINE) {
        sw = sw + S(i - 1, j - 1, KSW);
        se = se + S(i, j - 1, KNW);
        nw = nw + S(i - 1, j, KNW);
        ne = ne + S(i, j, KSW);
    }
    ci[Pc * LSW + pc] = sw * s;
    ci[Pc * LSE + pc] = se * s;
    ci[Pc * LNW + pc] = nw * s;
    ci[Pc * LNE + pc] = ne * s;
}

// ------------------------------------------------------------------------------------------
// Galerkin coarse operator, formed generically: K(X, Y) = sum_f sum_g P(f,X) A(f,g) P(g,Y)
// over the 3x3 fine supports of the two coarse points.  Coarse entries (lower half):
// c = K(C,C), w = -K(C,C-e_x), s = -K(C,C-e_y), sw = -K(C,C-e_x-e_y),
// nw(C) = -K(C-e_x, C-e_y).  Couplings to coarse ghosts are zero (Dirichlet).
// ------------------------------------------------------------------------------------------
// weight of fine point centre(ic,jc) + (di,dj) in the column of coarse point (ic, jc)
__device__ inline double pweight(const double *__restrict__ ci, std::size_t Pc, int iic, int ic,
                                 int jc, int di, int dj) {
    auto CI = [&](int a, int b, int k) { return ci[Pc * k + pidx(a, b, iic)]; };
    if (di == 0 && dj == 0) return 1.0;
    if (di == -1 && dj == 0) return CI(ic, jc, LR);
    if (di == 1 && dj == 0) return CI(ic + 1, jc, LL);
    if (di == 0 && dj == -1) return CI(ic, jc, LA);
    if (di == 0 && dj == 1) return CI(ic, jc + 1, LB);
    if (di == -1 && dj == -1) return CI(ic, jc, LNE);
    if (di == 1 && dj == -1) return CI(ic + 1, jc, LNW);
    if (di == -1 && dj == 1) return CI(ic, jc + 1, LSE);
    return CI(ic + 1, jc + 1, LSW);
}

// A(f, f + (dx, dy)) of the fine operator
template <bool NINE>
__device__ inline double aentry(const double *__restrict__ so, std::size_t P, int ii, int x, int y,
                                int dx, int dy) {
    const std::size_t p = pidx(x, y, ii);
    if (dx == 0 && dy == 0) return so[p];
    if (dx == -1 && dy == 0) return -so[P * KW + p];
    if (dx == 1 && dy == 0) return -so[P * KW + p + 1];
    if (dx == 0 && dy == -1) return -so[P * KS + p];
    if (dx == 0 && dy == 1) return -so[P * KS + p + ii];
    if (!NINE) return 0.0;
    if (dx == -1 && dy == -1) return -so[P * KSW + p];
    if (dx == 1 && dy == 1) return -so[P * KSW + p + ii + 1];
    if (dx == 1 && dy == -1) return -so[P * KNW + p + 1];
    return -so[P * KNW + p + ii];
}

template <bool NINE, int DXC, int DYC>
__device__ inline double kpair(const double *__restrict__ so, const double *__restrict__ ci,
                               int iif, int jjf, int iic, int jjc, int icx, int jcx) {
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc;
    const int nxf = iif - 2, nyf = jjf - 2;
    const int X0 = 2 * icx - 1, Y0 = 2 * jcx - 1;
    const int icy = icx + DXC, jcy = jcx + DYC;
    double sum = 0.0;
#pragma unroll
    for (int fy = -1; fy <= 1; ++fy) {
#pragma unroll
        for (int fx = -1; fx <= 1; ++fx) {
            const int x = X0 + fx, y = Y0 + fy;
            if (x < 1 || x > nxf || y < 1 || y > nyf) continue;
            double inner = 0.0;
            bool any = false;
#pragma unroll
            for (int dy = -1; dy <= 1; ++dy) {
#pragma unroll
                for (int dx = -1; dx <= 1; ++dx) {
                    if (!NINE && dx != 0 && dy != 0) continue;
                    const int gx = fx + dx - 2 * DXC, gy = fy + dy - 2 * DYC;
                    if (gx < -1 || gx > 1 || gy < -1 || gy > 1) continue;
                    const int xg = x + dx, yg = y + dy;
                    if (xg < 1 || xg > nxf || yg < 1 || yg > nyf) continue;
                    inner += aentry<NINE>(so, P, iif, x, y, dx, dy) *
                             pweight(ci, Pc, iic, icy, jcy, gx, gy);
                    any = true;
                }
            }
            if (any) sum += pweight(ci, Pc, iic, icx, jcx, fx, fy) * inner;
        }
    }
    return sum;
}

template <bool NINE>
__global__ __launch_bounds__(256) void galerkin_k(const double *__restrict__ so,
                                                  const double *__restrict__ ci,
                                                  double *__restrict__ soc, int iif, int jjf,
                                                  int iic, int jjc) {
    const int ic = blockIdx.x * 64 + (threadIdx.x % 64) + 1;
    const int jc = blockIdx.y * 4 + (threadIdx.x / 64) + 1;
    if (ic > iic - 2 || jc > jjc - 2) return;
    const std::size_t Pc = (std::size_t)iic * jjc, pc = pidx(ic, jc, iic), bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * (std::size_t)iif * jjf;
    ci += bz * 8 * Pc;
    soc += bz * 5 * Pc;
    soc[pc] = kpair<NINE, 0, 0>(so, ci, iif, jjf, iic, jjc, ic, jc);
    soc[Pc * KW + pc] = (ic >= 2) ? -kpair<NINE, -1, 0>(so, ci, iif, jjf, iic, jjc, ic, jc) : 0.0;
    soc[Pc * KS + pc] = (jc >= 2) ? -kpair<NINE, 0, -1>(so, ci, iif, jjf, iic, jjc, ic, jc) : 0.0;
    const bool corner = ic >= 2 && jc >= 2;
    soc[Pc * KSW + pc] = corner ? -kpair<NINE, -1, -1>(so, ci, iif, jjf, iic, jjc, ic, jc) : 0.0;
    soc[Pc * KNW + pc] = corner ? -kpair<NINE, 1, -1>(so, ci, iif, jjf, iic, jjc, ic - 1, jc) : 0.0;
}

// ------------------------------------------------------------------------------------------
// coarsest grid: banded Cholesky (DPBTF2 upper) and solve (DPBTRS = two DTBSV), FP64, one
// workgroup.  Band layout ABD(ii, n), diagonal in row kd+1 = ii, kd = ii-1
// (src/2d/ftn/BMG2_SymStd_SETUP_cg_LU.f90:92-118, src/2d/ftn/BMG2_SymStd_SOLVE_cg.f90:93-123).
// ------------------------------------------------------------------------------------------
__global__ __launch_bounds__(256) void setup_cg_k(const double *__restrict__ so, int nstncl,
                                                  double *__restrict__ abd, int ii, int jj,
                                                  int *__restrict__ info) {
    const int nx = ii - 2, ny = jj - 2, n = nx * ny, kd = ii - 1, ld = ii;
    const std::size_t P = (std::size_t)ii * jj;
    so += (std::size_t)blockIdx.x * nstncl * P;  // one workgroup per problem of a batch
    abd += (std::size_t)blockIdx.x * ld * n;
    auto AB = [&](int r, int c) -> double & { return abd[(std::size_t)(c - 1) * ld + (r - 1)]; };
    for (int kk = threadIdx.x; kk < n; kk += blockDim.x) {
        const int i = kk % nx + 1, j = kk / nx + 1;
        const std::size_t p = pidx(i, j, ii);
        const int c = kk + 1;
        for (int r = 1; r <= ld; ++r) AB(r, c) = 0.0;
        AB(ii, c) = so[p];
        AB(ii - 1, c) = -so[P * KW + p];
        AB(3, c) = (nstncl == 5) ? -so[P * KNW + p + 1] : 0.0;
        AB(2, c) = -so[P * KS + p];
        AB(1, c) = (nstncl == 5) ? -so[P * KSW + p] : 0.0;
    }
    __syncthreads();
    __shared__ int bad;
    band_factor_upper(abd, n, kd, ld, bad);
    if (threadIdx.x == 0 && bad) atomicMax(info, bad);
}

template <typename T>
__global__ __launch_bounds__(64) void solve_cg_k(T *__restrict__ q, const T *__restrict__ qf,
                                                 const double *__restrict__ abd,
                                                 double *__restrict__ x, int ii, int jj, int rep) {
    __shared__ double sh[CG_LDS];
    const int n = (ii - 2) * (jj - 2);
    q += (std::size_t)blockIdx.x * ii * jj;  // one workgroup per problem of a batch
    qf += (std::size_t)blockIdx.x * ii * jj;
    abd += operator_of(blockIdx.x, rep) * ii * n;
    x += (std::size_t)blockIdx.x * n;
    coarse_band_solve<T>(q, qf, abd, x, ii, jj, threadIdx.x, blockDim.x, sh);
}

// ------------------------------------------------------------------------------------------
// elementwise helpers
// ------------------------------------------------------------------------------------------
template <typename Tin, typename Tout>
__global__ __launch_bounds__(256) void convert_k(const Tin *__restrict__ in, Tout *__restrict__ out,
                                                 std::size_t n) {
    for (std::size_t k = (std::size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (std::size_t)gridDim.x * blockDim.x)
        out[k] = (Tout)in[k];
}

template <typename T>
__global__ __launch_bounds__(256) void fill_k(T *__restrict__ x, T v, std::size_t n) {
    for (std::size_t k = (std::size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (std::size_t)gridDim.x * blockDim.x)
        x[k] = v;
}

// fill of a 16-byte aligned array: 16-byte stores (a quarter of the store instructions of
// fill_k; the zero start of the FP32 correction at 4095^2: 11.8 against 18.5 us), the tail in
// scalars
template <typename T>
__global__ __launch_bounds__(256) void fill16_k(T *__restrict__ x, T v, std::size_t n) {
    constexpr int W = 16 / sizeof(T);
    struct __attribute__((aligned(16))) vec {
        T e[W];
    };
    vec w;
#pragma unroll
    for (int u = 0; u < W; ++u) w.e[u] = v;
    vec *xv = reinterpret_cast<vec *>(x);
    const std::size_t nv = n / W;
    for (std::size_t k = (std::size_t)blockIdx.x * blockDim.x + threadIdx.x; k < nv;
         k += (std::size_t)gridDim.x * blockDim.x)
        xv[k] = w;
    const std::size_t t = (std::size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n - nv * W) x[nv * W + t] = v;
}

__global__ __launch_bounds__(256) void add_correction_k(double *__restrict__ x, const float *__restrict__ e,
                                                        int ii, int jj) {
    const int i = blockIdx.x * 64 + (threadIdx.x % 64) + 1;
    const int j = blockIdx.y * 4 + (threadIdx.x / 64) + 1;
    if (i > ii - 2 || j > jj - 2) return;
    const std::size_t p = pidx(i, j, ii) + (std::size_t)blockIdx.z * ii * jj;
    x[p] = x[p] + (double)e[p];
}

// x[k] = xprev[k] for the problems of a batch with active[b] == 0 (whole arrays, ghosts included)
__global__ __launch_bounds__(256) void keep_inactive_k(double *__restrict__ x,
                                                       const double *__restrict__ xprev,
                                                       const int *__restrict__ active,
                                                       std::size_t per, std::size_t n) {
    for (std::size_t k = (std::size_t)blockIdx.x * blockDim.x + threadIdx.x; k < n;
         k += (std::size_t)gridDim.x * blockDim.x)
        if (active[k / per] == 0) x[k] = xprev[k];
}

inline unsigned grid1(std::size_t n) {
    std::size_t b = (n + 255) / 256;
    if (b > 65536) b = 65536;
    return (unsigned)(b ? b : 1);
}

}  // namespace

// ==========================================================================================
// launchers
// ==========================================================================================
std::size_t norm_partials(int ii, int jj) {
    const dim3 g = grid2(ii - 2, jj - 2, 64, 4);
    return (std::size_t)g.x * g.y;
}

// tiled grid over an nx x ny index range, one z-slice per problem of a batch
static dim3 gridb(int nx, int ny, int nb) {
    dim3 g = grid2(nx, ny, 64, 4);
    g.z = (unsigned)nb;
    return g;
}

template <typename T>
void residual(const T *so, int nstncl, const T *qf, const T *q, T *res, int ii, int jj,
              hipStream_t s, int nb, int rep) {
    const dim3 g = gridb(ii - 2, jj - 2, nb);
    if (nstncl == 5)
        residual_k<T, true, false><<<g, 256, 0, s>>>(so, qf, q, res, ii, jj, nullptr, rep);
    else
        residual_k<T, false, false><<<g, 256, 0, s>>>(so, qf, q, res, ii, jj, nullptr, rep);
}

template <typename T>
void residual_norm(const T *so, int nstncl, const T *qf, const T *q, T *res, int ii, int jj,
                   double *partials, double *sumsq_out, hipStream_t s, int nb, int rep) {
    const dim3 g = gridb(ii - 2, jj - 2, nb);
    if (nstncl == 5)
        residual_k<T, true, true><<<g, 256, 0, s>>>(so, qf, q, res, ii, jj, partials, rep);
    else
        residual_k<T, false, true><<<g, 256, 0, s>>>(so, qf, q, res, ii, jj, partials, rep);
    finalize_sum_k<<<nb, 1024, 0, s>>>(partials, (std::size_t)g.x * g.y, sumsq_out);
}

template <typename T>
void sumsq(const T *x, int ii, int jj, double *partials, double *out, hipStream_t s, int nb) {
    const dim3 g = gridb(ii - 2, jj - 2, nb);
    sumsq_k<T><<<g, 256, 0, s>>>(x, ii, jj, partials);
    finalize_sum_k<<<nb, 1024, 0, s>>>(partials, (std::size_t)g.x * g.y, out);
}

void residual_ir(const double *so, int nstncl, const double *qf, const double *x, const float *e,
                 double *xnew, float *r32, int ii, int jj, double *partials, double *sumsq_out,
                 hipStream_t s, int nb, const int *active, int rep, float *r32T) {
    // one workgroup per tile of an operator; nb = operators * rep
    const dim3 g((unsigned)((ii - 2 + 63) / 64), (unsigned)((jj - 2 + IR_ROWS - 1) / IR_ROWS),
                 (unsigned)(nb / rep));
    const unsigned nt = 64 * IR_ROWS;
    if (nstncl == 5) {
        if (e)
            residual_ir_k<true, true><<<g, nt, 0, s>>>(so, qf, x, e, xnew, r32, ii, jj, partials,
                                                       active, rep, r32T);
        else
            residual_ir_k<true, false><<<g, nt, 0, s>>>(so, qf, x, e, xnew, r32, ii, jj, partials,
                                                        active, rep, r32T);
    } else {
        if (e)
            residual_ir_k<false, true><<<g, nt, 0, s>>>(so, qf, x, e, xnew, r32, ii, jj, partials,
                                                        active, rep, r32T);
        else
            residual_ir_k<false, false><<<g, nt, 0, s>>>(so, qf, x, e, xnew, r32, ii, jj, partials,
                                                         active, rep, r32T);
    }
    finalize_sum_k<<<nb, 1024, 0, s>>>(partials, (std::size_t)g.x * g.y, sumsq_out);
}

void setup_recip(const double *so, int nstncl, double *sor, int ii, int jj, hipStream_t s,
                 int nb) {
    recip_k<<<gridb(ii - 2, jj - 2, nb), 256, 0, s>>>(so, sor, ii, jj, nstncl);
}

template <typename T>
void relax_gs(const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii, int jj,
              int updown, hipStream_t s, int nb, int rep) {
    if (nstncl == 5) {
        if (relax_gs9_rows<T>(so, qf, q, sor, ii, jj, updown, s, nb, rep)) return;
        // DOWN: (i odd, j odd), (even, odd), (odd, even), (even, even); UP: reverse
        static const int order[4][2] = {{1, 1}, {0, 1}, {1, 0}, {0, 0}};
        const dim3 g = gridb(ii / 2 + 1, jj / 2 + 1, nb);
        for (int t = 0; t < 4; ++t) {
            const int c = updown == 0 ? t : 3 - t;
            gs_colour_k<T, true><<<g, 256, 0, s>>>(so, qf, q, sor, ii, jj, order[c][0], order[c][1],
                                                   rep, t & 1);
        }
    } else {
        // DOWN: (i + j) even first; UP: odd first
        const dim3 g = gridb(ii / 2 + 1, jj - 2, nb);
        for (int t = 0; t < 2; ++t) {
            const int parity = updown == 0 ? t : 1 - t;
            gs_colour_k<T, false><<<g, 256, 0, s>>>(so, qf, q, sor, ii, jj, parity, 0, rep, t & 1);
        }
    }
}

// dst (cols x rows) = transpose of src (rows x cols), row-major, for each problem of a batch;
// 64 x 64 tiles through LDS, 512 threads (8 rows per pass)
template <typename T>
__global__ __launch_bounds__(512) void transpose_k(const T *__restrict__ src, T *__restrict__ dst,
                                                  int rows, int cols) {
    __shared__ T tile[64][65];
    const std::size_t off = (std::size_t)blockIdx.z * rows * cols;
    src += off;
    dst += off;
    const int c0 = blockIdx.x * 64, r0 = blockIdx.y * 64;
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    for (int k = ty; k < 64; k += 8) {
        const int r = r0 + k, c = c0 + tx;
        if (r < rows && c < cols) tile[k][tx] = src[(std::size_t)r * cols + c];
    }
    __syncthreads();
    for (int k = ty; k < 64; k += 8) {
        const int c = c0 + k, r = r0 + tx;
        if (c < cols && r < rows) dst[(std::size_t)c * rows + r] = tile[tx][k];
    }
}

// The operator of the transposed grid: plane k of problem b of soT is the transpose of plane
// from[k] of problem b of so (c <- c, w <- s, s <- w, sw <- sw, nw <- nw); z = b * nstncl + k.
template <typename T>
__global__ __launch_bounds__(512) void transpose_op_k(const T *__restrict__ so, T *__restrict__ soT,
                                                     int rows, int cols, int nstncl) {
    __shared__ T tile[64][65];
    const int k = (int)blockIdx.z % nstncl, b = (int)blockIdx.z / nstncl;
    const int from = k == 0 ? KO : k == 1 ? KS : k == 2 ? KW : k;
    const std::size_t P = (std::size_t)rows * cols;
    const T *src = so + ((std::size_t)b * nstncl + from) * P;
    T *dst = soT + ((std::size_t)b * nstncl + k) * P;
    const int c0 = blockIdx.x * 64, r0 = blockIdx.y * 64;
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    for (int m = ty; m < 64; m += 8) {
        const int r = r0 + m, c = c0 + tx;
        if (r < rows && c < cols) tile[m][tx] = src[(std::size_t)r * cols + c];
    }
    __syncthreads();
    for (int m = ty; m < 64; m += 8) {
        const int c = c0 + m, r = r0 + tx;
        if (c < cols && r < rows) dst[(std::size_t)c * rows + r] = tile[tx][m];
    }
}

// FP32: 64 x 128 tiles moved as pairs of floats (see float_pair), twice the bytes per instruction
// of the one-float form (5.1 against 4.6 TB/s on a 4097^2 grid).
__global__ __launch_bounds__(512) void transpose_pairs_k(const float *__restrict__ src,
                                                         float *__restrict__ dst, int rows,
                                                         int cols) {
    __shared__ float tile[64][129];
    const std::size_t off = (std::size_t)blockIdx.z * rows * cols;
    src += off;
    dst += off;
    const int c0 = blockIdx.x * 128, r0 = blockIdx.y * 64;
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    const int c = c0 + 2 * tx;  // this lane's pair of source columns
    // all 8 loads of a thread in flight before the first LDS store
    float_pair v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int k = ty + 8 * u, r = r0 + k;
        const float *p = src + (std::size_t)r * cols + c;
        v[u] = float_pair{0.f, 0.f};
        if (r < rows) {
            if (c + 1 < cols)
                __builtin_memcpy(&v[u], p, sizeof(float_pair));
            else if (c < cols)
                v[u].a = p[0];
        }
    }
#pragma unroll
    for (int u = 0; u < 8; ++u) {
        const int k = ty + 8 * u;
        if (r0 + k < rows && c < cols) {
            tile[k][2 * tx] = v[u].a;
            if (c + 1 < cols) tile[k][2 * tx + 1] = v[u].b;
        }
    }
    __syncthreads();
    // a half-wavefront writes 64 consecutive destination values (one source column) as 32 pairs
    const int h = tx % 32, r = r0 + 2 * h;
    for (int k = 2 * ty + tx / 32; k < 128; k += 16) {
        const int cc = c0 + k;
        if (cc >= cols) continue;
        float *p = dst + (std::size_t)cc * rows + r;
        if (r + 1 < rows) {
            const float_pair v{tile[2 * h][k], tile[2 * h + 1][k]};
            __builtin_memcpy(p, &v, sizeof(v));
        } else if (r < rows) {
            p[0] = tile[2 * h][k];
        }
    }
}

// ------------------------------------------------------------------------------------------
// Kernels that take the iterate in the transposed layout (qT: ii rows of jj values,
// qT[i * jj + j] = q(i, j)), for levels whose y sweeps run as x sweeps of the transposed grid:
// after the last y sweep of the pre-smoothing the iterate stays transposed through the residual
// and interp_add, and the first y sweep of the post-smoothing starts from it, so the two grid
// transposes between them are not needed.  Every point is evaluated with the same operations in
// the same order as residual_k / interp_add_k, so results are bitwise identical.
// ------------------------------------------------------------------------------------------
constexpr int kTI = 64, kTJ = 32;  // residual_qT_k tile: 64 (i) x 32 (j) points, 256 threads

template <typename T, bool NINE>
__global__ __launch_bounds__(256) void residual_qT_k(const T *__restrict__ so,
                                                     const T *__restrict__ qf,
                                                     const T *__restrict__ qT,
                                                     T *__restrict__ res, int ii, int jj, int rep) {
    __shared__ T sq[kTJ + 2][kTI + 3];  // q(i0-1 .. i0+64, j0-1 .. j0+32) as [j][i]
    const wg_pos g = tiled_wg(rep);
    const int i0 = g.x * kTI + 1, j0 = g.y * kTJ + 1;
    const std::size_t P = (std::size_t)ii * jj, bz = g.z;
    so += operator_of(bz, rep) * (NINE ? 5 : 3) * P;
    qf += bz * P;
    qT += bz * P;
    res += bz * P;
    // stage: consecutive threads read consecutive j of one row of qT (a column of q); all loads
    // of a thread in flight before its LDS stores
    constexpr int NS = (kTI + 2) * (kTJ + 2), NU = (NS + 255) / 256;
    T v[NU];
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = threadIdx.x + 256 * u;
        const int a = e / (kTJ + 2), b = e % (kTJ + 2);
        const int i = i0 - 1 + a, j = j0 - 1 + b;
        v[u] = (e < NS && i < ii && j < jj) ? qT[(std::size_t)i * jj + j] : T(0);
    }
#pragma unroll
    for (int u = 0; u < NU; ++u) {
        const int e = threadIdx.x + 256 * u;
        if (e < NS) sq[e % (kTJ + 2)][e / (kTJ + 2)] = v[u];
    }
    __syncthreads();
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    const int i = i0 + tx;
    if (i > ii - 2) return;
#pragma unroll
    for (int u = 0; u < kTJ / 4; ++u) {
        const int k = ty + 4 * u;
        const int j = j0 + k;
        if (j > jj - 2) break;
        const std::size_t p = pidx(i, j, ii);
        auto Q = [&](int di, int dj) { return sq[k + 1 + dj][tx + 1 + di]; };
        T acc = qf[p];
        acc = acc + so[P * KW + p] * Q(-1, 0);
        acc = acc + so[P * KW + p + 1] * Q(1, 0);
        acc = acc + so[P * KS + p] * Q(0, -1);
        acc = acc + so[P * KS + p + ii] * Q(0, 1);
        if (NINE) {
            acc = acc + so[P * KSW + p] * Q(-1, -1);
            acc = acc + so[P * KNW + p + 1] * Q(1, -1);
            acc = acc + so[P * KNW + p + ii] * Q(-1, 1);
            acc = acc + so[P * KSW + p + ii + 1] * Q(1, 1);
        }
        res[p] = acc - so[p] * Q(0, 0);
    }
}

// residual_qT_k for the nr (2..rq_maxr) right-hand sides of one operator in one workgroup
// (blockIdx.z: the operator): the iterate tiles of all of them are staged (36 KB of LDS), then
// each point's couplings are loaded once and applied to every right-hand side, in
// residual_qT_k's order.
template <typename T>
constexpr int rq_maxr = sizeof(T) == 8 ? 2 : 4;
template <typename T, bool NINE>
__global__ __launch_bounds__(256) void residual_qT_rhs_k(const T *__restrict__ so,
                                                         const T *__restrict__ qf,
                                                         const T *__restrict__ qT,
                                                         T *__restrict__ res, int ii, int jj,
                                                         int nr) {
    __shared__ T sq[rq_maxr<T>][kTJ + 2][kTI + 3];  // per right-hand side, as in residual_qT_k
    const int i0 = blockIdx.x * kTI + 1, j0 = blockIdx.y * kTJ + 1;
    const std::size_t P = (std::size_t)ii * jj, b0 = (std::size_t)blockIdx.z * nr;
    so += (std::size_t)blockIdx.z * (NINE ? 5 : 3) * P;
    for (int rh = 0; rh < nr; ++rh) {
        const T *q = qT + (b0 + rh) * P;
        for (int e = threadIdx.x; e < (kTI + 2) * (kTJ + 2); e += 256) {
            const int a = e / (kTJ + 2), b = e % (kTJ + 2);
            const int i = i0 - 1 + a, j = j0 - 1 + b;
            sq[rh][b][a] = (i < ii && j < jj) ? q[(std::size_t)i * jj + j] : T(0);
        }
    }
    __syncthreads();
    const int tx = threadIdx.x % 64, ty = threadIdx.x / 64;
    const int i = i0 + tx;
    if (i > ii - 2) return;
    for (int u = 0; u < kTJ / 4; ++u) {
        const int k = ty + 4 * u;
        const int j = j0 + k;
        if (j > jj - 2) break;
        const std::size_t p = pidx(i, j, ii);
        const T cw0 = so[P * KW + p], cw1 = so[P * KW + p + 1];
        const T cs0 = so[P * KS + p], cs1 = so[P * KS + p + ii];
        T csw0 = T(0), cnw0 = T(0), cnw1 = T(0), csw1 = T(0);
        if (NINE) {
            csw0 = so[P * KSW + p];
            cnw0 = so[P * KNW + p + 1];
            cnw1 = so[P * KNW + p + ii];
            csw1 = so[P * KSW + p + ii + 1];
        }
        const T co = so[p];
        for (int rh = 0; rh < nr; ++rh) {
            auto Q = [&](int di, int dj) { return sq[rh][k + 1 + dj][tx + 1 + di]; };
            const std::size_t pb = (b0 + rh) * P + p;
            T acc = qf[pb];
            acc = acc + cw0 * Q(-1, 0);
            acc = acc + cw1 * Q(1, 0);
            acc = acc + cs0 * Q(0, -1);
            acc = acc + cs1 * Q(0, 1);
            if (NINE) {
                acc = acc + csw0 * Q(-1, -1);
                acc = acc + cnw0 * Q(1, -1);
                acc = acc + cnw1 * Q(-1, 1);
                acc = acc + csw1 * Q(1, 1);
            }
            res[pb] = acc - co * Q(0, 0);
        }
    }
}

// interp_add with the fine iterate transposed: phase 1 forms, per fine point of a 64 x 32 tile
// (32 x 16 blocks of 2 x 2 points, one thread each), the one (coarse point) or two (others) terms
// that interp_add_k adds, in its order; phase 2 adds them to qT with j-contiguous accesses.
template <typename T>
__global__ __launch_bounds__(512) void interp_add_qT_k(T *__restrict__ qT, const T *__restrict__ qc,
                                                       const T *__restrict__ res,
                                                       const T *__restrict__ so,
                                                       const T *__restrict__ ci, int iic, int jjc,
                                                       int iif, int jjf, int ns, int rep) {
    // one workgroup per tile of one operator (blockIdx.z) does the rep right-hand sides of that
    // operator (problems z * rep ..) one after another, with the block's interpolation weights
    // and operator diagonal loaded once into registers
    __shared__ T t1[32][65], t2[32][65];  // [j - jt][i - it]
    const int m0 = blockIdx.x * 32 + 1, n0 = blockIdx.y * 16 + 1;
    const int it = 2 * m0 - 1, jt = 2 * n0 - 1;  // first fine point of the tile
    const std::size_t Pc = (std::size_t)iic * jjc, Pf = (std::size_t)iif * jjf;
    const std::size_t b0 = (std::size_t)blockIdx.z * rep;
    so += (std::size_t)blockIdx.z * ns * Pf;
    ci += (std::size_t)blockIdx.z * 8 * Pc;
    const int imax = iif - 2 + ((iif - 2) % 2 == 0 ? 1 : 0);
    const int jmax = jjf - 2 + ((jjf - 2) % 2 == 0 ? 1 : 0);
    const int m = m0 + threadIdx.x % 32, n = n0 + threadIdx.x / 32;
    const int i0 = 2 * m - 1, j0 = 2 * n - 1;
    const bool act = i0 <= imax && j0 <= jmax;
    const bool xe = act && i0 + 1 <= imax, ye = act && j0 + 1 <= jmax;
    const int li = i0 - it, lj = j0 - jt;
    auto CI = [&](int a, int b, int k) { return ci[Pc * k + pidx(a, b, iic)]; };
    // res / c at the block's F-points (the raw res beyond the interior, as interp_add_k)
    auto fpt = [&](int i, int j, T &c) {
        const bool raw = i > iif - 2 || j > jjf - 2;
        c = raw ? T(1) : so[pidx(i, j, iif)];
        return raw;
    };
    T cLR = T(0), cLL = T(0), cLA = T(0), cLB = T(0);
    T cSW = T(0), cNW = T(0), cNE = T(0), cSE = T(0);
    T c10 = T(1), c01 = T(1), c11 = T(1);
    bool r10 = true, r01 = true, r11 = true;
    if (xe) {
        cLR = CI(m + 1, n, LR);
        cLL = CI(m + 1, n, LL);
        r10 = fpt(i0 + 1, j0, c10);
    }
    if (ye) {
        cLA = CI(m, n + 1, LA);
        cLB = CI(m, n + 1, LB);
        r01 = fpt(i0, j0 + 1, c01);
    }
    if (xe && ye) {
        cSW = CI(m + 1, n + 1, LSW);
        cNW = CI(m + 1, n + 1, LNW);
        cNE = CI(m + 1, n + 1, LNE);
        cSE = CI(m + 1, n + 1, LSE);
        r11 = fpt(i0 + 1, j0 + 1, c11);
    }
    for (int rh = 0; rh < rep; ++rh) {
        const std::size_t bz = b0 + rh;
        const T *qcb = qc + bz * Pc;
        const T *rsb = res + bz * Pf;
        T *qTb = qT + bz * Pf;
        if (rh > 0) __syncthreads();  // phase 2 of the previous right-hand side is done
        // phase 1: the one (coarse point) or two (others) terms interp_add_k adds, in its order
        if (act) {
            auto QC = [&](int a, int b) { return qcb[pidx(a, b, iic)]; };
            auto R = [&](int i, int j, bool raw, T c) {
                const T v = rsb[pidx(i, j, iif)];
                return raw ? v : v / c;
            };
            const T q00 = QC(m, n);
            t1[lj][li] = q00;
            if (xe) {
                t1[lj][li + 1] = cLR * QC(m + 1, n) + cLL * q00;
                t2[lj][li + 1] = R(i0 + 1, j0, r10, c10);
            }
            if (ye) {
                t1[lj + 1][li] = cLA * QC(m, n + 1) + cLB * q00;
                t2[lj + 1][li] = R(i0, j0 + 1, r01, c01);
            }
            if (xe && ye) {
                T a = cSW * q00;
                a = a + cNW * QC(m, n + 1);
                a = a + cNE * QC(m + 1, n + 1);
                a = a + cSE * QC(m + 1, n);
                t1[lj + 1][li + 1] = a;
                t2[lj + 1][li + 1] = R(i0 + 1, j0 + 1, r11, c11);
            }
        }
        __syncthreads();
        // phase 2: thread e -> (i offset e / 32, j offset e % 32): j-contiguous runs of 32 in
        // qT.  The thread's 4 points are distinct, so all 4 loads are issued before the first
        // store
        constexpr int NP = 64 * 32 / 512;
        T v[NP];
        bool ok[NP];
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int e = threadIdx.x + u * 512, pi = e / 32, pj = e % 32;
            const int i = it + pi, j = jt + pj;
            ok[u] = i <= imax && j <= jmax;
            v[u] = ok[u] ? qTb[(std::size_t)i * jjf + j] : T(0);
        }
#pragma unroll
        for (int u = 0; u < NP; ++u) {
            const int e = threadIdx.x + u * 512, pi = e / 32, pj = e % 32;
            if (!ok[u]) continue;
            T w = v[u] + t1[pj][pi];
            if (!((pi % 2 == 0) && (pj % 2 == 0))) w = w + t2[pj][pi];
            qTb[(std::size_t)(it + pi) * jjf + (jt + pj)] = w;
        }
    }
}

template <typename T>
void transpose(const T *src, T *dst, int rows, int cols, hipStream_t s, int nb) {
    if constexpr (sizeof(T) == 4) {
        const dim3 g((unsigned)((cols + 127) / 128), (unsigned)((rows + 63) / 64), (unsigned)nb);
        transpose_pairs_k<<<g, 512, 0, s>>>(src, dst, rows, cols);
    } else {
        const dim3 g((unsigned)((cols + 63) / 64), (unsigned)((rows + 63) / 64), (unsigned)nb);
        transpose_k<T><<<g, 512, 0, s>>>(src, dst, rows, cols);
    }
}

template <typename T>
void transpose_op(const T *so, T *soT, int nstncl, int ii, int jj, hipStream_t s, int nb) {
    // every stencil plane of every problem in one launch (z = problem * nstncl + plane)
    const dim3 g((unsigned)((ii + 63) / 64), (unsigned)((jj + 63) / 64), (unsigned)(nb * nstncl));
    transpose_op_k<T><<<g, 512, 0, s>>>(so, soT, jj, ii, nstncl);
}

template <typename T>
void restrict_(const T *ci, const T *q, T *qc, int iif, int jjf, int iic, int jjc, hipStream_t s,
               int nb, int rep) {
    restrict_k<T><<<gridb(iic - 2, jjc - 2, nb), 256, 0, s>>>(ci, q, qc, iif, jjf, iic, jjc, rep);
}

template <typename T>
void restrict_cycle(const T *ci, const T *q, T *qc, T *xc, T *qcT, int iif, int jjf, int iic,
                    int jjc, hipStream_t s, int nb, int rep) {
    const dim3 g((unsigned)((iic + 63) / 64), (unsigned)((jjc + 15) / 16), (unsigned)nb);
    restrict_cycle_k<T><<<g, 64 * rc_rows<T>, 0, s>>>(ci, q, qc, xc, qcT, iif, jjf, iic, jjc, rep);
}

template <typename T>
void interp_add(T *q, const T *qc, const T *res, const T *so, int nstncl, const T *ci, int iic,
                int jjc, int iif, int jjf, hipStream_t s, int nb, int rep) {
    // one thread per 2 x 2 fine block (the range includes the ghost point of even sizes)
    interp_add_k<T><<<gridb(iif / 2, jjf / 2, nb), 256, 0, s>>>(q, qc, res, so, ci, iic, jjc, iif,
                                                                jjf, nstncl, rep);
}

template <typename T>
void residual_qT(const T *so, int nstncl, const T *qf, const T *qT, T *res, int ii, int jj,
                 hipStream_t s, int nb, int rep) {
    if (rep >= 2 && rep <= rq_maxr<T>) {  // one workgroup per operator tile, all its rhs
        const dim3 g((unsigned)((ii - 2 + kTI - 1) / kTI), (unsigned)((jj - 2 + kTJ - 1) / kTJ),
                     (unsigned)(nb / rep));
        if (nstncl == 5)
            residual_qT_rhs_k<T, true><<<g, 256, 0, s>>>(so, qf, qT, res, ii, jj, rep);
        else
            residual_qT_rhs_k<T, false><<<g, 256, 0, s>>>(so, qf, qT, res, ii, jj, rep);
        return;
    }
    const dim3 g((unsigned)((ii - 2 + kTI - 1) / kTI), (unsigned)((jj - 2 + kTJ - 1) / kTJ),
                 (unsigned)nb);
    if (nstncl == 5)
        residual_qT_k<T, true><<<g, 256, 0, s>>>(so, qf, qT, res, ii, jj, rep);
    else
        residual_qT_k<T, false><<<g, 256, 0, s>>>(so, qf, qT, res, ii, jj, rep);
}

template <typename T>
void interp_add_qT(T *qT, const T *qc, const T *res, const T *so, int nstncl, const T *ci,
                   int iic, int jjc, int iif, int jjf, hipStream_t s, int nb, int rep) {
    // tiles of 32 x 16 blocks of 2 x 2 fine points over the blocks m <= iif/2, n <= jjf/2
    // (one workgroup per tile of an operator; nb = operators * rep)
    const dim3 g((unsigned)((iif / 2 + 31) / 32), (unsigned)((jjf / 2 + 15) / 16),
                 (unsigned)(nb / rep));
    interp_add_qT_k<T><<<g, 512, 0, s>>>(qT, qc, res, so, ci, iic, jjc, iif, jjf, nstncl, rep);
}

void setup_interp(const double *so, int nstncl, double *ci, int iif, int jjf, int iic, int jjc,
                  hipStream_t s, int nb) {
    const int icmax = (iif - 2) / 2 + 1, jcmax = (jjf - 2) / 2 + 1;
    const int ne = icmax > iic - 2 ? icmax : iic - 2;
    const int me = jcmax > jjc - 2 ? jcmax : jjc - 2;
    const dim3 ge = gridb(ne, me, nb);
    const dim3 gc = gridb(icmax - 1, jcmax - 1, nb);
    if (nstncl == 5) {
        oi_edges_k<true><<<ge, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc);
        oi_corners_k<true><<<gc, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc);
    } else {
        oi_edges_k<false><<<ge, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc);
        oi_corners_k<false><<<gc, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc);
    }
}

void setup_galerkin(const double *so, int nstncl, const double *ci, double *soc, int iif, int jjf,
                    int iic, int jjc, hipStream_t s, int nb) {
    const dim3 g = gridb(iic - 2, jjc - 2, nb);
    if (nstncl == 5)
        galerkin_k<true><<<g, 256, 0, s>>>(so, ci, soc, iif, jjf, iic, jjc);
    else
        galerkin_k<false><<<g, 256, 0, s>>>(so, ci, soc, iif, jjf, iic, jjc);
}

void setup_cg(const double *so, int nstncl, double *abd, int ii, int jj, int *info, hipStream_t s,
              int nb) {
    setup_cg_k<<<nb, 256, 0, s>>>(so, nstncl, abd, ii, jj, info);
}

template <typename T>
void solve_cg(T *q, const T *qf, const double *abd, double *bbd, int ii, int jj, hipStream_t s,
              int nb, int rep) {
    solve_cg_k<T><<<nb, 64, 0, s>>>(q, qf, abd, bbd, ii, jj, rep);
}

template <typename Tin, typename Tout>
void convert(const Tin *in, Tout *out, std::size_t n, hipStream_t s) {
    convert_k<Tin, Tout><<<grid1(n), 256, 0, s>>>(in, out, n);
}

template <typename T>
void fill(T *x, T v, std::size_t n, hipStream_t s) {
    if (reinterpret_cast<std::uintptr_t>(x) % 16 == 0 && (16 / sizeof(T)) > 1)
        fill16_k<T><<<grid1(n / (16 / sizeof(T)) + 1), 256, 0, s>>>(x, v, n);
    else
        fill_k<T><<<grid1(n), 256, 0, s>>>(x, v, n);
}

void finalize_sum(const double *partials, std::size_t n, double *out, int nb, hipStream_t s) {
    finalize_sum_k<<<nb, 1024, 0, s>>>(partials, n, out);
}

void keep_inactive(double *x, const double *xprev, const int *active, std::size_t per, int nb,
                   hipStream_t s) {
    const std::size_t n = per * (std::size_t)nb;
    keep_inactive_k<<<grid1(n), 256, 0, s>>>(x, xprev, active, per, n);
}

void add_correction(double *x, const float *e, int ii, int jj, hipStream_t s, int nb) {
    add_correction_k<<<gridb(ii - 2, jj - 2, nb), 256, 0, s>>>(x, e, ii, jj);
}

// ------------------------------------------------------------------------------------------
// Periodic boundaries (the JPN != 0 branches of the reference's 2D kernels).  jpn is the BoxMG
// boundary id of BMG_get_bc (src/2d/ftn/BMG_get_bc.f90): 2 periodic in x, 1 in y, 3 in both.
// The periodic images live in the ghost rows and columns: Q(1,J) = Q(II-1,J), Q(II,J) = Q(2,J)
// and Q(I,1) = Q(I,JJ-1), Q(I,JJ) = Q(I,2) in the reference's 1-based indices.
// ------------------------------------------------------------------------------------------
namespace {

__host__ __device__ inline bool per_x(int jpn) { return jpn == 2 || jpn == 3 || jpn == -2 || jpn == -3; }
__host__ __device__ inline bool per_y(int jpn) { return jpn == 1 || jpn == 3 || jpn == -1 || jpn == -3; }

// x images of rows j0, j0 + jstep, ... <= j1 (0-based rows)
template <typename T>
__global__ __launch_bounds__(256) void ghost_x_k(T *__restrict__ q, int ii, int jj, int j0, int j1,
                                                 int jstep) {
    const int j = j0 + (int)(blockIdx.x * 256 + threadIdx.x) * jstep;
    if (j > j1) return;
    q += (std::size_t)blockIdx.z * ii * jj;
    const std::size_t r = (std::size_t)j * ii;
    q[r] = q[r + ii - 2];
    q[r + ii - 1] = q[r + 1];
}

// y images of columns i0 .. i1
template <typename T>
__global__ __launch_bounds__(256) void ghost_y_k(T *__restrict__ q, int ii, int jj, int i0, int i1) {
    const int i = i0 + (int)(blockIdx.x * 256 + threadIdx.x);
    if (i > i1) return;
    q += (std::size_t)blockIdx.z * ii * jj;
    q[i] = q[(std::size_t)(jj - 2) * ii + i];
    q[(std::size_t)(jj - 1) * ii + i] = q[(std::size_t)ii + i];
}

template <typename T>
void ghost_x(T *q, int ii, int jj, int j0, int j1, int jstep, hipStream_t s, int nb) {
    if (j1 < j0) return;
    const int n = (j1 - j0) / jstep + 1;
    ghost_x_k<T><<<dim3((unsigned)((n + 255) / 256), 1, (unsigned)nb), 256, 0, s>>>(q, ii, jj, j0,
                                                                                   j1, jstep);
}
template <typename T>
void ghost_y(T *q, int ii, int jj, int i0, int i1, hipStream_t s, int nb) {
    if (i1 < i0) return;
    const int n = i1 - i0 + 1;
    ghost_y_k<T><<<dim3((unsigned)((n + 255) / 256), 1, (unsigned)nb), 256, 0, s>>>(q, ii, jj, i0,
                                                                                   i1);
}

// ---- operator-induced interpolation, periodic branch -------------------------------------
// (src/2d/ftn/BMG2_SymStd_SETUP_interp_OI.f90:259-616).  Loop bounds of the reference; the fine
// index of coarse index c follows I = MAX(MOD(I+2, N), MIN(I+2, 3)) from I = beg, which is
// 2(c-1) except at the periodic end, where it wraps to 3.
struct oi_bounds {
    int ibeg, ibegc, iendc, ibeg_x, iend_x, iifc;
    int jbeg, jbegc, jendc, jbeg_y, jend_y, jjfc;
};

__device__ inline int oi_fine(int c, int cbeg, int beg, int n) {
    const int prev = c == cbeg ? beg : 2 * (c - 2);
    const int a = (prev + 2) % n, b = prev + 2 < 3 ? prev + 2 : 3;
    return a > b ? a : b;
}

#define SOF(i, j, k) so[(std::size_t)((k) - 1) * P + (std::size_t)((j) - 1) * iif + ((i) - 1)]
#define CIF(i, j, k) ci[(std::size_t)((k) - 1) * Pc + (std::size_t)((j) - 1) * iic + ((i) - 1)]

__device__ inline double oi_lumped(double c, double sum, double ep) {
    const double emach = 0x1.0p-53;  // D1MACH(3)
    return (c - sum) * fmax(c - (1.0 + ep) * sum, 0.0) / (fabs(c - (1.0 + ep) * sum) + emach);
}

template <bool NINE>
__device__ void oi_xedge(const double *__restrict__ so, double *__restrict__ ci, std::size_t P,
                         std::size_t Pc, int iif, int iic, int i, int j, int ic, int jc) {
    constexpr int KO = 1, KW = 2, KS = 3, KSW = 4, KNW = 5, LL = 1, LR = 2;
    double a, b;
    if (NINE) {
        a = SOF(i, j, KW) + SOF(i, j, KNW) + SOF(i, j + 1, KSW);
        b = SOF(i - 1, j, KW) + SOF(i - 1, j, KSW) + SOF(i - 1, j + 1, KNW);
    } else {
        a = SOF(i, j, KW);
        b = SOF(i - 1, j, KW);
    }
    const double c = SOF(i - 1, j, KO);
    const double ep = fmin(fabs(a / c), fabs(b / c));
    double sum = a + b + SOF(i - 1, j, KS) + SOF(i - 1, j + 1, KS);
    sum = a + b + oi_lumped(c, sum, ep);
    sum = 1.0 / sum;
    CIF(ic, jc, LR) = a * sum;
    CIF(ic, jc, LL) = b * sum;
}

template <bool NINE>
__device__ void oi_yedge(const double *__restrict__ so, double *__restrict__ ci, std::size_t P,
                         std::size_t Pc, int iif, int iic, int i, int j, int ic, int jc) {
    constexpr int KO = 1, KW = 2, KS = 3, KSW = 4, KNW = 5, LA = 3, LB = 4;
    double a, b;
    if (NINE) {
        a = SOF(i, j, KS) + SOF(i, j, KNW) + SOF(i + 1, j, KSW);
        b = SOF(i, j - 1, KS) + SOF(i, j - 1, KSW) + SOF(i + 1, j - 1, KNW);
    } else {
        a = SOF(i, j, KS);
        b = SOF(i, j - 1, KS);
    }
    const double c = SOF(i, j - 1, KO);
    double sum = a + b + SOF(i, j - 1, KW) + SOF(i + 1, j - 1, KW);
    const double ep = fmin(fabs(a / c), fabs(b / c));
    sum = a + b + oi_lumped(c, sum, ep);
    sum = 1.0 / sum;
    CIF(ic, jc, LA) = a * sum;
    CIF(ic, jc, LB) = b * sum;
}

template <bool NINE>
__device__ void oi_corner(const double *__restrict__ so, double *__restrict__ ci, std::size_t P,
                          std::size_t Pc, int iif, int iic, int i, int j, int ic, int jc) {
    constexpr int KO = 1, KW = 2, KS = 3, KSW = 4, KNW = 5;
    constexpr int LL = 1, LR = 2, LA = 3, LB = 4, LSW = 5, LNW = 6, LNE = 7, LSE = 8;
    const double c = SOF(i - 1, j - 1, KO);
    double sum, ep;
    if (NINE) {
        sum = SOF(i - 1, j - 1, KW) + SOF(i - 1, j, KNW) + SOF(i - 1, j, KS) + SOF(i, j, KSW) +
              SOF(i, j - 1, KW) + SOF(i, j - 1, KNW) + SOF(i - 1, j - 1, KS) + SOF(i - 1, j - 1, KSW);
        const double e1 = fabs((SOF(i - 1, j - 1, KSW) + SOF(i - 1, j - 1, KW) + SOF(i - 1, j, KNW)) / c);
        const double e2 = fabs((SOF(i - 1, j, KNW) + SOF(i - 1, j, KS) + SOF(i, j, KSW)) / c);
        const double e3 = fabs((SOF(i, j, KSW) + SOF(i, j - 1, KW) + SOF(i, j - 1, KNW)) / c);
        const double e4 = fabs((SOF(i, j - 1, KNW) + SOF(i - 1, j - 1, KS) + SOF(i - 1, j - 1, KSW)) / c);
        ep = fmin(fmin(fmin(e1, e2), e3), e4);
    } else {
        sum = SOF(i - 1, j - 1, KW) + SOF(i - 1, j, KS) + SOF(i, j - 1, KW) + SOF(i - 1, j - 1, KS);
        const double e1 = fabs(SOF(i - 1, j - 1, KW) / c);
        const double e2 = fabs(SOF(i - 1, j, KS) / c);
        const double e3 = fabs(SOF(i, j - 1, KW) / c);
        const double e4 = fabs(SOF(i - 1, j - 1, KS) / c);
        ep = fmin(fmin(fmin(e1, e2), e3), e4);
    }
    sum = sum + oi_lumped(c, sum, ep);
    const double s = 1.0 / sum;
    if (NINE) {
        CIF(ic, jc, LSW) = (SOF(i - 1, j - 1, KS) * CIF(ic, jc - 1, LL) +
                            SOF(i - 1, j - 1, KW) * CIF(ic - 1, jc, LB) + SOF(i - 1, j - 1, KSW)) * s;
        CIF(ic, jc, LSE) = (SOF(i - 1, j - 1, KS) * CIF(ic, jc - 1, LR) +
                            SOF(i, j - 1, KW) * CIF(ic, jc, LB) + SOF(i, j - 1, KNW)) * s;
        CIF(ic, jc, LNW) = (SOF(i - 1, j - 1, KW) * CIF(ic - 1, jc, LA) +
                            SOF(i - 1, j, KS) * CIF(ic, jc, LL) + SOF(i - 1, j, KNW)) * s;
        CIF(ic, jc, LNE) = (SOF(i - 1, j, KS) * CIF(ic, jc, LR) +
                            SOF(i, j - 1, KW) * CIF(ic, jc, LA) + SOF(i, j, KSW)) * s;
    } else {
        CIF(ic, jc, LSW) = (SOF(i - 1, j - 1, KS) * CIF(ic, jc - 1, LL) +
                            SOF(i - 1, j - 1, KW) * CIF(ic - 1, jc, LB)) * s;
        CIF(ic, jc, LSE) = (SOF(i - 1, j - 1, KS) * CIF(ic, jc - 1, LR) +
                            SOF(i, j - 1, KW) * CIF(ic, jc, LB)) * s;
        CIF(ic, jc, LNW) = (SOF(i - 1, j - 1, KW) * CIF(ic - 1, jc, LA) +
                            SOF(i - 1, j, KS) * CIF(ic, jc, LL)) * s;
        CIF(ic, jc, LNE) = (SOF(i - 1, j, KS) * CIF(ic, jc, LR) +
                            SOF(i, j - 1, KW) * CIF(ic, jc, LA)) * s;
    }
}
#undef SOF
#undef CIF

// x-edge weights: rows jc = 2..jjc-1 (blockIdx.y rows of 4), and when periodic in y the two
// ghost rows jjc (from fine row jbeg_y) and 1 (from fine row jend_y) as rows jjc-1+1, jjc-1+2
template <bool NINE>
__global__ __launch_bounds__(256) void oi_per_xedge_k(const double *__restrict__ so,
                                                      double *__restrict__ ci, int iif, int jjf,
                                                      int iic, int jjc, oi_bounds B, int extra) {
    const int ic = B.ibegc + (int)(blockIdx.x * 64 + (threadIdx.x % 64));
    const int r = (int)(blockIdx.y * 4 + (threadIdx.x / 64));  // 0-based row item
    const int nrow = jjc - 2 + extra;
    if (ic > B.iendc || r >= nrow) return;
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc, bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * P;
    ci += bz * 8 * Pc;
    const int i = oi_fine(ic, B.ibegc, B.ibeg, B.iifc);
    int jc, j;
    if (r < jjc - 2) {
        jc = r + 2;
        j = 2 * (jc - 1);
    } else if (r == jjc - 2) {
        jc = jjc;
        j = B.jbeg_y;
    } else {
        jc = 1;
        j = B.jend_y;
    }
    oi_xedge<NINE>(so, ci, P, Pc, iif, iic, i, j, ic, jc);
}

// y-edge weights: columns ic = 2..iic-1, and when periodic in x the ghost columns iic (from fine
// column ibeg_x) and 1 (from iend_x); rows jc = jbegc..jendc
template <bool NINE>
__global__ __launch_bounds__(256) void oi_per_yedge_k(const double *__restrict__ so,
                                                      double *__restrict__ ci, int iif, int jjf,
                                                      int iic, int jjc, oi_bounds B, int extra) {
    const int c = (int)(blockIdx.x * 64 + (threadIdx.x % 64));  // 0-based column item
    const int jc = B.jbegc + (int)(blockIdx.y * 4 + (threadIdx.x / 64));
    const int ncol = iic - 2 + extra;
    if (c >= ncol || jc > B.jendc) return;
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc, bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * P;
    ci += bz * 8 * Pc;
    const int j = oi_fine(jc, B.jbegc, B.jbeg, B.jjfc);
    int ic, i;
    if (c < iic - 2) {
        ic = c + 2;
        i = 2 * (ic - 1);
    } else if (c == iic - 2) {
        ic = iic;
        i = B.ibeg_x;
    } else {
        ic = 1;
        i = B.iend_x;
    }
    oi_yedge<NINE>(so, ci, P, Pc, iif, iic, i, j, ic, jc);
}

template <bool NINE>
__global__ __launch_bounds__(256) void oi_per_corner_k(const double *__restrict__ so,
                                                       double *__restrict__ ci, int iif, int jjf,
                                                       int iic, int jjc, oi_bounds B) {
    const int ic = B.ibegc + (int)(blockIdx.x * 64 + (threadIdx.x % 64));
    const int jc = B.jbegc + (int)(blockIdx.y * 4 + (threadIdx.x / 64));
    if (ic > B.iendc || jc > B.jendc) return;
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc, bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * P;
    ci += bz * 8 * Pc;
    const int i = oi_fine(ic, B.ibegc, B.ibeg, B.iifc);
    const int j = oi_fine(jc, B.jbegc, B.jbeg, B.jjfc);
    oi_corner<NINE>(so, ci, P, Pc, iif, iic, i, j, ic, jc);
}

// Galerkin coarse operator in the reference's hand-expanded form (the ITLI products of
// src/2d/ftn/BMG2_SymStd_SETUP_ITLI_ex.f90:94-331), one thread per coarse point.  With periodic
// boundaries these formulas read the periodic images in the ghost rows and columns of SO and CI,
// which the generic P^T A P of galerkin_k does not visit; Dirichlet problems keep galerkin_k.
template <bool NINE>
__global__ __launch_bounds__(256) void galerkin_itli_k(const double *__restrict__ so,
                                                       const double *__restrict__ ci,
                                                       double *__restrict__ soc, int iif, int jjf,
                                                       int iic, int jjc) {
    const int ic = blockIdx.x * 64 + (threadIdx.x % 64) + 2;  // Fortran indices
    const int jc = blockIdx.y * 4 + (threadIdx.x / 64) + 2;
    if (ic > iic - 1 || jc > jjc - 1) return;
    const std::size_t P = (std::size_t)iif * jjf, Pc = (std::size_t)iic * jjc, bz = blockIdx.z;
    so += bz * (NINE ? 5 : 3) * P;
    ci += bz * 8 * Pc;
    soc += bz * 5 * Pc;
#define SO(i, j, k) so[(std::size_t)((k) - 1) * P + (std::size_t)((j) - 1) * iif + ((i) - 1)]
#define CI(i, j, k) ci[(std::size_t)((k) - 1) * Pc + (std::size_t)((j) - 1) * iic + ((i) - 1)]
#define SOC(i, j, k) soc[(std::size_t)((k) - 1) * Pc + (std::size_t)((j) - 1) * iic + ((i) - 1)]
    constexpr int KO = 1, KW = 2, KS = 3, KSW = 4, KNW = 5;
    constexpr int LL = 1, LR = 2, LA = 3, LB = 4, LSW = 5, LNW = 6, LNE = 7, LSE = 8;
    const int j = 2 * jc - 2, i = 2 * ic - 2;
    if (NINE) {
        double CO = SO(i, j + 1, KNW) * CI(ic, jc + 1, LSW) + SO(i, j, KW) * CI(ic, jc, LL)
                  + SO(i, j, KSW) * CI(ic, jc, LNW);
        double CS = SO(i, j - 1, KW) * CI(ic, jc, LNW) + SO(i, j, KNW) * CI(ic, jc, LL);
        double CSW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LNW) + SO(i - 1, j - 1, KW) * CI(ic - 1, jc, LA)
                   + SO(i - 1, j, KNW) + SO(i - 1, j, KS) * CI(ic, jc, LL);
        double CW = -SO(i - 1, j, KO) * CI(ic, jc, LL) + SO(i - 1, j, KS) * CI(ic, jc, LNW)
                  + SO(i - 1, j, KSW) * CI(ic - 1, jc, LA) + SO(i - 1, j, KW)
                  + SO(i - 1, j + 1, KNW) * CI(ic - 1, jc + 1, LB)
                  + SO(i - 1, j + 1, KS) * CI(ic, jc + 1, LSW);
        double CNW = -SO(i - 1, j + 1, KO) * CI(ic, jc + 1, LSW) + SO(i - 1, j + 1, KS) * CI(ic, jc, LL)
                   + SO(i - 1, j + 1, KSW) + SO(i - 1, j + 1, KW) * CI(ic - 1, jc + 1, LB);
        double CN = SO(i, j + 1, KSW) * CI(ic, jc, LL) + SO(i, j + 1, KW) * CI(ic, jc + 1, LSW);
        SOC(ic, jc, KW) = CO + CI(ic, jc, LA) * CS + CI(ic, jc, LNE) * CSW + CI(ic, jc, LR) * CW
                        + CI(ic, jc + 1, LSE) * CNW + CI(ic, jc + 1, LB) * CN;
        double COSW = SO(i, j, KSW) * CI(ic, jc, LSW);
        double CSSW = SO(i, j - 1, KSW) * CI(ic, jc - 1, LL) + SO(i, j - 1, KW) * CI(ic, jc, LSW);
        double CSWSW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LSW) + SO(i - 1, j - 1, KS) * CI(ic, jc - 1, LL)
                     + SO(i - 1, j - 1, KSW) + SO(i - 1, j - 1, KW) * CI(ic - 1, jc, LB);
        double CWSW = SO(i - 1, j, KS) * CI(ic, jc, LSW) + SO(i - 1, j, KSW) * CI(ic - 1, jc, LB);
        SOC(ic, jc, KSW) = COSW + CI(ic, jc, LA) * CSSW + CI(ic, jc, LNE) * CSWSW
                         + CI(ic, jc, LR) * CWSW;
        double COA = SO(i, j, KSW) * CI(ic, jc, LSE) + SO(i, j, KS) * CI(ic, jc, LB)
                   + SO(i + 1, j, KNW) * CI(ic + 1, jc, LSW);
        double CEA = SO(i + 1, j, KS) * CI(ic + 1, jc, LSW) + SO(i + 1, j, KSW) * CI(ic, jc, LB);
        double CSEA = -SO(i + 1, j - 1, KO) * CI(ic + 1, jc, LSW) + SO(i + 1, j - 1, KS) * CI(ic + 1, jc - 1, LL)
                    + SO(i + 1, j - 1, KSW) + SO(i + 1, j - 1, KW) * CI(ic, jc, LB);
        double CSA = -SO(i, j - 1, KO) * CI(ic, jc, LB) + SO(i + 1, j - 1, KW) * CI(ic + 1, jc, LSW)
                   + SO(i + 1, j - 1, KNW) * CI(ic + 1, jc - 1, LL) + SO(i, j - 1, KS)
                   + SO(i, j - 1, KSW) * CI(ic, jc - 1, LR) + SO(i, j - 1, KW) * CI(ic, jc, LSE);
        double CSWA = -SO(i - 1, j - 1, KO) * CI(ic, jc, LSE) + SO(i, j - 1, KW) * CI(ic, jc, LB)
                    + SO(i, j - 1, KNW) + SO(i - 1, j - 1, KS) * CI(ic, jc - 1, LR);
        double CWA = SO(i, j, KNW) * CI(ic, jc, LB) + SO(i - 1, j, KS) * CI(ic, jc, LSE);
        SOC(ic, jc, KS) = COA + CI(ic + 1, jc, LL) * CEA + CI(ic + 1, jc, LNW) * CSEA
                        + CI(ic, jc, LA) * CSA + CI(ic, jc, LNE) * CSWA + CI(ic, jc, LR) * CWA;
        double CONW = SO(i - 1, j, KNW) * CI(ic, jc, LSE);
        double CENW = SO(i, j, KNW) * CI(ic, jc, LB) + SO(i - 1, j, KS) * CI(ic, jc, LSE);
        double CSENW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LSE) + SO(i, j - 1, KW) * CI(ic, jc, LB)
                     + SO(i, j - 1, KNW) + SO(i - 1, j - 1, KS) * CI(ic, jc - 1, LR);
        double CFNW = SO(i - 1, j - 1, KW) * CI(ic, jc, LSE) + SO(i - 1, j - 1, KNW) * CI(ic, jc - 1, LR);
        SOC(ic, jc, KNW) = CONW + CI(ic, jc, LL) * CENW + CI(ic, jc, LNW) * CSENW
                         + CI(ic - 1, jc, LA) * CFNW;
        {
            double CO = SO(i, j, KW) * CI(ic, jc, LR) + SO(i, j + 1, KNW) * CI(ic, jc + 1, LSE)
                      + SO(i, j + 1, KS) * CI(ic, jc + 1, LB) + SO(i + 1, j + 1, KSW) * CI(ic + 1, jc + 1, LSW)
                      + SO(i + 1, j, KW) * CI(ic + 1, jc, LL) + SO(i + 1, j, KNW) * CI(ic + 1, jc, LNW)
                      + SO(i, j, KS) * CI(ic, jc, LA) + SO(i, j, KSW) * CI(ic, jc, LNE) - SO(i, j, KO);
            double CW = -SO(i - 1, j, KO) * CI(ic, jc, LR) + SO(i - 1, j + 1, KS) * CI(ic, jc + 1, LSE)
                      + SO(i, j + 1, KSW) * CI(ic, jc + 1, LB) + SO(i, j, KW) + SO(i, j, KNW) * CI(ic, jc, LA)
                      + SO(i - 1, j, KS) * CI(ic, jc, LNE);
            double CNW = -SO(i - 1, j + 1, KO) * CI(ic, jc + 1, LSE) + SO(i, j + 1, KW) * CI(ic, jc + 1, LB)
                       + SO(i, j + 1, KNW) + SO(i - 1, j + 1, KS) * CI(ic, jc, LR);
            double CN = -SO(i, j + 1, KO) * CI(ic, jc + 1, LB) + SO(i + 1, j + 1, KNW) * CI(ic + 1, jc, LL)
                      + SO(i, j + 1, KS) + SO(i, j + 1, KSW) * CI(ic, jc, LR)
                      + SO(i, j + 1, KW) * CI(ic, jc + 1, LSE) + SO(i + 1, j + 1, KW) * CI(ic + 1, jc + 1, LSW);
            double CNE = -SO(i + 1, j + 1, KO) * CI(ic + 1, jc + 1, LSW) + SO(i + 1, j + 1, KS) * CI(ic + 1, jc, LL)
                       + SO(i + 1, j + 1, KSW) + SO(i + 1, j + 1, KW) * CI(ic, jc + 1, LB);
            double CE = -SO(i + 1, j, KO) * CI(ic + 1, jc, LL) + SO(i + 1, j, KS) * CI(ic + 1, jc, LNW)
                      + SO(i + 1, j, KSW) * CI(ic, jc, LA) + SO(i + 1, j, KW)
                      + SO(i + 1, j + 1, KNW) * CI(ic, jc + 1, LB) + SO(i + 1, j + 1, KS) * CI(ic + 1, jc + 1, LSW);
            double CSE = -SO(i + 1, j - 1, KO) * CI(ic + 1, jc, LNW) + SO(i + 1, j - 1, KW) * CI(ic, jc, LA)
                       + SO(i + 1, j, KNW) + SO(i + 1, j, KS) * CI(ic + 1, jc, LL);
            double CS = -SO(i, j - 1, KO) * CI(ic, jc, LA) + SO(i, j - 1, KW) * CI(ic, jc, LNE)
                      + SO(i, j, KNW) * CI(ic, jc, LR) + SO(i, j, KS) + SO(i + 1, j, KSW) * CI(ic + 1, jc, LL)
                      + SO(i + 1, j - 1, KW) * CI(ic + 1, jc, LNW);
            double CSW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LNE) + SO(i - 1, j, KS) * CI(ic, jc, LR)
                       + SO(i, j, KSW) + SO(i, j - 1, KW) * CI(ic, jc, LA);
            SOC(ic, jc, KO) = -CI(ic, jc + 1, LSE) * CNW - CI(ic, jc + 1, LB) * CN
                            - CI(ic + 1, jc + 1, LSW) * CNE - CI(ic, jc, LR) * CW - CO
                            - CI(ic + 1, jc, LL) * CE - CI(ic, jc, LNE) * CSW
                            - CI(ic, jc, LA) * CS - CI(ic + 1, jc, LNW) * CSE;
        }
    } else {
        double CO = SO(i, j, KW) * CI(ic, jc, LL);
        double CS = SO(i, j - 1, KW) * CI(ic, jc, LNW);
        double CSW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LNW) + SO(i - 1, j - 1, KW) * CI(ic - 1, jc, LA)
                   + SO(i - 1, j, KS) * CI(ic, jc, LL);
        double CW = -SO(i - 1, j, KO) * CI(ic, jc, LL) + SO(i - 1, j, KS) * CI(ic, jc, LNW)
                  + SO(i - 1, j, KW) + SO(i - 1, j + 1, KS) * CI(ic, jc + 1, LSW);
        double CNW = -SO(i - 1, j + 1, KO) * CI(ic, jc + 1, LSW) + SO(i - 1, j + 1, KS) * CI(ic, jc, LL)
                   + SO(i - 1, j + 1, KW) * CI(ic - 1, jc + 1, LB);
        double CN = SO(i, j + 1, KW) * CI(ic, jc + 1, LSW);
        SOC(ic, jc, KW) = CO + CI(ic, jc, LA) * CS + CI(ic, jc, LNE) * CSW + CI(ic, jc, LR) * CW
                        + CI(ic, jc + 1, LSE) * CNW + CI(ic, jc + 1, LB) * CN;
        double CSSW = SO(i, j - 1, KW) * CI(ic, jc, LSW);
        double CSWSW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LSW) + SO(i - 1, j - 1, KS) * CI(ic, jc - 1, LL)
                     + SO(i - 1, j - 1, KW) * CI(ic - 1, jc, LB);
        double CWSW = SO(i - 1, j, KS) * CI(ic, jc, LSW);
        SOC(ic, jc, KSW) = CI(ic, jc, LA) * CSSW + CI(ic, jc, LNE) * CSWSW + CI(ic, jc, LR) * CWSW;
        double COA = SO(i, j, KS) * CI(ic, jc, LB);
        double CEA = SO(i + 1, j, KS) * CI(ic + 1, jc, LSW);
        double CSEA = -SO(i + 1, j - 1, KO) * CI(ic + 1, jc, LSW) + SO(i + 1, j - 1, KS) * CI(ic + 1, jc - 1, LL)
                    + SO(i + 1, j - 1, KW) * CI(ic, jc, LB);
        double CSA = -SO(i, j - 1, KO) * CI(ic, jc, LB) + SO(i + 1, j - 1, KW) * CI(ic + 1, jc, LSW)
                   + SO(i, j - 1, KS) + SO(i, j - 1, KW) * CI(ic, jc, LSE);
        double CSWA = -SO(i - 1, j - 1, KO) * CI(ic, jc, LSE) + SO(i, j - 1, KW) * CI(ic, jc, LB)
                    + SO(i - 1, j - 1, KS) * CI(ic, jc - 1, LR);
        double CWA = SO(i - 1, j, KS) * CI(ic, jc, LSE);
        SOC(ic, jc, KS) = COA + CI(ic + 1, jc, LL) * CEA + CI(ic + 1, jc, LNW) * CSEA
                        + CI(ic, jc, LA) * CSA + CI(ic, jc, LNE) * CSWA + CI(ic, jc, LR) * CWA;
        double CENW = SO(i - 1, j, KS) * CI(ic, jc, LSE);
        double CSENW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LSE) + SO(i, j - 1, KW) * CI(ic, jc, LB)
                     + SO(i - 1, j - 1, KS) * CI(ic, jc - 1, LR);
        double CSNW = SO(i - 1, j - 1, KW) * CI(ic, jc, LSE);
        SOC(ic, jc, KNW) = CI(ic, jc, LL) * CENW + CI(ic, jc, LNW) * CSENW + CI(ic - 1, jc, LA) * CSNW;
        CO = SO(i, j, KW) * CI(ic, jc, LR) + SO(i, j + 1, KS) * CI(ic, jc + 1, LB)
           + SO(i + 1, j, KW) * CI(ic + 1, jc, LL) + SO(i, j, KS) * CI(ic, jc, LA) - SO(i, j, KO);
        CW = -SO(i - 1, j, KO) * CI(ic, jc, LR) + SO(i - 1, j + 1, KS) * CI(ic, jc + 1, LSE)
           + SO(i, j, KW) + SO(i - 1, j, KS) * CI(ic, jc, LNE);
        CNW = -SO(i - 1, j + 1, KO) * CI(ic, jc + 1, LSE) + SO(i, j + 1, KW) * CI(ic, jc + 1, LB)
            + SO(i - 1, j + 1, KS) * CI(ic, jc, LR);
        CN = -SO(i, j + 1, KO) * CI(ic, jc + 1, LB) + SO(i, j + 1, KS)
           + SO(i, j + 1, KW) * CI(ic, jc + 1, LSE) + SO(i + 1, j + 1, KW) * CI(ic + 1, jc + 1, LSW);
        double CNE = -SO(i + 1, j + 1, KO) * CI(ic + 1, jc + 1, LSW) + SO(i + 1, j + 1, KS) * CI(ic + 1, jc, LL)
                   + SO(i + 1, j + 1, KW) * CI(ic, jc + 1, LB);
        double CE = -SO(i + 1, j, KO) * CI(ic + 1, jc, LL) + SO(i + 1, j, KS) * CI(ic + 1, jc, LNW)
                  + SO(i + 1, j, KW) + SO(i + 1, j + 1, KS) * CI(ic + 1, jc + 1, LSW);
        double CSE = -SO(i + 1, j - 1, KO) * CI(ic + 1, jc, LNW) + SO(i + 1, j - 1, KW) * CI(ic, jc, LA)
                   + SO(i + 1, j, KS) * CI(ic + 1, jc, LL);
        CS = -SO(i, j - 1, KO) * CI(ic, jc, LA) + SO(i, j - 1, KW) * CI(ic, jc, LNE) + SO(i, j, KS)
           + SO(i + 1, j - 1, KW) * CI(ic + 1, jc, LNW);
        CSW = -SO(i - 1, j - 1, KO) * CI(ic, jc, LNE) + SO(i - 1, j, KS) * CI(ic, jc, LR)
            + SO(i, j - 1, KW) * CI(ic, jc, LA);
        SOC(ic, jc, KO) = -CI(ic, jc + 1, LSE) * CNW - CI(ic, jc + 1, LB) * CN
                        - CI(ic + 1, jc + 1, LSW) * CNE - CI(ic, jc, LR) * CW - CO
                        - CI(ic + 1, jc, LL) * CE - CI(ic, jc, LNE) * CSW
                        - CI(ic, jc, LA) * CS - CI(ic + 1, jc, LNW) * CSE;
    }
#undef SO
#undef CI
#undef SOC
}


// periodic images of the coarse operator (all 5 planes): rows first, then columns
// (src/2d/ftn/BMG2_SymStd_SETUP_ITLI_ex.f90:219-246)
__global__ __launch_bounds__(256) void soc_ghost_y_k(double *__restrict__ soc, int iic, int jjc) {
    const int i = (int)(blockIdx.x * 256 + threadIdx.x);
    if (i >= iic) return;
    const std::size_t Pc = (std::size_t)iic * jjc;
    soc += (std::size_t)blockIdx.z * 5 * Pc;
    for (int k = 0; k < 5; ++k) {
        double *s = soc + k * Pc;
        s[(std::size_t)(jjc - 1) * iic + i] = s[(std::size_t)iic + i];
        s[i] = s[(std::size_t)(jjc - 2) * iic + i];
    }
}
__global__ __launch_bounds__(256) void soc_ghost_x_k(double *__restrict__ soc, int iic, int jjc) {
    const int j = (int)(blockIdx.x * 256 + threadIdx.x);
    if (j >= jjc) return;
    const std::size_t Pc = (std::size_t)iic * jjc;
    soc += (std::size_t)blockIdx.z * 5 * Pc;
    for (int k = 0; k < 5; ++k) {
        double *s = soc + k * Pc + (std::size_t)j * iic;
        s[iic - 1] = s[1];
        s[0] = s[iic - 2];
    }
}

// ---- coarsest grid, periodic: dense matrix, Cholesky, solve with mean removal ----------------
// Assembly of the upper triangle as src/2d/ftn/BMG2_SymStd_SETUP_cg_LU.f90:119-227 (9-point)
// and :251-335 (5-point) write it (one thread: the writes overlap by design), then an upper
// Cholesky in DPOTF2's order: each pivot by one lane, the row of U across the workgroup, every
// entry's dot product summed in index order.  ABD(n, n) column-major, n = nx*ny, per problem.
__global__ __launch_bounds__(256) void setup_cg_per_k(const double *__restrict__ so, int nstncl,
                                                      double *__restrict__ abd, int ii, int jj,
                                                      int jpn, int *__restrict__ info) {
    const int i1 = ii - 1, j1 = jj - 1, i2 = i1 - 1, n = i2 * (j1 - 1);
    const std::size_t P = (std::size_t)ii * jj;
    so += (std::size_t)blockIdx.x * nstncl * P;
    abd += (std::size_t)blockIdx.x * n * n;
    for (std::size_t t = threadIdx.x; t < (std::size_t)n * n; t += blockDim.x) abd[t] = 0.0;
    __syncthreads();
    auto SO = [&](int i, int j, int k) { return so[(std::size_t)(k - 1) * P + (std::size_t)(j - 1) * ii + (i - 1)]; };
    auto A = [&](int r, int c) -> double & { return abd[(std::size_t)(c - 1) * n + (r - 1)]; };
    constexpr int KO = 1, KW = 2, KS = 3, KSW = 4, KNW = 5;
    const bool nine = nstncl == 5, px = per_x(jpn), py = per_y(jpn), pxy = jpn == 3 || jpn == -3;
    if (threadIdx.x == 0) {
        int kk = 1;
        A(1, 1) = SO(2, 2, KO);
        for (int i = 3; i <= i1; ++i) {
            ++kk;
            A(kk, kk) = SO(i, 2, KO);
            A(kk - 1, kk) = -SO(i, 2, KW);
        }
        if (px) A(kk - i2 + 1, kk) = -SO(ii, 2, KW);
        for (int j = 3; j <= j1; ++j) {
            if (px) A(kk, kk + 1) = nine ? -SO(2, j, KSW) : 0.0;
            for (int i = 2; i <= i1; ++i) {
                ++kk;
                A(kk, kk) = SO(i, j, KO);
                if (i != 2) {
                    A(kk - 1, kk) = -SO(i, j, KW);
                    A(kk - i2 - 1, kk) = nine ? -SO(i, j, KSW) : 0.0;
                }
                A(kk - i2 + 1, kk) = nine ? -SO(i + 1, j, KNW) : 0.0;
                A(kk - i2, kk) = -SO(i, j, KS);
            }
            if (px) {
                A(kk - i2 + 1, kk) = -SO(ii, j, KW);
                A(kk - 2 * i2 + 1, kk) = nine ? -SO(ii, j, KNW) : 0.0;
            }
        }
        if (py) {
            kk = kk - i2;
            const int j2 = (j1 - 2) * i2;
            ++kk;
            A(kk - j2, kk) = -SO(2, jj, KS);
            A(kk - j2 + 1, kk) = nine ? -SO(3, jj, KSW) : 0.0;
            if (pxy) A(i2, kk) = nine ? -SO(2, jj, KNW) : 0.0;
            for (int i = 3; i <= i1; ++i) {
                ++kk;
                A(kk - j2, kk) = -SO(i, jj, KS);
                A(kk - j2 - 1, kk) = nine ? -SO(i, jj, KNW) : 0.0;
                A(kk - j2 + 1, kk) = nine ? -SO(i + 1, jj, KSW) : 0.0;
            }
            A(kk - j2 + 1, kk) = 0.0;
            if (pxy) A(1, kk) = nine ? -SO(ii, jj, KSW) : 0.0;
            if (px) A(kk - 2 * i2 + 1, kk) = nine ? -SO(ii, j1, KNW) : 0.0;
        }
    }
    __syncthreads();
    __shared__ double piv;
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    for (int j = 1; j <= n; ++j) {
        if (threadIdx.x == 0) {
            double ajj = A(j, j);
            for (int k = 1; k < j; ++k) ajj -= A(k, j) * A(k, j);
            if (!(ajj > 0.0)) {
                A(j, j) = ajj;
                bad = j;
            } else {
                ajj = sqrt(ajj);
                A(j, j) = ajj;
            }
            piv = ajj;
        }
        __syncthreads();
        if (bad) break;
        for (int c = j + 1 + (int)threadIdx.x; c <= n; c += (int)blockDim.x) {
            double s = A(j, c);
            for (int k = 1; k < j; ++k) s -= A(k, j) * A(k, c);
            A(j, c) = s / piv;
        }
        __syncthreads();
    }
    if (threadIdx.x == 0 && bad) atomicMax(info, bad);
}

// DPOTRS on the factor, then the mean removal and the periodic images
// (src/2d/ftn/BMG2_SymStd_SOLVE_cg.f90:93-163); one lane per problem
template <typename T>
__global__ void solve_cg_per_k(T *__restrict__ q, const T *__restrict__ qf,
                               const double *__restrict__ abd, double *__restrict__ x, int ii,
                               int jj, int jpn) {
    if (threadIdx.x != 0) return;
    const int i1 = ii - 1, j1 = jj - 1, nx = ii - 2, n = nx * (jj - 2);
    q += (std::size_t)blockIdx.x * ii * jj;
    qf += (std::size_t)blockIdx.x * ii * jj;
    abd += (std::size_t)blockIdx.x * n * n;
    x += (std::size_t)blockIdx.x * n;
    auto A = [&](int r, int c) { return abd[(std::size_t)(c - 1) * n + (r - 1)]; };
    for (int kk = 0; kk < n; ++kk) x[kk] = (double)qf[pidx(kk % nx + 1, kk / nx + 1, ii)];
    for (int j = 1; j <= n; ++j) {
        double s = x[j - 1];
        for (int k = 1; k < j; ++k) s -= A(k, j) * x[k - 1];
        x[j - 1] = s / A(j, j);
    }
    for (int j = n; j >= 1; --j) {
        double s = x[j - 1];
        for (int k = j + 1; k <= n; ++k) s -= A(j, k) * x[k - 1];
        x[j - 1] = s / A(j, j);
    }
    // mean removal, sums in FP64 and in Fortran order (kk runs i fastest)
    double qint = 0.0, cint = 0.0;
    for (int kk = 0; kk < n; ++kk) {
        qint = qint + x[kk];
        cint = cint + 1.0;
    }
    const double c = -qint / cint;
    for (int kk = 0; kk < n; ++kk) q[pidx(kk % nx + 1, kk / nx + 1, ii)] = (T)(x[kk] + c);
    auto Q = [&](int i, int j) -> T & { return q[pidx(i - 1, j - 1, ii)]; };  // 1-based
    if (per_y(jpn))
        for (int i = 2; i <= i1; ++i) {
            Q(i, jj) = Q(i, 2);
            Q(i, 1) = Q(i, j1);
        }
    if (per_x(jpn))
        for (int j = 2; j <= j1; ++j) {
            Q(ii, j) = Q(2, j);
            Q(1, j) = Q(i1, j);
        }
    if (jpn == 3 || jpn == -3) {
        Q(1, 1) = Q(i1, j1);
        Q(ii, 1) = Q(2, j1);
        Q(1, jj) = Q(i1, 2);
        Q(ii, jj) = Q(2, 2);
    }
}

}  // namespace

template <typename T>
void relax_gs_per(const T *so, int nstncl, const T *qf, T *q, const T *sor, int ii, int jj,
                  int updown, int jpn, hipStream_t s, int nb) {
    if (nstncl == 5) {
        // per colour (i parity, j parity) as in relax_gs; after a colour the x images of the rows
        // it swept (the reference refreshes them row by row, src/2d/ftn/BMG2_SymStd_relax_GS.f90
        // :176-182)
        static const int order[4][2] = {{1, 1}, {0, 1}, {1, 0}, {0, 0}};
        const dim3 g = gridb(ii / 2 + 1, jj / 2 + 1, nb);
        for (int t = 0; t < 4; ++t) {
            const int c = updown == 0 ? t : 3 - t;
            gs_colour_k<T, true><<<g, 256, 0, s>>>(so, qf, q, sor, ii, jj, order[c][0], order[c][1], 1);
            if (per_x(jpn)) ghost_x<T>(q, ii, jj, order[c][1] == 1 ? 1 : 2, jj - 2, 2, s, nb);
        }
    } else {
        const dim3 g = gridb(ii / 2 + 1, jj - 2, nb);
        for (int t = 0; t < 2; ++t) {
            const int parity = updown == 0 ? t : 1 - t;
            gs_colour_k<T, false><<<g, 256, 0, s>>>(so, qf, q, sor, ii, jj, parity, 0, 1);
            if (per_x(jpn)) ghost_x<T>(q, ii, jj, 1, jj - 2, 1, s, nb);
        }
    }
    if (per_y(jpn)) ghost_y<T>(q, ii, jj, 0, ii - 1, s, nb);
}

template <typename T>
void restrict_per(const T *ci, T *q, T *qc, int iif, int jjf, int iic, int jjc, int jpn,
                  hipStream_t s, int nb) {
    // src/2d/ftn/BMG2_SymStd_restrict.f90:100-111: images of the fine grid refreshed in place
    // when the fine extent is even
    if (per_y(jpn) && jjf / 2 + 1 == jjc) ghost_y<T>(q, iif, jjf, 0, iif - 1, s, nb);
    if (per_x(jpn) && iif / 2 + 1 == iic) ghost_x<T>(q, iif, jjf, 0, jjf - 1, 1, s, nb);
    restrict_<T>(ci, q, qc, iif, jjf, iic, jjc, s, nb, 1);
}

template <typename T>
void interp_add_per(T *q, const T *qc, const T *res, const T *so, int nstncl, const T *ci, int iic,
                    int jjc, int iif, int jjf, int jpn, hipStream_t s, int nb) {
    interp_add<T>(q, qc, res, so, nstncl, ci, iic, jjc, iif, jjf, s, nb, 1);
    // src/2d/ftn/BMG2_SymStd_interp_add.f90:145-156
    if (per_y(jpn)) ghost_y<T>(q, iif, jjf, 0, iif - 1, s, nb);
    if (per_x(jpn)) ghost_x<T>(q, iif, jjf, 0, jjf - 1, 1, s, nb);
}

void setup_interp_per(const double *so, int nstncl, double *ci, int iif, int jjf, int iic, int jjc,
                      int jpn, hipStream_t s, int nb) {
    oi_bounds B;
    const int iicf = (iif - 2) / 2 + 3, jjcf = (jjf - 2) / 2 + 3;
    B.iifc = 2 * (iicf - 2) + 2;
    B.jjfc = 2 * (jjcf - 2) + 2;
    B.ibeg = 2; B.ibegc = 3; B.ibeg_x = 2; B.iend_x = iif - 2; B.iendc = iicf - 1;
    B.jendc = jjcf - 1;
    if (per_x(jpn)) {
        B.ibeg = 0;
        B.ibegc = 2;
        if (iic == iicf) {
            B.iendc = iicf;
            B.ibeg_x = 3;
            B.iend_x = iif - 1;
        }
    }
    B.jbeg = 2; B.jbegc = 3; B.jbeg_y = 2; B.jend_y = jjf - 2;
    if (per_y(jpn)) {
        B.jbeg = 0;
        B.jbegc = 2;
        if (jjc == jjcf) {
            B.jendc = jjcf;
            B.jbeg_y = 3;
            B.jend_y = jjf - 1;
        }
    }
    const int ex = per_y(jpn) ? 2 : 0, ey = per_x(jpn) ? 2 : 0;
    const int nic = B.iendc - B.ibegc + 1, njc = B.jendc - B.jbegc + 1;
    const dim3 gx = gridb(nic, jjc - 2 + ex, nb), gy = gridb(iic - 2 + ey, njc, nb);
    const dim3 gc = gridb(nic, njc, nb);
    if (nstncl == 5) {
        if (nic > 0) oi_per_xedge_k<true><<<gx, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc, B, ex);
        if (njc > 0) oi_per_yedge_k<true><<<gy, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc, B, ey);
        if (nic > 0 && njc > 0)
            oi_per_corner_k<true><<<gc, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc, B);
    } else {
        if (nic > 0) oi_per_xedge_k<false><<<gx, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc, B, ex);
        if (njc > 0) oi_per_yedge_k<false><<<gy, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc, B, ey);
        if (nic > 0 && njc > 0)
            oi_per_corner_k<false><<<gc, 256, 0, s>>>(so, ci, iif, jjf, iic, jjc, B);
    }
}

void setup_galerkin_per(const double *so, int nstncl, const double *ci, double *soc, int iif,
                        int jjf, int iic, int jjc, int jpn, hipStream_t s, int nb) {
    const dim3 g = gridb(iic - 2, jjc - 2, nb);
    if (nstncl == 5)
        galerkin_itli_k<true><<<g, 256, 0, s>>>(so, ci, soc, iif, jjf, iic, jjc);
    else
        galerkin_itli_k<false><<<g, 256, 0, s>>>(so, ci, soc, iif, jjf, iic, jjc);
    if (per_y(jpn))
        soc_ghost_y_k<<<dim3((unsigned)((iic + 255) / 256), 1, (unsigned)nb), 256, 0, s>>>(soc, iic, jjc);
    if (per_x(jpn))
        soc_ghost_x_k<<<dim3((unsigned)((jjc + 255) / 256), 1, (unsigned)nb), 256, 0, s>>>(soc, iic, jjc);
}

void setup_cg_per(const double *so, int nstncl, double *abd, int ii, int jj, int jpn, int *info,
                  hipStream_t s, int nb) {
    setup_cg_per_k<<<nb, 256, 0, s>>>(so, nstncl, abd, ii, jj, jpn, info);
}

template <typename T>
void solve_cg_per(T *q, const T *qf, const double *abd, double *bbd, int ii, int jj, int jpn,
                  hipStream_t s, int nb) {
    solve_cg_per_k<T><<<nb, 64, 0, s>>>(q, qf, abd, bbd, ii, jj, jpn);
}

template <typename T>
void periodic_images(T *q, int ii, int jj, int jpn, hipStream_t s, int nb) {
    if (per_y(jpn)) ghost_y<T>(q, ii, jj, 0, ii - 1, s, nb);
    if (per_x(jpn)) ghost_x<T>(q, ii, jj, 0, jj - 1, 1, s, nb);
}

template <typename T>
void copy(const T *src, T *dst, std::size_t n, hipStream_t s) {
    convert_k<T, T><<<grid1(n), 256, 0, s>>>(src, dst, n);
}

// explicit instantiations
#define CDR_INST(T)                                                                               \
    template void residual<T>(const T *, int, const T *, const T *, T *, int, int,                \
        hipStream_t, int, int);                                                                   \
    template void residual_norm<T>(const T *, int, const T *, const T *, T *, int, int, double    \
        *, double *, hipStream_t, int, int);                                                      \
    template void sumsq<T>(const T *, int, int, double *, double *, hipStream_t, int);            \
    template void relax_gs<T>(const T *, int, const T *, T *, const T *, int, int, int,           \
        hipStream_t, int, int);                                                                   \
    template void transpose<T>(const T *, T *, int, int, hipStream_t, int);                       \
    template void transpose_op<T>(const T *, T *, int, int, int, hipStream_t, int);               \
    template void residual_qT<T>(const T *, int, const T *, const T *, T *, int, int,             \
        hipStream_t, int, int);                                                                   \
    template void interp_add_qT<T>(T *, const T *, const T *, const T *, int, const T *, int,     \
        int, int, int, hipStream_t, int, int);                                                    \
    template void restrict_<T>(const T *, const T *, T *, int, int, int, int, hipStream_t,        \
        int, int);                                                                                \
    template void restrict_cycle<T>(const T *, const T *, T *, T *, T *, int, int, int, int,      \
        hipStream_t, int, int);                                                                   \
    template void interp_add<T>(T *, const T *, const T *, const T *, int, const T *, int,        \
        int, int, int, hipStream_t, int, int);                                                    \
    template void solve_cg<T>(T *, const T *, const double *, double *, int, int, hipStream_t,    \
        int, int);                                                                                \
    template void fill<T>(T *, T, std::size_t, hipStream_t);                                      \
    template void relax_gs_per<T>(const T *, int, const T *, T *, const T *, int, int, int,       \
        int, hipStream_t, int);                                                                   \
    template void restrict_per<T>(const T *, T *, T *, int, int, int, int, int, hipStream_t,      \
        int);                                                                                     \
    template void interp_add_per<T>(T *, const T *, const T *, const T *, int, const T *, int,    \
        int, int, int, int, hipStream_t, int);                                                    \
    template void solve_cg_per<T>(T *, const T *, const double *, double *, int, int, int,        \
        hipStream_t, int);                                                                        \
    template void copy<T>(const T *, T *, std::size_t, hipStream_t);                              \
    template void periodic_images<T>(T *, int, int, int, hipStream_t, int);
CDR_INST(double)
CDR_INST(float)
#undef CDR_INST
template void fill<int>(int *, int, std::size_t, hipStream_t);
template void convert<double, float>(const double *, float *, std::size_t, hipStream_t);
template void convert<float, double>(const float *, double *, std::size_t, hipStream_t);

}  // namespace k2
}  // namespace cdr
