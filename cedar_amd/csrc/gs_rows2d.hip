// Nine-point Gauss-Seidel, both colours of a row in one launch
// (src/2d/ftn/BMG2_SymStd_relax_GS.f90:137-181; colours and operation order as gs_colour_k of
// bmg2_kernels.hip, built with -ffp-contract=off, so bitwise the same).
#include "bmg2_launch.hpp"
#include "row_pairs.hpp"
#include "tile_order.hpp"

#include <hip/hip_runtime.h>

namespace cdr {
namespace k2 {

namespace {

// The four colours (i parity, j parity) come in the order (1,1) (0,1) (1,0) (0,0) or its
// reverse, so the two colours of a row follow each other, and the second needs from the first
// only the new values in its own row: rows of the other parity do not change between them.  One
// launch relaxes the rows of one parity, W threads per row with PP pairs (odd point, even point)
// each: the first colour's values go through LDS to the second, whose other products are formed
// beforehand and wait in registers.  Bound by memory: a row's operator and iterate are read once
// instead of once per colour with every other point unused.  A sweep of 2047 x 1500 in FP64 takes
// 2 x 24.5 us, where one launch per colour took 4 x 25.8; below 512 points a side, where a launch
// costs 3.3 to 4.8 us whatever it does, half the launches.
//
// ODD: the odd points of a row come first.  The launcher gives R rows to a workgroup of W * R
// threads; no point outside the launch's rows changes during it.
template <typename T, int W, int PP, bool ODD>
__global__ __launch_bounds__(W < 256 ? 256 : W) void gs9_rows_k(const T *__restrict__ so,
                                                                const T *__restrict__ qf,
                                                                T *__restrict__ q,
                                                                const T *__restrict__ sor, int ii,
                                                                int jj, int first, int rep, int rev) {
    constexpr int R = W < 256 ? 256 / W : 1;
    __shared__ T fresh[R][W * PP + 2];  // [t + 1]: the first colour's value of pair t
    const int tx = threadIdx.x % W, r = threadIdx.x / W;
    const wg_pos g = tiled_wg(rep);
    const std::size_t P = (std::size_t)ii * jj, bz = g.z, bo = operator_of(bz, rep);
    const int blk = rev ? (int)gridDim.x - 1 - g.x : g.x;
    const int j = first + 2 * (blk * R + r);
    const bool row = j <= jj - 2;
    const int np = (ii - 1) / 2;  // pairs of the row; the last may lack its even point
    so += bo * 5 * P;
    qf += bz * P;
    q += bz * P;
    sor += bo * 2 * P;
    const T *w = so + P * KW, *s = so + P * KS, *sw = so + P * KSW, *nw = so + P * KNW;
    T kf[PP], kl[PP], kr[PP], kprod[PP][6], krec[PP], kedge[PP], first_v[PP];
#pragma unroll
    for (int u = 0; u < PP; ++u) {
        const int t = tx + u * W;
        if (!row || t >= np) continue;
        const std::size_t p = (std::size_t)j * ii + 2 * t + 1, pn = p + ii, pm = p - ii;
        const bool has1 = 2 * t + 2 <= ii - 2;
        const row_pair<T> f = load2(qf + p), rc = load2(sor + P + p);
        const row_pair<T> w0 = load2(w + p), w1 = load2_next(w + p, has1);
        const row_pair<T> s0 = load2(s + p), s1 = load2(s + pn);
        const row_pair<T> a0 = load2(sw + p), a1 = load2_next(sw + pn, has1);
        const row_pair<T> b0 = load2_next(nw + p, has1), b1 = load2(nw + pn);
        const row_pair<T> ql = load2(q + p - 1), qr = load2_next(q + p, has1);
        const row_pair<T> dl = load2(q + pm - 1), dr = load2_next(q + pm, has1);
        const row_pair<T> ul = load2(q + pn - 1), ur = load2_next(q + pn, has1);
        __builtin_amdgcn_sched_barrier(0);  // every load in flight before the first product
        // odd point p between ql.a and qr.a, even point p + 1 between ql.b and qr.b
        T v;
        if (ODD) {
            v = f.a + w0.a * ql.a + w0.b * qr.a;
            v = v + s0.a * dl.b + s1.a * ul.b;
            v = v + a0.a * dl.a + b0.a * dr.a;
            v = v + b1.a * ul.a + a1.a * ur.a;
            v = v * rc.a;
            kf[u] = f.b;
            kl[u] = w0.b;
            kr[u] = w1.b;
            kprod[u][0] = s0.b * dr.a;
            kprod[u][1] = s1.b * ur.a;
            kprod[u][2] = a0.b * dl.b;
            kprod[u][3] = b0.b * dr.b;
            kprod[u][4] = b1.b * ul.b;
            kprod[u][5] = a1.b * ur.b;
            krec[u] = rc.b;
            kedge[u] = qr.b;
        } else {
            v = f.b + w0.b * ql.b + w1.b * qr.b;
            v = v + s0.b * dr.a + s1.b * ur.a;
            v = v + a0.b * dl.b + b0.b * dr.b;
            v = v + b1.b * ul.b + a1.b * ur.b;
            v = has1 ? v * rc.b : qr.a;  // no even point: the boundary value there
            kf[u] = f.a;
            kl[u] = w0.a;
            kr[u] = w0.b;
            kprod[u][0] = s0.a * dl.b;
            kprod[u][1] = s1.a * ul.b;
            kprod[u][2] = a0.a * dl.a;
            kprod[u][3] = b0.a * dr.a;
            kprod[u][4] = b1.a * ul.a;
            kprod[u][5] = a1.a * ur.a;
            krec[u] = rc.a;
            kedge[u] = ql.a;
        }
        first_v[u] = v;
        fresh[r][t + 1] = v;
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PP; ++u) {
        const int t = tx + u * W;
        if (!row || t >= np) continue;
        const std::size_t p = (std::size_t)j * ii + 2 * t + 1;
        const bool has1 = 2 * t + 2 <= ii - 2;
        const T left = ODD ? first_v[u] : (t > 0 ? fresh[r][t] : kedge[u]);
        const T right = ODD ? (t + 1 < np ? fresh[r][t + 2] : kedge[u]) : first_v[u];
        T v = kf[u] + kl[u] * left + kr[u] * right;
#pragma unroll
        for (int k = 0; k < 6; ++k) v = v + kprod[u][k];
        v = v * krec[u];
        const T odd = ODD ? first_v[u] : v, even = ODD ? v : first_v[u];
        if (has1)
            store2(q + p, odd, even);
        else
            q[p] = odd;
    }
}

template <typename T, int W, int PP>
void launch_rows(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int updown,
                 hipStream_t s, int nb, int rep) {
    constexpr int NT = W < 256 ? 256 : W, R = NT / W;
    for (int t = 0; t < 2; ++t) {
        const int first = (updown == 0) == (t == 0) ? 1 : 2;  // rows of odd index first going down
        if (first > jj - 2) continue;
        const int rows = (jj - 2 - first) / 2 + 1;
        const dim3 g((unsigned)((rows + R - 1) / R), 1, (unsigned)nb);
        if (updown == 0)
            gs9_rows_k<T, W, PP, true><<<g, NT, 0, s>>>(so, qf, q, sor, ii, jj, first, rep, t);
        else
            gs9_rows_k<T, W, PP, false><<<g, NT, 0, s>>>(so, qf, q, sor, ii, jj, first, rep, t);
    }
}

}  // namespace

template <typename T>
bool relax_gs9_rows(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int updown,
                    hipStream_t s, int nb, int rep) {
    const int np = (ii - 1) / 2;
    if (np <= 32)
        launch_rows<T, 32, 1>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else if (np <= 64)
        launch_rows<T, 64, 1>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else if (np <= 128)
        launch_rows<T, 128, 1>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else if (np <= 256)
        launch_rows<T, 256, 1>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else if (np <= 512)
        launch_rows<T, 256, 2>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else if (np <= 1024)
        launch_rows<T, 512, 2>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else if (np <= 2048)
        launch_rows<T, 1024, 2>(so, qf, q, sor, ii, jj, updown, s, nb, rep);
    else
        return false;
    return true;
}

template bool relax_gs9_rows<double>(const double *, const double *, double *, const double *, int,
                                     int, int, hipStream_t, int, int);
template bool relax_gs9_rows<float>(const float *, const float *, float *, const float *, int, int,
                                    int, hipStream_t, int, int);

}  // namespace k2
}  // namespace cdr
