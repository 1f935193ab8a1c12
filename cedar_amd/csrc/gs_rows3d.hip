// 27-point Gauss-Seidel, both colours of a row in one launch
// (src/3d/ftn/BMG3_SymStd_relax_GS.f90:79-181; colours and operation order as gs27_colour_k of
// bmg3_kernels.hip, built with -ffp-contract=off, so bitwise the same).
#include "bmg3_launch.hpp"
#include "bmg3_stencil.hpp"
#include "row_pairs.hpp"

#include <hip/hip_runtime.h>

namespace cdr {
namespace k3 {

namespace {

template <int W>
constexpr int row_threads = W < 64 ? 64 : 256;

// As gs9_rows_k (gs_rows2d.hip): the eight colours come in pairs that differ only in the parity
// of i, and the second of a pair needs from the first only the new values in its own row.  One
// launch relaxes the rows of one (j, k) parity, W threads per row with one pair of points each
// (i = 2 t + 1 and 2 t + 2, 0-based).  ODD: the points at 2 t + 1 come first.  Short rows go into
// workgroups of one wavefront, so that a small level still spreads over the chip.  Four launches
// per sweep instead of eight: 4 x 13 us at 100^3 in FP64 (4 x 11 at 127 x 127 x 95 in FP32) and
// 4 x 3 to 5 us on the levels below, where the loads' latency is the bound (7.6 us per launch
// while the compiler waited for a few loads at a time).
template <typename T, int W, bool ODD>
__global__ __launch_bounds__(row_threads<W>, 1) __attribute__((amdgpu_waves_per_eu(1, 2)))
void gs27_rows_k(const T *__restrict__ so, const T *__restrict__ qf, T *__restrict__ q,
                 const T *__restrict__ sor, int ii, int jj, int kk, int j0, int k0, int nj, int rows,
                 int rev) {
    constexpr int R = row_threads<W> / W;
    __shared__ T fresh[R][W + 2];  // [t + 1]: the first colour's value of pair t
    const int t = threadIdx.x % W, r = threadIdx.x / W;
    const int blk = rev ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;
    const int row = blk * R + r;  // rows of the parity, j fastest
    const int j = j0 + 2 * (row % nj), k = k0 + 2 * (row / nj);
    const int np = (ii - 1) / 2;
    const bool in = row < rows && t < np;
    const std::size_t A = (std::size_t)ii * jj, P = A * kk;
    const std::size_t p = in ? (std::size_t)k * A + (std::size_t)j * ii + 2 * t + 1 : 0;
    const bool has1 = 2 * t + 2 <= ii - 2;
    T kf = T(0), kl = T(0), kr = T(0), krec = T(0), kedge = T(0), first = T(0), prod[26];
    if (in) {
        // q at i - 1 .. i + 2 of the 9 rows around the pair
        T qv[3][3][4];
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
            for (int b = 0; b < 3; ++b) {
                const T *qr = q + p + (std::ptrdiff_t)(c - 1) * (std::ptrdiff_t)A + (b - 1) * ii;
                const row_pair<T> lo = load2(qr - 1), hi = load2_next(qr, has1);
                qv[c][b][0] = lo.a;
                qv[c][b][1] = lo.b;
                qv[c][b][2] = hi.a;
                qv[c][b][3] = hi.b;
            }
        const row_pair<T> f = load2(qf + p), rc = load2(sor + P + p);
        row_pair<T> c[26];
        int n = 0;
#define ROW27_LOAD(di, dj, dk, plane, oi, oj, ok)                                                 \
    {                                                                                             \
        const T *cp = so + (std::size_t)((plane)-1) * P + p + (dj)*ii + (dk)*A;                   \
        c[n++] = (di) ? load2_next(cp, has1) : load2(cp);                                         \
    }
        NB27_LIST(ROW27_LOAD)
#undef ROW27_LOAD
        // every load in flight before the first product: left to itself the compiler waits for
        // them a few at a time
        __builtin_amdgcn_sched_barrier(0);
        T v = ODD ? f.a : f.b;
        n = 0;
#define ROW27_TERM(di, dj, dk, plane, oi, oj, ok)                                                 \
    {                                                                                             \
        const T a = c[n].a * qv[(ok) + 1][(oj) + 1][(oi) + 1];                                    \
        const T b = c[n].b * qv[(ok) + 1][(oj) + 1][(oi) + 2];                                    \
        v = v + (ODD ? a : b);                                                                    \
        prod[n++] = ODD ? b : a;                                                                  \
    }
        NB27_LIST(ROW27_TERM)
#undef ROW27_TERM
        kl = ODD ? c[0].b : c[0].a;  // the first and the fifth term couple the point to its row
        kr = ODD ? c[4].b : c[4].a;
        if (ODD) {
            first = v * rc.a;
            kf = f.b;
            krec = rc.b;
            kedge = qv[1][1][3];
        } else {
            first = has1 ? v * rc.b : qv[1][1][2];  // no second point: the boundary value there
            kf = f.a;
            krec = rc.a;
            kedge = qv[1][1][0];
        }
        fresh[r][t + 1] = first;
    }
    __syncthreads();
    if (!in) return;
    const T left = ODD ? first : (t > 0 ? fresh[r][t] : kedge);
    const T right = ODD ? (t + 1 < np ? fresh[r][t + 2] : kedge) : first;
    T v = kf + kl * left;
#pragma unroll
    for (int n = 1; n < 26; ++n) v = v + (n == 4 ? kr * right : prod[n]);
    v = v * krec;
    const T odd = ODD ? first : v, even = ODD ? v : first;
    if (has1)
        store2(q + p, odd, even);
    else
        q[p] = odd;
}

template <typename T, int W>
void launch_rows(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int kk, int updown,
                 hipStream_t s) {
    constexpr int R = row_threads<W> / W;
    for (int t = 0; t < 4; ++t) {
        // going down the colours run from (even, even, even) 0-based interior parity to (odd, odd,
        // odd): DOWN pts = 8 .. 1, rows (j, k) start at 2, 1 by the bits of pts - 1, i likewise
        const int b = updown == 0 ? 3 - t : t;
        const int j0 = 1 + (b & 1), k0 = 1 + (b >> 1);
        const int nj = (jj - 2 - j0) / 2 + 1, nk = (kk - 2 - k0) / 2 + 1;
        if (jj - 2 < j0 || kk - 2 < k0) continue;
        const int rows = nj * nk;
        const unsigned g = (unsigned)((rows + R - 1) / R);
        if (updown == 0)
            gs27_rows_k<T, W, false><<<g, row_threads<W>, 0, s>>>(so, qf, q, sor, ii, jj, kk, j0, k0,
                                                                     nj, rows, t & 1);
        else
            gs27_rows_k<T, W, true><<<g, row_threads<W>, 0, s>>>(so, qf, q, sor, ii, jj, kk, j0, k0,
                                                                     nj, rows, t & 1);
    }
}

}  // namespace

template <typename T>
bool relax_gs27_rows(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int kk,
                     int updown, hipStream_t s) {
    const int np = (ii - 1) / 2;
    if (np <= 8)
        launch_rows<T, 8>(so, qf, q, sor, ii, jj, kk, updown, s);
    else if (np <= 16)
        launch_rows<T, 16>(so, qf, q, sor, ii, jj, kk, updown, s);
    else if (np <= 32)
        launch_rows<T, 32>(so, qf, q, sor, ii, jj, kk, updown, s);
    else if (np <= 64)
        launch_rows<T, 64>(so, qf, q, sor, ii, jj, kk, updown, s);
    else if (np <= 128)
        launch_rows<T, 128>(so, qf, q, sor, ii, jj, kk, updown, s);
    else if (np <= 256)
        launch_rows<T, 256>(so, qf, q, sor, ii, jj, kk, updown, s);
    else
        return false;
    return true;
}

template bool relax_gs27_rows<double>(const double *, const double *, double *, const double *, int,
                                      int, int, int, hipStream_t);
template bool relax_gs27_rows<float>(const float *, const float *, float *, const float *, int, int,
                                     int, int, hipStream_t);

}  // namespace k3
}  // namespace cdr
