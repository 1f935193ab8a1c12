// Periodic zebra line relaxation (src/2d/ftn/BMG2_SymStd_relax_lines_x.f90:170-300,
// _y.f90:176-310): lines of a periodic grid, solved in the reference's sequential DPTTRS order
// and, where the line direction itself is periodic, corrected by Sherman-Morrison with the solve
// z = T^-1 B of the wrap couplings.  Layout and batching as in bmg2_kernels.hip; built with
// -ffp-contract=off, so every operation rounds as the reference's.
#include "bmg2_launch.hpp"

#include <hip/hip_runtime.h>

namespace cdr {
namespace k2 {

namespace {

__host__ __device__ inline bool per_x(int jpn) { return jpn == 2 || jpn == 3 || jpn == -2 || jpn == -3; }
__host__ __device__ inline bool per_y(int jpn) { return jpn == 1 || jpn == 3 || jpn == -1 || jpn == -3; }

// Right-hand side of point p on an x-line (DIR 0) or y-line (DIR 1): f and the couplings to the
// neighbouring lines.  W(i, j) lives at the point, its right neighbour's W is the coupling to it.
template <typename T, bool NINE, int DIR>
__device__ inline T per_rhs(const T *__restrict__ so, const T *__restrict__ qf, const T *q,
                            std::size_t P, std::size_t p, int ii) {
    T v;
    if (DIR == 0)
        v = qf[p] + so[P * KS + p] * q[p - ii] + so[P * KS + p + ii] * q[p + ii];
    else
        v = qf[p] + so[P * KW + p] * q[p - 1] + so[P * KW + p + 1] * q[p + 1];
    if (NINE)
        v = v + so[P * KSW + p] * q[p - ii - 1] + so[P * KNW + p + 1] * q[p - ii + 1] +
            so[P * KNW + p + ii] * q[p + ii - 1] + so[P * KSW + p + ii + 1] * q[p + ii + 1];
    return v;
}

// v[k] = v[k] - v[k -+ 1] * e over a whole vector in LDS by one lane, upwards (e = E[k-1]) or
// downwards (e = E[k]).  The recurrence is a chain of one product and one difference per element;
// the operands of the next block of U are read while the chain runs through the current one.
template <typename T, bool UP>
__device__ inline void chain(T *v, const T *E, int n) {
    constexpr int U = 8;
    T prev = UP ? v[0] : v[n - 1];
    auto at = [&](int t) { return UP ? t : n - 1 - t; };  // position of element t of the chain
    int t = 1;
    if (t + U <= n) {
        T x[U], e[U], y[U], g[U];
        auto load = [&](int t) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                x[u] = v[at(t + u)];
                e[u] = E[UP ? t + u - 1 : at(t + u)];
            }
        };
        load(t);
        for (; t + U <= n; t += U) {
#pragma unroll
            for (int u = 0; u < U; ++u) {
                y[u] = x[u];
                g[u] = e[u];
            }
            load(min(t + U, n - U));
#pragma unroll
            for (int u = 0; u < U; ++u) y[u] = prev = y[u] - prev * g[u];
#pragma unroll
            for (int u = 0; u < U; ++u) v[at(t + u)] = y[u];
        }
    }
    for (; t < n; ++t) v[at(t)] = prev = v[at(t)] - prev * E[UP ? t - 1 : at(t)];
}

// One colour of lines, G lines per workgroup, lines held in LDS: right-hand sides by all threads
// (row-contiguous loads), the two recurrences by one lane per vector (the line's right-hand side
// and, with sm, its Sherman-Morrison vector on another lane of the same wavefront), the divisions
// between them and the correction by all threads again.  Bound by the recurrences, n dependent
// products and differences per sweep; the launcher takes G small as long as every line of a colour
// then runs at once (lines_per_group).  With one lane per line walking memory the 512 x 511 FP64
// Poisson sweep took 765 us (x) and 420 us (y) per colour.
//
// img: this launch also writes the periodic images that only it or later sweeps read.
//   1: the lines run along the one periodic direction; each line's own images, and those of the
//      two lines beyond the grid (their interior is not relaxed);
//   2: the lines run across the one periodic direction and this is the sweep's second colour,
//      which owns exactly one of the two lines at the seam (an even number of lines): its
//      workgroup writes both image lines once it has read them.
template <typename T, bool NINE, int DIR, int G>
__global__ __launch_bounds__(256) void relax_lines_per_k(const T *__restrict__ so,
                                                         const T *__restrict__ qf, T *q,
                                                         const T *__restrict__ sor, int ii, int jj,
                                                         int first, int sm, int img) {
    extern __shared__ __align__(16) unsigned char lds_raw[];
    constexpr int NT = 256;
    const int tid = threadIdx.x;
    const int nl = DIR == 0 ? jj - 2 : ii - 2, n = DIR == 0 ? ii - 2 : jj - 2;
    const int L0 = first + 2 * G * (int)blockIdx.x;  // lines L0, L0 + 2, ... of this workgroup
    const int ng = min(G, (nl - L0) / 2 + 1);
    const std::size_t P = (std::size_t)ii * jj, bz = blockIdx.y;
    so += bz * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    sor += bz * 2 * P;
    const int ld = n | 1;
    T *B = reinterpret_cast<T *>(lds_raw), *E = B + G * ld, *Z = E + G * ld;
    const std::size_t ldf = DIR == 0 ? ii : jj;  // the factors of a line are contiguous
    auto pos = [&](int L, int k) {
        return DIR == 0 ? (std::size_t)L * ii + k + 1 : (std::size_t)(k + 1) * ii + L;
    };
    // element t of the workgroup's ng * n points, in the order of q's memory
    auto split = [&](int t, int &g, int &k) {
        if (DIR == 0) {
            g = G == 1 ? 0 : t / n;
            k = t - g * n;
        } else {
            g = t % G;
            k = t / G;
        }
    };
    const int cnt = (DIR == 0 ? ng : G) * n;
    for (int t = tid; t < cnt; t += NT) {
        int g, k;
        split(t, g, k);
        if (g < ng) B[g * ld + k] = per_rhs<T, NINE, DIR>(so, qf, q, P, pos(L0 + 2 * g, k), ii);
    }
    for (int t = tid; t < ng * n; t += NT) {
        const int g = t / n, k = t - g * n, L = L0 + 2 * g;
        if (k < n - 1) E[g * ld + k] = sor[P + L * ldf + k + 2];
        if (sm) {
            T z = T(0);
            if (k == 0) z = DIR == 0 ? -so[P * KW + (std::size_t)L * ii + 1] : -so[P * KS + (std::size_t)ii + L];
            if (k == n - 1)
                z = DIR == 0 ? -so[P * KW + (std::size_t)L * ii + ii - 1]
                             : -so[P * KS + (std::size_t)(jj - 1) * ii + L];
            Z[g * ld + k] = z;
        }
    }
    __syncthreads();
    const int nv = sm ? 2 * ng : ng;  // vectors of the workgroup: right-hand sides, then z
    T *mine = tid < ng ? B + tid * ld : Z + (tid - ng) * ld;
    const T *myE = E + (tid < ng ? tid : tid - ng) * ld;
    if (tid < nv) chain<T, true>(mine, myE, n);
    __syncthreads();
    for (int t = tid; t < ng * n; t += NT) {
        const int g = t / n, k = t - g * n;
        const T d = sor[(L0 + 2 * g) * ldf + k + 1];
        B[g * ld + k] = B[g * ld + k] / d;
        if (sm) Z[g * ld + k] = Z[g * ld + k] / d;
    }
    __syncthreads();
    if (tid < nv) chain<T, false>(mine, myE, n);
    __syncthreads();
    for (int t = tid; t < cnt; t += NT) {
        int g, k;
        split(t, g, k);
        if (g >= ng) continue;
        const int L = L0 + 2 * g;
        T v = B[g * ld + k];
        if (sm) {
            const T alpha = Z[g * ld] + Z[g * ld + n - 1];
            T beta = B[g * ld] + B[g * ld + n - 1];
            beta = beta / (T(1) + alpha);
            v = v - beta * Z[g * ld + k];
        }
        q[pos(L, k)] = v;
        if (img == 1) {
            const int far = k == 0 ? n : k == n - 1 ? -1 : -2;  // position of the image of point k
            if (far >= -1) q[pos(L, far)] = v;
        } else if (img == 2 && (L == 1 || L == nl)) {
            q[pos(L == 1 ? nl + 1 : 0, k)] = v;                     // the image of this line
            q[pos(L == 1 ? 0 : nl + 1, k)] = q[pos(L == 1 ? nl : 1, k)];  // and of the other one
        }
    }
    if (img == 1) {
        // the lines beyond the grid: line 0 is read by line 1 alone, which the first workgroup
        // relaxes or no workgroup of this launch does; line nl + 1 and the last one likewise
        for (int L = 0; L <= nl + 1; L += nl + 1)
            if (tid == 0 && blockIdx.x == (L == 0 ? 0 : gridDim.x - 1)) {
                q[pos(L, -1)] = q[pos(L, n - 1)];
                q[pos(L, n)] = q[pos(L, 0)];
            }
    } else if (img == 2 && tid < 2) {
        // the ends of the two image lines, outside the lines' own range
        for (int g = 0; g < ng; ++g) {
            const int L = L0 + 2 * g, k = tid == 0 ? -1 : n;
            if (L != 1 && L != nl) continue;
            q[pos(0, k)] = q[pos(nl, k)];
            q[pos(nl + 1, k)] = q[pos(1, k)];
        }
    }
}

// Lines too long for LDS: one lane per line walks memory, z kept in the scratch at the line's
// positions.  Same operations in the same order.
template <typename T, bool NINE, int DIR>
__global__ __launch_bounds__(64) void relax_lines_per_long_k(const T *__restrict__ so,
                                                             const T *__restrict__ qf, T *q,
                                                             const T *__restrict__ sor, T *z, int ii,
                                                             int jj, int first, int sm) {
    const int L = first + 2 * (int)(blockIdx.x * 64 + threadIdx.x);
    if (L > (DIR == 0 ? jj - 2 : ii - 2)) return;
    const std::size_t P = (std::size_t)ii * jj, bz = blockIdx.y;
    so += bz * (NINE ? 5 : 3) * P;
    qf += bz * P;
    q += bz * P;
    z += bz * P;
    sor += bz * 2 * P;
    const int n = DIR == 0 ? ii - 2 : jj - 2;
    auto pos = [&](int k) {
        return DIR == 0 ? (std::size_t)L * ii + k + 1 : (std::size_t)(k + 1) * ii + L;
    };
    const T *D = sor + (std::size_t)L * (DIR == 0 ? ii : jj) + 1, *E = D + P + 1;
    for (int k = 0; k < n; ++k) q[pos(k)] = per_rhs<T, NINE, DIR>(so, qf, q, P, pos(k), ii);
    auto dpttrs = [&](T *b) {
        if (n <= 1) {
            b[pos(0)] = b[pos(0)] * (T(1) / D[0]);
            return;
        }
        for (int k = 1; k < n; ++k) b[pos(k)] = b[pos(k)] - b[pos(k - 1)] * E[k - 1];
        b[pos(n - 1)] = b[pos(n - 1)] / D[n - 1];
        for (int k = n - 2; k >= 0; --k) b[pos(k)] = b[pos(k)] / D[k] - b[pos(k + 1)] * E[k];
    };
    dpttrs(q);
    if (!sm) return;
    for (int k = 0; k < n; ++k) z[pos(k)] = T(0);
    if (DIR == 0) {
        z[pos(0)] = -so[P * KW + (std::size_t)L * ii + 1];
        z[pos(n - 1)] = -so[P * KW + (std::size_t)L * ii + ii - 1];
    } else {
        z[pos(0)] = -so[P * KS + (std::size_t)ii + L];
        z[pos(n - 1)] = -so[P * KS + (std::size_t)(jj - 1) * ii + L];
    }
    dpttrs(z);
    const T alpha = z[pos(0)] + z[pos(n - 1)];
    T beta = q[pos(0)] + q[pos(n - 1)];
    beta = beta / (T(1) + alpha);
    for (int k = 0; k < n; ++k) q[pos(k)] = q[pos(k)] - beta * z[pos(k)];
}

// LDS of one workgroup: per line its right-hand side, multipliers and (sm) z
constexpr std::size_t kLineLdsMax = 128 * 1024;
template <typename T>
std::size_t line_lds(int n, int G, int sm) {
    return (std::size_t)(n | 1) * sizeof(T) * G * (sm ? 3 : 2);
}

template <typename T, bool NINE, int DIR, int G>
void launch_per(const T *so, const T *qf, T *q, const T *sor, int ii, int jj, int first, int sm,
                int img, int lines, hipStream_t s, int nb) {
    const std::size_t lds = line_lds<T>(DIR == 0 ? ii - 2 : jj - 2, G, sm);
    if (lds > 64 * 1024)
        (void)hipFuncSetAttribute(reinterpret_cast<const void *>(relax_lines_per_k<T, NINE, DIR, G>),
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLineLdsMax);
    relax_lines_per_k<T, NINE, DIR, G><<<dim3((unsigned)((lines + G - 1) / G), (unsigned)nb), 256,
                                         lds, s>>>(so, qf, q, sor, ii, jj, first, sm, img);
}

// Lines per workgroup where a colour has cnt lines (of all problems) of n points: 64, 16, or gw, one for
// x-lines and four for y-lines.  A workgroup costs 7 us however short its lines, and the chip runs about
// 1024 at once, so beyond that many of gw lines short ones share workgroups.  A sweep of 65536 x-lines of
// 8 points (FP64, nine-point, wrap in x) takes 182 us by one line and 23 by 16; of 2 points 153 by one,
// 14 by 16 and 9 by 64, of 8 points no less by 64 than by 16.  Lines of more than 32 points give every
// thread work by themselves and share only at four times as many lines: 4096 FP32 x-lines of 48 points 15
// us by one, 18 by 16; 32768 FP64 ones of 64 points (five-point, no wrap) 163 and 37.  (One lane per line walking memory: 70
// us at 65536 x 8, 131 at 32768 x 64.)
constexpr int kLongestShared = 128;
inline int lines_per_group(int n, std::size_t cnt, int gw) {
    if (n > kLongestShared || cnt <= (std::size_t)1024 * gw * (n <= 32 ? 1 : 4)) return gw;
    return n <= 4 ? 64 : 16;
}

template <typename T, bool NINE, int DIR>
void sweep_per(const T *so, const T *qf, T *q, const T *sor, T *work, int ii, int jj, int updown,
               int jpn, hipStream_t s, int nb) {
    const bool sm = DIR == 0 ? per_x(jpn) : per_y(jpn);
    const bool both = per_x(jpn) && per_y(jpn);
    const int nl = DIR == 0 ? jj - 2 : ii - 2, n = DIR == 0 ? ii - 2 : jj - 2;
    // y-lines: four neighbouring columns of a colour share the 64-byte pieces of the rows they
    // read; x-lines are contiguous by themselves.  A single line where four do not fit.
    constexpr int GW = DIR == 0 ? 1 : 4;
    const bool fits = n >= 2 && line_lds<T>(n, 1, sm) <= kLineLdsMax;
    const bool wide = line_lds<T>(n, GW, sm) <= kLineLdsMax;
    // the images that the kernel itself can write (see there): one periodic direction, and an
    // even number of lines where they run across it
    const bool own = fits && !both && nl >= 2 && (sm || nl % 2 == 0);
    for (int pass = 0; pass < 2; ++pass) {
        // DOWN relaxes the lines of odd Fortran index 3, 5, ... (C index 2, 4, ...) first
        const int first = (pass == 0) == (updown == 0) ? 2 : 1;
        const int cnt = first > nl ? 0 : (nl - first) / 2 + 1;
        const int img = !own ? 0 : sm ? 1 : pass == 1 ? 2 : 0;
        const int G = lines_per_group(n, (std::size_t)cnt * nb, GW);
        if (cnt > 0) {
            if (!fits)
                relax_lines_per_long_k<T, NINE, DIR><<<dim3((unsigned)((cnt + 63) / 64), (unsigned)nb),
                                                       64, 0, s>>>(so, qf, q, sor, work, ii, jj,
                                                                   first, sm);
            else if (G == 64)
                launch_per<T, NINE, DIR, 64>(so, qf, q, sor, ii, jj, first, sm, img, cnt, s, nb);
            else if (G == 16)
                launch_per<T, NINE, DIR, 16>(so, qf, q, sor, ii, jj, first, sm, img, cnt, s, nb);
            else if (wide)
                launch_per<T, NINE, DIR, GW>(so, qf, q, sor, ii, jj, first, sm, img, cnt, s, nb);
            else
                launch_per<T, NINE, DIR, 1>(so, qf, q, sor, ii, jj, first, sm, img, cnt, s, nb);
        }
        // images refreshed after each colour of lines along a periodic direction, else after the
        // sweep
        if (!own && (sm || pass == 1)) periodic_images<T>(q, ii, jj, jpn, s, nb);
    }
}

}  // namespace

template <typename T>
void relax_lines_per(int dir, const T *so, int nstncl, const T *qf, T *q, const T *sor, T *work,
                     int ii, int jj, int updown, int jpn, hipStream_t s, int nb) {
    if (dir == 0) {
        if (nstncl == 5)
            sweep_per<T, true, 0>(so, qf, q, sor, work, ii, jj, updown, jpn, s, nb);
        else
            sweep_per<T, false, 0>(so, qf, q, sor, work, ii, jj, updown, jpn, s, nb);
    } else {
        if (nstncl == 5)
            sweep_per<T, true, 1>(so, qf, q, sor, work, ii, jj, updown, jpn, s, nb);
        else
            sweep_per<T, false, 1>(so, qf, q, sor, work, ii, jj, updown, jpn, s, nb);
    }
}

#define CDR_INST(T)                                                                               \
    template void relax_lines_per<T>(int, const T *, int, const T *, T *, const T *, T *, int, int, \
                                     int, int, hipStream_t, int);
CDR_INST(double)
CDR_INST(float)

}  // namespace k2
}  // namespace cdr
