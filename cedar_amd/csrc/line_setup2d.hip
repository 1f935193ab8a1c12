// Line relaxation setup (src/2d/ftn/BMG2_SymStd_SETUP_lines_{x,y}.f90): diag = c, off = -w (x) or
// -s (y), then LAPACK DPTTRF per line.  x factors: sor[0][p] = D, sor[1][p] = E at (i, j) as in the
// reference; y factors stored transposed: plane k element (j, i) at k*ii*jj + i*jj + j.
#include "bmg2_launch.hpp"

#include <hip/hip_runtime.h>

namespace cdr {
namespace k2 {

namespace {

// The factorisation of a line is a chain of one division, product and difference per element
// (kept in DPTTRF's order, so the factors are the reference's bit for bit), which bounds the
// kernel: about 60 ns per element whatever the number of lines.  One wavefront of the workgroup
// runs the chains of kLines lines, a lane each, out of LDS; the other three move the tiles, with
// unit stride in memory for either direction: the next one in, the previous one out (kBufs = 3; a line
// of one tile needs one buffer).  A lane that walked its line in memory paid a round trip per element:
// 320 us (x) and 245 us (y) on average over the nine levels of 1500 x 1100.
//
// per: the line direction is periodic, so its wrap couplings are added to the end diagonals
// (src/2d/ftn/BMG2_SymStd_SETUP_lines_x.f90:75-82, _y.f90:77-84) before the factorisation
template <int DIR, int kLines, int kTile, int kBufs>
__global__ __launch_bounds__(256) void setup_lines_k(const double *__restrict__ so,
                                                     double *__restrict__ sor, int ii, int jj,
                                                     int ns, int *__restrict__ info, int per) {
    __shared__ double D[kBufs][kLines][kTile + 1], E[kBufs][kLines][kTile + 1];
    const std::size_t P = (std::size_t)ii * jj;
    so += (std::size_t)blockIdx.y * ns * P;
    sor += (std::size_t)blockIdx.y * 2 * P;
    const int n = DIR == 0 ? ii - 2 : jj - 2, nl = DIR == 0 ? jj - 2 : ii - 2;
    const int l0 = blockIdx.x * kLines + 1, ng = min(kLines, nl - l0 + 1);
    const double *off = so + P * (DIR == 0 ? KW : KS);
    // point of element k of line g of the workgroup, in the operator and in the factors
    auto at = [&](int g, int k) {
        return DIR == 0 ? (std::size_t)(l0 + g) * ii + k + 1 : (std::size_t)(k + 1) * ii + l0 + g;
    };
    auto fac = [&](int g, int k) { return (std::size_t)(l0 + g) * (DIR == 0 ? ii : jj) + k + 1; };
    auto load = [&](int t, int tid, int nt) {
        const int buf = t % kBufs, k0 = t * kTile;
        for (int e = tid; e < kLines * kTile; e += nt) {
            const int g = DIR == 0 ? e / kTile : e % kLines, r = DIR == 0 ? e % kTile : e / kLines;
            const int k = k0 + r;
            if (g >= ng || k >= n) continue;
            double d = so[at(g, k)];
            if (per && k == 0) d = d + off[at(g, 0)];
            if (per && k == n - 1) d = d + off[at(g, n)];
            D[buf][g][r] = d;
            E[buf][g][r] = -off[at(g, k)];
        }
    };
    auto store = [&](int t, int tid, int nt) {
        const int buf = t % kBufs, k0 = t * kTile;
        for (int e = tid; e < kLines * kTile; e += nt) {
            const int g = e / kTile, r = e % kTile;
            if (g >= ng || k0 + r >= n) continue;
            sor[fac(g, k0 + r)] = D[buf][g][r];
            sor[P + fac(g, k0 + r)] = E[buf][g][r];
        }
    };
    const int tid = threadIdx.x, tiles = (n + kTile - 1) / kTile;
    double prev = 0.0;  // the line's last pivot
    int failed = 0;     // 1-based pivot that was not positive: the rest stays as assembled
    load(0, tid, 256);
    __syncthreads();
    for (int t = 0; t < tiles; ++t) {
        if (tid < 64) {
            if (tid < ng) {
                double *d = D[t % kBufs][tid], *e = E[t % kBufs][tid];
                const int m = min(kTile, n - t * kTile);
                for (int r0 = 0; r0 < m; r0 += 8) {
                    double c[8], w[8];
#pragma unroll
                    for (int u = 0; u < 8; ++u) {  // operands ahead of the chain
                        c[u] = d[min(r0 + u, m - 1)];
                        w[u] = e[min(r0 + u, m - 1)];
                    }
#pragma unroll
                    for (int u = 0; u < 8; ++u) {  // by selects: a branch costs more than it saves
                        const int k = t * kTile + r0 + u;
                        const bool live = r0 + u < m && failed == 0;
                        const double l = w[u] / prev;
                        const double v = k > 0 ? c[u] - l * w[u] : c[u];
                        e[r0 + u] = live && k > 0 ? l : w[u];
                        d[r0 + u] = live ? v : c[u];
                        prev = live ? v : prev;
                        failed = live && !(v > 0.0) ? k + 1 : failed;
                    }
                }
            }
        } else {
            if (t > 0) store(t - 1, tid - 64, 192);
            if (t + 1 < tiles) load(t + 1, tid - 64, 192);
        }
        __syncthreads();
    }
    if (failed) atomicMax(info, failed);
    store(tiles - 1, tid, 256);
}

void setup_lines(int dir, const double *so, int nstncl, double *sor, int ii, int jj, int *info,
                 hipStream_t s, int nb, int per) {
    const int nl = dir == 0 ? jj - 2 : ii - 2;
    const int n = dir == 0 ? ii - 2 : jj - 2;
    // Three buffers of 16 lines by 64 take 50 KB, three workgroups a CU: too few where many lines are
    // short.  Lines of one tile come without the other buffers, and those of at most 8 points 64 to a
    // workgroup: 200000 x-lines of 4 points 81 -> 32 us (54 by a lane per line walking memory), 65536
    // of 64 points 85 -> 60.
    auto launch = [&](auto kernel, int lines) {
        const dim3 g((unsigned)((nl + lines - 1) / lines), (unsigned)nb);
        kernel<<<g, 256, 0, s>>>(so, sor, ii, jj, nstncl, info, per);
    };
    if (n <= 8)
        dir == 0 ? launch(setup_lines_k<0, 64, 8, 1>, 64) : launch(setup_lines_k<1, 64, 8, 1>, 64);
    else if (n <= 64)
        dir == 0 ? launch(setup_lines_k<0, 16, 64, 1>, 16) : launch(setup_lines_k<1, 16, 64, 1>, 16);
    else
        dir == 0 ? launch(setup_lines_k<0, 16, 64, 3>, 16) : launch(setup_lines_k<1, 16, 64, 3>, 16);
}

}  // namespace

void setup_lines_x(const double *so, int nstncl, double *sor, int ii, int jj, int *info,
                   hipStream_t s, int nb) {
    setup_lines(0, so, nstncl, sor, ii, jj, info, s, nb, 0);
}

void setup_lines_y(const double *so, int nstncl, double *sor, int ii, int jj, int *info,
                   hipStream_t s, int nb) {
    setup_lines(1, so, nstncl, sor, ii, jj, info, s, nb, 0);
}

void setup_lines_per(int dir, const double *so, int nstncl, double *sor, int ii, int jj, int jpn,
                     int *info, hipStream_t s, int nb) {
    const bool px = jpn == 2 || jpn == 3 || jpn == -2 || jpn == -3;
    const bool py = jpn == 1 || jpn == 3 || jpn == -1 || jpn == -3;
    setup_lines(dir, so, nstncl, sor, ii, jj, info, s, nb, (dir == 0 ? px : py) ? 1 : 0);
}

}  // namespace k2
}  // namespace cdr
