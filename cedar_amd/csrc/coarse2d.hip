// The coarse levels of a 2D V-cycle in one launch.
#include "../../include/cedar_hip.h"
#include "bmg2_device.hpp"
#include "bmg2_launch.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>

namespace cdr {
namespace k2 {

namespace {

// ---- fused coarse-level V-cycle ---------------------------------------------------------------
// One workgroup per problem runs the whole V-cycle below a level of at most 64*CH points per side
// (smoothing, residual, restriction, coarsest band solve, interpolation) with workgroup barriers
// between the steps instead of one launch per step.  Every point is computed by the same device
// functions and in the same order as in the grid kernels, so the result is bitwise that of the
// unfused cycle.  Levels of a fused cycle are always 9-point (Galerkin operators).
//
// A chain of 60 to 150 short steps, each waiting for the one before: bound by the latency of a
// step.  The arrays sit in LDS as far as they fit, addressed as LDS (MODE is a template parameter
// and no pointer may be either, or every access becomes a flat one that waits for memory and LDS
// alike), and a step's threads are dealt to exactly the points it updates, by shifts.

// Lines of one colour, in place, by one wavefront: 64 / w lines of at most w = 64, 32 or 16 points
// side by side (one line of at most 64*CH points where CH > 1), lane k of a line owning its
// element k.  The scans stop where the lines do: the steps left out of scan_affine_dpp would
// combine with the identity only, so a line's result does not depend on w.  x-lines (dir 0) lie
// along rows, y-lines (dir 1) along columns; line = the wavefront's first of them.
template <typename T, int CH>
__device__ inline void wave_lines(const T *__restrict__ so, const T *__restrict__ qf, T *q,
                                  const T *__restrict__ sor, int ii, int jj, int dir, int first,
                                  int nlines, int line, int w) {
    const int lane = threadIdx.x % WAVE, e = lane & (w - 1), sub = lane & ~(w - 1);
    const int P = ii * jj, n = dir == 0 ? ii - 2 : jj - 2;
    const int mine = line + (int)((unsigned)sub / (unsigned)w);
    const bool act = mine < nlines;
    const int fixed = first + 2 * (act ? mine : nlines - 1);
    const int step = dir == 0 ? 1 : ii, cross = dir == 0 ? ii : 1;
    const int base = fixed * cross + step;  // element 0
    const T *D = sor + fixed * (dir == 0 ? ii : jj) + 1, *E = D + P + 1;
    const T *sc = so + P * (dir == 0 ? KS : KW), *sw = so + P * KSW, *nw = so + P * KNW;
    T a[CH], b[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const int k = u * WAVE + e, kc = min(k, n - 1), p = base + kc * step;
        line_raw<T> r;
        r.qf = qf[p];
        r.s0 = sc[p];
        r.q0 = q[p - cross];
        r.s1 = sc[p + cross];
        r.q1 = q[p + cross];
        r.sw0 = sw[p];
        r.q0m = q[p - ii - 1];
        r.nw0 = nw[p + 1];
        r.q0p = q[p - ii + 1];
        r.nw1 = nw[p + ii];
        r.q1m = q[p + ii - 1];
        r.sw1 = sw[p + ii + 1];
        r.q1p = q[p + ii + 1];
        const T m = E[max(kc - 1, 0)];
        b[u] = line_rhs<T, true>(r);
        a[u] = (k > 0) ? -m : T(0);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) scan_affine_rows(a[u], b[u], w);
    T carry = T(0);
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const T y = affine(a[u], carry, b[u]);
        if (CH > 1) carry = last_lane(y);
        b[u] = div_pivot(y, D[min(u * WAVE + e, n - 1)]);
    }
    const int r = w - 1 - e;  // the backward pass runs from a line's last element
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const int k = u * WAVE + r;
        const T c = __shfl(b[u], sub + r, WAVE);
        const T m = E[min(k, max(n - 2, 0))];
        a[u] = (k < n - 1) ? -m : T(0);
        a[u] = (k < n) ? a[u] : T(1);
        b[u] = (k < n) ? c : T(0);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) scan_affine_rows(a[u], b[u], w);
    carry = T(0);
#pragma unroll
    for (int u = CH - 1; u >= 0; --u) {
        b[u] = affine(a[u], carry, b[u]);
        if (CH > 1) carry = last_lane(b[u]);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const int k = u * WAVE + r;
        if (act && k < n) q[base + k * step] = b[u];
    }
}

// LDS bytes the fused cycle needs to hold the arrays of one level on chip (per level: the
// operator, both relaxation factors, x, b, res and, below the first level, the interpolation),
// each array rounded up to 16 bytes.  first_mode (the first level of lds_mode 2 or 3): x, b
// and res (2) or x alone (3).
template <typename T>
__host__ __device__ inline std::size_t fused_level_bytes(int ii, int jj, bool has_ci,
                                                        int first_mode = 1) {
    const std::size_t plane = ((std::size_t)ii * jj * sizeof(T) + 15) / 16 * 16;
    if (first_mode == 2) return 3 * plane;
    if (first_mode == 3) return plane;
    return plane * (5 + 2 + 2 + 3 + (has_ci ? 8 : 0));
}

// a pointer read from memory, known to point to memory (and not to LDS)
template <typename T>
__device__ inline T *global_ptr(T *p) {
    return (T *)(__attribute__((address_space(1))) T *)(std::uintptr_t)p;
}

// smallest power of two >= n, as a shift
__device__ inline int log2_up(int n) { return n <= 1 ? 0 : 32 - __clz(n - 1); }

// MODE 1: every array of every level lives in LDS for the whole cycle (the launcher checked that
// they fit); the first level's b comes in from memory and its x goes back at the end, the only
// values the caller exchanges with the fused levels.  For a first level too large to hold whole,
// MODE 2 keeps only its x, b and res in LDS and MODE 3 its x alone; its other arrays stay in
// memory, where the sweeps only read them, so that a sweep does not wait on memory for the
// previous sweep's writes.  MODE 0: everything in memory.
template <typename T, int CH, int MODE>
__global__ __launch_bounds__(1024) void coarse_cycle_k(const coarse_level<T> *__restrict__ lv,
                                                       int nlev, int relax, int npre, int npost,
                                                       const double *__restrict__ abd,
                                                       double *__restrict__ bbd, int rep) {
    constexpr int NT = 1024, NWAVE = NT / WAVE;
    constexpr int M0 = MODE >= 2 ? MODE : 1;  // fused_level_bytes mode of the first level
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ double cg_sh[CG_LDS];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const std::size_t bz = blockIdx.x, bo = bz / rep;
    auto in_memory = [&](int l) {  // the level's arrays of problem bz (operator bo)
        coarse_level<T> d = lv[l];
        const std::size_t P = (std::size_t)d.ii * d.jj;
        d.so = global_ptr(d.so) + bo * 5 * P;
        d.x = global_ptr(d.x) + bz * P;
        d.b = global_ptr(d.b) + bz * P;
        d.res = global_ptr(d.res) + bz * P;
        d.sor0 = global_ptr(d.sor0) + bo * 2 * P;
        d.sor1 = global_ptr(d.sor1) + bo * 2 * P;
        d.ci = global_ptr(d.ci) + bo * 8 * P;  // not there on level 0
        return d;
    };
    // offset of level l in LDS, given that of a neighbour (the levels lie one after another)
    auto bytes_of = [&](int l) {
        return (unsigned)fused_level_bytes<T>(lv[l].ii, lv[l].jj, l > 0, l == 0 ? M0 : 1);
    };
    auto on_chip = [&](int l, unsigned off) {
        coarse_level<T> d;
        d.ii = lv[l].ii;
        d.jj = lv[l].jj;
        const unsigned plane = ((unsigned)(d.ii * d.jj) * sizeof(T) + 15) / 16 * 16;
        unsigned char *base = lds + off;
        d.so = reinterpret_cast<T *>(base);
        d.sor0 = reinterpret_cast<T *>(base + 5 * plane);
        d.sor1 = reinterpret_cast<T *>(base + 7 * plane);
        d.x = reinterpret_cast<T *>(base + 9 * plane);
        d.b = reinterpret_cast<T *>(base + 10 * plane);
        d.res = reinterpret_cast<T *>(base + 11 * plane);
        d.ci = reinterpret_cast<T *>(base + 12 * plane);  // not there on level 0
        return d;
    };
    auto lower = [&](int l, unsigned off) {
        if constexpr (MODE == 0)
            return in_memory(l);
        else
            return on_chip(l, off);
    };
    auto first_level = [&] {  // MODE 2 and 3
        coarse_level<T> d = in_memory(0);
        const unsigned plane = ((unsigned)(d.ii * d.jj) * sizeof(T) + 15) / 16 * 16;
        d.x = reinterpret_cast<T *>(lds);
        if constexpr (MODE == 2) {
            d.b = reinterpret_cast<T *>(lds + plane);
            d.res = reinterpret_cast<T *>(lds + 2 * plane);
        }
        return d;
    };
    {
        const int n = (lv[nlev - 1].ii - 2) * (lv[nlev - 1].jj - 2);
        coarse_band_stage(abd + bo * (std::size_t)lv[nlev - 1].ii * n, lv[nlev - 1].ii,
                          lv[nlev - 1].jj, tid, NT, cg_sh);
    }
    if constexpr (MODE != 0) {
        unsigned off = 0;
        for (int l = 0; l < nlev; ++l) {
            const coarse_level<T> g = in_memory(l);
            const int P = g.ii * g.jj;
            if (MODE >= 2 && l == 0) {
                const coarse_level<T> d = first_level();
                for (int k = tid; k < P; k += NT) {
                    d.x[k] = g.x[k];
                    if constexpr (MODE == 2) {
                        d.b[k] = g.b[k];
                        d.res[k] = T(0);
                    }
                }
            } else {
                const coarse_level<T> d = on_chip(l, off);
                for (int k = tid; k < 5 * P; k += NT) const_cast<T *>(d.so)[k] = g.so[k];
                for (int k = tid; k < 2 * P; k += NT) {
                    const_cast<T *>(d.sor0)[k] = g.sor0[k];
                    const_cast<T *>(d.sor1)[k] = g.sor1[k];
                }
                if (l > 0)
                    for (int k = tid; k < 8 * P; k += NT) const_cast<T *>(d.ci)[k] = g.ci[k];
                // res and, below the first level, b start at zero as in memory: their ghosts are
                // never written, and interp_add adds the ghost res of an even-sized level to the
                // ghost of x
                for (int k = tid; k < P; k += NT) {
                    d.res[k] = T(0);
                    d.b[k] = l == 0 ? g.b[k] : T(0);
                    if (l == 0) d.x[k] = g.x[k];
                }
            }
            off += bytes_of(l);
        }
    }
    __syncthreads();
    // Steps over the points (i, j) = (i0 + di * c, j0 + dj * r), c < nc, r < nr: threads along a row
    // of the smallest power of two that holds it
    auto each = [&](int nc, int nr, auto &&f) {
        const int sh = min(log2_up(nc), 10);
        for (int r = tid >> sh; r < nr; r += NT >> sh)
            for (int c = tid & ((1 << sh) - 1); c < nc; c += 1 << sh) f(c, r);
    };
    auto smooth = [&](const coarse_level<T> &d, int updown) {
        const int nrep = updown == 0 ? npre : npost;
        const int nx = d.ii - 2, ny = d.jj - 2, P = d.ii * d.jj;
        if (relax == CDR_RELAX_POINT) {
            for (int t = 0; t < 4 * nrep; ++t) {
                // DOWN: (i odd, j odd), (even, odd), (odd, even), (even, even); UP: reverse
                const int c = updown == 0 ? t & 3 : 3 - (t & 3), pi = c & 1, pj = c >> 1;
                each((nx + 1 - pi) / 2, (ny + 1 - pj) / 2, [&](int ic, int jc) {
                    const int p = (2 * jc + 1 + pj) * d.ii + 2 * ic + 1 + pi;
                    const T v = apply_offdiag<T, true>(d.so, P, d.x, p, d.ii, d.b[p]);
                    d.x[p] = v * d.sor0[P + p];
                });
                __syncthreads();
            }
            return;
        }
        const bool xy = relax == CDR_RELAX_LINE_XY;
        for (int t = 0; t < nrep * (xy ? 4 : 2); ++t) {
            // line-xy: x then y going down, y then x going up; two colours each
            const int dir = xy ? ((t >> 1) ^ updown) & 1 : relax == CDR_RELAX_LINE_Y;
            const int first = (t & 1) == updown ? 2 : 1;
            const int nfix = dir == 0 ? ny : nx, n = dir == 0 ? nx : ny;
            if (first <= nfix) {
                const int nlines = (nfix - first) / 2 + 1;
                const int w = n <= 16 ? 16 : n <= 32 ? 32 : 64, per = WAVE / w;
                const T *sor = xy && dir ? d.sor1 : d.sor0;
                for (int line = wave * per; line < nlines; line += NWAVE * per) {
                    if (CH > 1 && n > WAVE)
                        wave_lines<T, CH>(d.so, d.b, d.x, sor, d.ii, d.jj, dir, first, nlines, line, WAVE);
                    else
                        wave_lines<T, 1>(d.so, d.b, d.x, sor, d.ii, d.jj, dir, first, nlines, line, w);
                }
            }
            __syncthreads();
        }
    };
    // going down: residual and restriction to the next level's b, whose x becomes zero
    auto down = [&](const coarse_level<T> &F, const coarse_level<T> &C) {
        const int P = F.ii * F.jj, Pc = C.ii * C.jj;
        each(F.ii - 2, F.jj - 2, [&](int c, int r) {
            const int p = (r + 1) * F.ii + c + 1;
            T v = apply_offdiag<T, true>(F.so, P, F.x, p, F.ii, F.b[p]);
            F.res[p] = v - F.so[p] * F.x[p];
        });
        __syncthreads();
        each(C.ii - 2, C.jj - 2, [&](int c, int r) {
            C.b[(r + 1) * C.ii + c + 1] = restrict_point<T>(C.ci, F.res, F.ii, C.ii, Pc, c + 1, r + 1);
        });
        for (int k = tid; k < Pc; k += NT) C.x[k] = T(0);
        __syncthreads();
    };
    auto up = [&](const coarse_level<T> &F, const coarse_level<T> &C) {
        each(F.ii / 2, F.jj / 2, [&](int c, int r) {
            interp_block<T>(F.x, C.x, F.res, F.so, C.ci, C.ii, C.jj, F.ii, F.jj, c + 1, r + 1);
        });
        __syncthreads();
    };
    // the levels l0 .. nlev - 1, all addressed alike, at off; one copy of each step for all of them
    auto cycle = [&](int l0, unsigned off) {
        const int nd = nlev - 1 - l0;  // levels above the coarsest
        int l = l0;
        for (int s = 0; s < 2 * nd || s == 0; ++s) {
            const bool rise = s >= nd;
            if (s == nd) {  // coarsest level: band Cholesky solve (as solve_cg_k)
                const coarse_level<T> C = lower(l, off);
                const int n = (C.ii - 2) * (C.jj - 2);
                coarse_band_solve<T>(C.x, C.b, abd + bo * (std::size_t)C.ii * n, bbd + bz * n, C.ii,
                                     C.jj, tid, NT, cg_sh, true);
                __syncthreads();
            }
            if (nd == 0) break;
            if (rise) {
                --l;
                off -= bytes_of(l);
            }
            const coarse_level<T> F = lower(l, off), C = lower(l + 1, off + bytes_of(l));
            if (rise) up(F, C);
            smooth(F, rise ? 1 : 0);
            if (!rise) {
                down(F, C);
                off += bytes_of(l);
                ++l;
            }
        }
    };
    if constexpr (MODE >= 2) {
        const coarse_level<T> F = first_level();
        const unsigned off = bytes_of(0);
        for (int s = 0; s < 2; ++s) {
            const coarse_level<T> C = on_chip(1, off);
            if (s == 1) up(F, C);
            smooth(F, s);
            if (s == 0) {
                down(F, C);
                cycle(1, off);
            }
        }
    } else {
        cycle(0, 0);
    }
    if constexpr (MODE != 0) {  // the smoothing ends with a workgroup barrier
        const coarse_level<T> g = in_memory(0);
        const T *x = MODE >= 2 ? first_level().x : on_chip(0, 0).x;
        for (int k = tid; k < g.ii * g.jj; k += NT) g.x[k] = x[k];
    }
}

}  // namespace

std::size_t fused_cycle_lds_bytes(int wbytes, const int *ii, const int *jj, int nlev,
                                  int lds_mode) {
    std::size_t b = 0;
    for (int l = 0; l < nlev; ++l) {
        const int m = l == 0 ? lds_mode : 1;
        b += wbytes == 8 ? fused_level_bytes<double>(ii[l], jj[l], l > 0, m)
                         : fused_level_bytes<float>(ii[l], jj[l], l > 0, m);
    }
    return b;
}

template <typename T>
void coarse_cycle(const coarse_level<T> *lv, int nlev, int max_side, int relax, int npre,
                  int npost, const double *abd, double *bbd, hipStream_t s, int nb, int rep,
                  std::size_t lds_bytes, int lds_mode) {
    const int mode = lds_bytes > 0 ? lds_mode : 0;
    auto launch = [&](auto kernel) {
        if (mode)
            (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes);
        kernel<<<nb, 1024, lds_bytes, s>>>(lv, nlev, relax, npre, npost, abd, bbd, rep);
    };
    const bool one = max_side <= 64;  // lines of one 64-element chunk
    switch (mode) {
    case 0: one ? launch(coarse_cycle_k<T, 1, 0>) : launch(coarse_cycle_k<T, 2, 0>); break;
    case 1: one ? launch(coarse_cycle_k<T, 1, 1>) : launch(coarse_cycle_k<T, 2, 1>); break;
    case 2: one ? launch(coarse_cycle_k<T, 1, 2>) : launch(coarse_cycle_k<T, 2, 2>); break;
    default: one ? launch(coarse_cycle_k<T, 1, 3>) : launch(coarse_cycle_k<T, 2, 3>); break;
    }
}

#define CDR_INST(T)                                                                               \
    template void coarse_cycle<T>(const coarse_level<T> *, int, int, int, int, int, const         \
        double *, double *, hipStream_t, int, int, std::size_t, int);
CDR_INST(double)
CDR_INST(float)
#undef CDR_INST

}  // namespace k2
}  // namespace cdr
