// The coarse levels of a 2D V-cycle in one launch.
#include "../../include/cedar_hip.h"
#include "bmg2_device.hpp"
#include "bmg2_launch.hpp"
#include "tile_order.hpp"

#include <hip/hip_runtime.h>

#include <cstdint>
#include <type_traits>

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
// step.  The arrays sit in LDS as far as they fit, addressed as LDS (what lies where is a template
// parameter and no pointer may be either, or every access becomes a flat one that waits for memory
// and LDS alike); a step's threads are dealt to exactly the points it updates, by shifts; the
// operands of a smoothing are loaded once and held in registers where they fit, y-lines of a
// first level in memory from a transposed copy so that they arrive with unit stride; a wavefront
// without points in a step goes straight to its barrier (four wavefronts share a SIMD, and what
// the idle ones executed on the way was most of a small level's step); the arrays come in as
// chunks dealt over the wavefronts, all of a chunk's loads in flight.  V(2,1) point relaxation
// in FP64 from 32^2 down: 62 us with flat accesses, 38 addressed as LDS, 33 as it is; from 64^2
// down 127, 80, 69; xy-lines in FP32 from 64^2 down 83 -> 71; 12 problems, lines from 66^2 down,
// 152 -> 120.

// Operands of one element of a line (everything but the iterate): right-hand side, couplings to
// the neighbouring lines, multipliers of the forward and backward pass, pivot.
template <typename T>
struct line_ops {
    T qf, s0, s1, sw0, nw0, nw1, sw1, ef, eb, d;
};

// Where the operands of the lines of one direction lie: element k of line L at L * line + (k + 1) *
// elem of the operator planes and of b, at L * flen + k of D and E.
template <typename T>
struct line_src {
    const T *sc, *sw, *nw, *b, *D, *E;
    int elem, line, flen, nw0, nw1;
};

// dir 0: rows, 1: columns.  so holds the grid itself, or with transposed (dir 1) the operator of the
// transposed grid, b transposed likewise.  The factors of a line are contiguous either way.
template <typename T>
__device__ inline line_src<T> line_source(const T *so, const T *b, const T *sor, int ii, int jj,
                                          int dir, bool transposed) {
    line_src<T> r;
    const int P = ii * jj;
    r.elem = dir == 0 || transposed ? 1 : ii;
    r.line = dir == 0 ? ii : transposed ? jj : 1;
    r.flen = dir == 0 ? ii : jj;
    r.sc = so + P * (dir == 0 || transposed ? KS : KW);
    r.sw = so + P * KSW;
    r.nw = so + P * KNW;
    r.b = b;
    r.D = sor + 1;
    r.E = sor + P + 2;
    r.nw0 = dir == 0 ? r.elem : r.line;
    r.nw1 = dir == 0 ? r.line : r.elem;
    return r;
}

// operands of element k of line L of n elements, and the backward multiplier of element kb
template <typename T>
__device__ inline void load_ops(line_ops<T> &o, const line_src<T> &r, int L, int k, int kb, int n) {
    const int kc = min(k, n - 1), p = L * r.line + (kc + 1) * r.elem, f = L * r.flen;
    o.qf = r.b[p];
    o.s0 = r.sc[p];
    o.s1 = r.sc[p + r.line];
    o.sw0 = r.sw[p];
    o.nw0 = r.nw[p + r.nw0];
    o.nw1 = r.nw[p + r.nw1];
    o.sw1 = r.sw[p + r.elem + r.line];
    o.ef = r.E[f + max(kc - 1, 0)];
    o.d = r.D[f + kc];
    o.eb = r.E[f + min(kb, max(n - 2, 0))];
}

// Lines of one colour, in place, by one wavefront: 64 / w lines of at most w = 64, 32 or 16 points
// side by side (w = 1 << ws; one line of at most 64*CH points where CH > 1), lane k of a line
// owning its element k.  The scans stop where the lines do: the steps left out of scan_affine_dpp
// would combine with the identity only, so a line's result does not depend on w.  act: the
// lane's line exists; L: its index.
template <typename T, int CH>
__device__ inline void solve_lines(const line_ops<T> (&o)[CH], T *q, int ii, int jj, int dir, int L,
                                   bool act, int ws) {
    const int w = 1 << ws, lane = threadIdx.x % WAVE, e = lane & (w - 1), sub = lane - e;
    const int n = dir == 0 ? ii - 2 : jj - 2;
    const int step = dir == 0 ? 1 : ii, cross = dir == 0 ? ii : 1;
    const int base = L * cross + step;  // element 0
    T a[CH], b[CH];
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const int k = u * WAVE + e, p = base + min(k, n - 1) * step;
        line_raw<T> r{o[u].qf, o[u].s0, q[p - cross],  o[u].s1, q[p + cross],  o[u].sw0, q[p - ii - 1],
                      o[u].nw0, q[p - ii + 1], o[u].nw1, q[p + ii - 1], o[u].sw1, q[p + ii + 1]};
        b[u] = line_rhs<T, true>(r);
        a[u] = (k > 0) ? -o[u].ef : T(0);
    }
#pragma unroll
    for (int u = 0; u < CH; ++u) scan_affine_rows(a[u], b[u], w);
    T carry = T(0);
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const T y = affine(a[u], carry, b[u]);
        if (CH > 1) carry = last_lane(y);
        b[u] = div_pivot(y, o[u].d);
    }
    const int r = w - 1 - e;  // the backward pass runs from a line's last element
#pragma unroll
    for (int u = 0; u < CH; ++u) {
        const int k = u * WAVE + r;
        const T c = __shfl(b[u], sub + r, WAVE);
        a[u] = (k < n - 1) ? -o[u].eb : T(0);
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

// operands of one point of a Gauss-Seidel colour
template <typename T>
struct point_ops {
    T b, w0, w1, s0, s1, sw0, nw0, nw1, sw1, rec;
};
template <typename T>
__device__ inline void load_point(point_ops<T> &o, const T *so, const T *b, const T *sor, int P,
                                  int p, int ii) {
    o.b = b[p];
    o.w0 = so[P * KW + p];
    o.w1 = so[P * KW + p + 1];
    o.s0 = so[P * KS + p];
    o.s1 = so[P * KS + p + ii];
    o.sw0 = so[P * KSW + p];
    o.nw0 = so[P * KNW + p + 1];
    o.nw1 = so[P * KNW + p + ii];
    o.sw1 = so[P * KSW + p + ii + 1];
    o.rec = sor[P + p];
}
// the new value of point p, in the order of apply_offdiag
template <typename T>
__device__ inline T relax_point(const point_ops<T> &o, const T *q, int p, int ii) {
    T v = o.b + o.w0 * q[p - 1];
    v = v + o.w1 * q[p + 1];
    v = v + o.s0 * q[p - ii];
    v = v + o.s1 * q[p + ii];
    v = v + o.sw0 * q[p - ii - 1];
    v = v + o.nw0 * q[p - ii + 1];
    v = v + o.nw1 * q[p + ii - 1];
    v = v + o.sw1 * q[p + ii + 1];
    return v * o.rec;
}

// planes of the relaxation data a level keeps on chip: 1 / c, the factors of one direction, or
// those of both
__host__ __device__ inline int relax_planes(int relax) {
    return relax == CDR_RELAX_POINT ? 1 : relax == CDR_RELAX_LINE_XY ? 4 : 2;
}

// LDS bytes of one level: the operator, the relaxation data, x, b, res and, where ci, the
// interpolation stored on it; each array rounded up to 16 bytes.  first_mode (the first level of
// lds_mode 2 or 3): x, b and res (2) or x alone (3).
template <typename T>
__host__ __device__ inline std::size_t fused_level_bytes(int ii, int jj, bool ci, int first_mode,
                                                        int relax) {
    const std::size_t plane = ((std::size_t)ii * jj * sizeof(T) + 15) / 16 * 16;
    if (first_mode == 2) return 3 * plane;
    if (first_mode == 3) return plane;
    return plane * (5 + relax_planes(relax) + 3 + (ci ? 8 : 0));
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
// memory.  MODE 0: everything in memory.  CI: the interpolation weights are on chip too (each is
// used once going down and once going up).
template <typename T, int CH, int MODE, bool CI>
__global__ __launch_bounds__(1024) void coarse_cycle_k(const coarse_level<T> *__restrict__ lv,
                                                       int nlev, int relax, int npre, int npost,
                                                       const double *__restrict__ abd,
                                                       double *__restrict__ bbd, int rep) {
    constexpr int NT = 1024, NWAVE = NT / WAVE;
    constexpr int M0 = MODE >= 2 ? MODE : 1;  // fused_level_bytes mode of the first level
    extern __shared__ __align__(16) unsigned char lds[];
    __shared__ double cg_sh[CG_LDS];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
    const std::size_t bz = blockIdx.x, bo = operator_of(bz, rep);
    const int nsor = relax_planes(relax);
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
        return (unsigned)fused_level_bytes<T>(lv[l].ii, lv[l].jj, CI && l > 0, l == 0 ? M0 : 1, relax);
    };
    auto on_chip = [&](int l, unsigned off) {
        coarse_level<T> d;
        d.ii = lv[l].ii;
        d.jj = lv[l].jj;
        const int P = d.ii * d.jj;
        const unsigned plane = ((unsigned)P * sizeof(T) + 15) / 16 * 16;
        T *base = reinterpret_cast<T *>(lds + off);
        const unsigned pl = plane / sizeof(T);
        d.x = base;
        d.b = base + pl;
        d.res = base + 2 * pl;
        d.so = base + 3 * pl;
        T *sor = base + 8 * pl;
        d.sor0 = relax == CDR_RELAX_POINT ? sor - P : sor;  // point: the reciprocals are plane 1
        d.sor1 = sor + 2 * pl;
        if constexpr (CI)
            d.ci = base + (8 + nsor) * pl;
        else
            d.ci = global_ptr(lv[l].ci) + bo * 8 * (std::size_t)P;
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
        const unsigned pl = (((unsigned)(d.ii * d.jj) * sizeof(T) + 15) / 16 * 16) / sizeof(T);
        d.x = reinterpret_cast<T *>(lds);
        if constexpr (MODE == 2) {
            d.b = d.x + pl;
            d.res = d.x + 2 * pl;
        }
        return d;
    };
    // MODE 2 and 3: the first level's operator and (3) b for its y-lines, transposed; b is
    // transposed here, into the scratch the caller gives, as it is new in every cycle
    const T *soT = nullptr;
    T *bT = nullptr;
    {
        const int n = (lv[nlev - 1].ii - 2) * (lv[nlev - 1].jj - 2);
        coarse_band_stage(abd + bo * (std::size_t)lv[nlev - 1].ii * n, lv[nlev - 1].ii,
                          lv[nlev - 1].jj, tid, NT, cg_sh);
    }
    if constexpr (MODE != 0) {
        constexpr int U = 16;  // elements of a chunk per lane
        int job = 0;           // chunks dealt so far
        auto copy_in = [&](const T *src, T *dst, int n) {
            const int lane = tid % WAVE, chunks = (n + WAVE * U - 1) / (WAVE * U);
            for (int c = (wave - job) & (NWAVE - 1); c < chunks; c += NWAVE) {
                T v[U];
                const int k0 = c * WAVE * U + lane;
#pragma unroll
                for (int u = 0; u < U; ++u) v[u] = src[min(k0 + u * WAVE, n - 1)];
                __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                for (int u = 0; u < U; ++u)
                    if (k0 + u * WAVE < n) dst[k0 + u * WAVE] = v[u];
            }
            job += chunks;
        };
        unsigned off = 0;
        for (int l = 0; l < nlev; ++l) {
            const coarse_level<T> g = in_memory(l);
            const int P = g.ii * g.jj;
            if (MODE >= 2 && l == 0) {
                const coarse_level<T> d = first_level();
                copy_in(g.x, d.x, P);
                if constexpr (MODE == 2) {
                    copy_in(g.b, d.b, P);
                    for (int k = tid; k < P; k += NT) d.res[k] = T(0);
                }
                if (lv[0].soT != nullptr &&
                    (relax == CDR_RELAX_LINE_Y || relax == CDR_RELAX_LINE_XY)) {
                    soT = global_ptr(lv[0].soT) + bo * 5 * (std::size_t)P;
                    bT = global_ptr(lv[0].bT) + bz * (std::size_t)P;
                    if constexpr (MODE == 3)
                        for (int k = tid; k < P; k += NT) bT[(k % g.ii) * g.jj + k / g.ii] = g.b[k];
                }
            } else {
                const coarse_level<T> d = on_chip(l, off);
                copy_in(g.so, const_cast<T *>(d.so), 5 * P);
                if (relax == CDR_RELAX_POINT)
                    copy_in(g.sor0 + P, const_cast<T *>(d.sor0) + P, P);
                else
                    copy_in(g.sor0, const_cast<T *>(d.sor0), 2 * P);
                if (nsor == 4) copy_in(g.sor1, const_cast<T *>(d.sor1), 2 * P);
                if (CI && l > 0) copy_in(g.ci, const_cast<T *>(d.ci), 8 * P);
                // res and, below the first level, b start at zero as in memory: their ghosts are
                // never written, and interp_add adds the ghost res of an even-sized level to the
                // ghost of x
                if (l == 0) {
                    copy_in(g.x, d.x, P);
                    copy_in(g.b, d.b, P);
                }
                for (int k = tid; k < P; k += NT) {
                    d.res[k] = T(0);
                    if (l > 0) d.b[k] = T(0);
                }
            }
            off += bytes_of(l);
        }
    }
    __syncthreads();
    // after a step that writes on chip alone: operands on their way from memory need not have arrived
    auto x_barrier = [] {
        if constexpr (MODE == 0)
            __syncthreads();
        else
            lds_barrier();
    };
    // Steps over the points (c, r), c < nc, r < nr: threads along a row of the smallest power of two
    // that holds it
    auto each = [&](int nc, int nr, auto &&f) {
        const int sh = min(log2_up(nc), 10);
        if ((wave * WAVE) >> sh >= nr) return;
        for (int r = tid >> sh; r < nr; r += NT >> sh)
            for (int c = tid & ((1 << sh) - 1); c < nc; c += 1 << sh) f(c, r);
    };
    // sweep t of a smoothing: colour of a point sweep; direction and first line of a line sweep
    // (line-xy: x then y going down, y then x going up; two colours each)
    const bool xy = relax == CDR_RELAX_LINE_XY;
    auto colour = [&](int t, int updown, int &pi, int &pj) {
        // DOWN: (i odd, j odd), (even, odd), (odd, even), (even, even); UP: reverse
        const int c = updown == 0 ? t & 3 : 3 - (t & 3);
        pi = c & 1;
        pj = c >> 1;
    };
    auto sweep = [&](int t, int updown, int &dir, int &first) {
        dir = xy ? ((t >> 1) ^ updown) & 1 : relax == CDR_RELAX_LINE_Y;
        first = (t & 1) == updown ? 2 : 1;
    };
    auto width = [](int n) { return n <= 16 ? 4 : n <= 32 ? 5 : 6; };  // log2 of lanes per line
    // the lane's line of wavefront wv, counted along the colour
    auto lane_line = [&](int wv, int ws) { return (wv << (6 - ws)) + ((tid % WAVE) >> ws); };
    auto smooth = [&](const coarse_level<T> &d, int updown) {
        const int nrep = updown == 0 ? npre : npost;
        const int nx = d.ii - 2, ny = d.jj - 2, P = d.ii * d.jj;
        if (relax == CDR_RELAX_POINT) {
            for (int t = 0; t < 4 * nrep; ++t) {
                int pi, pj;
                colour(t, updown, pi, pj);
                each((nx + 1 - pi) / 2, (ny + 1 - pj) / 2, [&](int ic, int jc) {
                    const int p = (2 * jc + 1 + pj) * d.ii + 2 * ic + 1 + pi;
                    point_ops<T> o;
                    load_point(o, d.so, d.b, d.sor0, P, p, d.ii);
                    d.x[p] = relax_point(o, d.x, p, d.ii);
                });
                x_barrier();
            }
            return;
        }
        for (int t = 0; t < nrep * (xy ? 4 : 2); t += 2) {  // the two colours of a direction
            int dir, first;
            sweep(t, updown, dir, first);
            const int nfix = dir == 0 ? ny : nx, n = dir == 0 ? nx : ny;
            const line_src<T> src =
                line_source<T>(d.so, d.b, xy && dir ? d.sor1 : d.sor0, d.ii, d.jj, dir, false);
            const int ws = width(n), e = tid & ((1 << ws) - 1);
            for (int c = 0; c < 2; ++c, first = 3 - first) {
                const int nlines = (nfix - first + 2) / 2;
                for (int wv = wave; wv << (6 - ws) < nlines; wv += NWAVE) {
                    const int m = lane_line(wv, ws);
                    const bool act = m < nlines;
                    const int L = first + 2 * (act ? m : nlines - 1);
                    if (CH > 1 && n > WAVE) {
                        line_ops<T> o[CH];
#pragma unroll
                        for (int u = 0; u < CH; ++u)
                            load_ops(o[u], src, L, u * WAVE + e, u * WAVE + WAVE - 1 - e, n);
                        solve_lines<T, CH>(o, d.x, d.ii, d.jj, dir, L, act, 6);
                    } else {
                        line_ops<T> o[1];
                        load_ops(o[0], src, L, e, (1 << ws) - 1 - e, n);
                        solve_lines<T, 1>(o, d.x, d.ii, d.jj, dir, L, act, ws);
                    }
                }
                x_barrier();
            }
        }
    };
    // smooth() of a level so small that a thread has at most one point of a colour (64 points a
    // side) or a wavefront one group of lines: the operands of all its sweeps are loaded before the
    // first one and stay in registers, so that a sweep waits for the iterate alone.
    auto smooth_points = [&](const coarse_level<T> &d, int updown) {
        const int nrep = updown == 0 ? npre : npost;
        const int nx = d.ii - 2, ny = d.jj - 2, P = d.ii * d.jj;
        point_ops<T> o[4];
        int p[4];
        bool on[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            int pi, pj;
            colour(t, updown, pi, pj);
            const int nc = (nx + 1 - pi) / 2, nr = (ny + 1 - pj) / 2, sh = log2_up(nc);
            const int ic = tid & ((1 << sh) - 1), jc = tid >> sh;
            p[t] = (2 * jc + 1 + pj) * d.ii + 2 * ic + 1 + pi;
            on[t] = ic < nc && jc < nr;
            if (!on[t]) p[t] = d.ii + 1;
        }
        const bool work = (wave * WAVE) >> log2_up((nx + 1) / 2) < (ny + 1) / 2;
        if (work)
#pragma unroll
            for (int t = 0; t < 4; ++t) load_point(o[t], d.so, d.b, d.sor0, P, p[t], d.ii);
        for (int r = 0; r < nrep; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (work) {
                    const T v = relax_point(o[t], d.x, p[t], d.ii);
                    if (on[t]) d.x[p[t]] = v;
                }
                x_barrier();
            }
    };
    auto smooth_lines = [&](const coarse_level<T> &d, int updown) {  // at most 32 points a side
        const int nrep = updown == 0 ? npre : npost;
        const int nx = d.ii - 2, ny = d.jj - 2;
        line_ops<T> o[4][1];
        int L[4];
        bool act[4], any[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            if (t >= 2 && !xy) continue;
            int dir, first;
            sweep(t, updown, dir, first);
            const int n = dir == 0 ? nx : ny, nlines = ((dir == 0 ? ny : nx) - first + 2) / 2;
            const int ws = width(n), e = tid & ((1 << ws) - 1), m = lane_line(wave, ws);
            any[t] = wave << (6 - ws) < nlines;
            if (!any[t]) continue;
            act[t] = m < nlines;
            L[t] = first + 2 * (act[t] ? m : nlines - 1);
            load_ops(o[t][0],
                     line_source<T>(d.so, d.b, xy && dir ? d.sor1 : d.sor0, d.ii, d.jj, dir, false),
                     L[t], e, (1 << ws) - 1 - e, n);
        }
        for (int r = 0; r < nrep; ++r)
#pragma unroll
            for (int t = 0; t < 4; ++t) {
                if (t >= 2 && !xy) continue;
                int dir, first;
                sweep(t, updown, dir, first);
                if (any[t])
                    solve_lines<T, 1>(o[t], d.x, d.ii, d.jj, dir, L[t], act[t],
                                      width(dir == 0 ? nx : ny));
                x_barrier();
            }
    };
    auto smooth_level = [&](const coarse_level<T> &d, int updown) {
        if constexpr (CH == 1 && MODE != 0) {
            if (relax == CDR_RELAX_POINT) return smooth_points(d, updown);
            if constexpr (sizeof(T) == 4)  // FP64 operands of four sweeps do not fit the registers
                if (max(d.ii, d.jj) - 2 <= 32) return smooth_lines(d, updown);
        }
        smooth(d, updown);
    };
    // the smoothing of a first level whose operator is in memory
    auto smooth_first = [&](const coarse_level<T> &d, int updown) {
        if constexpr (CH == 1) {
            if (relax == CDR_RELAX_POINT) return smooth_points(d, updown);
        }
        const int nrep = updown == 0 ? npre : npost;
        const int nx = d.ii - 2, ny = d.jj - 2;
        if (relax == CDR_RELAX_POINT) return smooth(d, updown);
        for (int t = 0; t < nrep * (xy ? 4 : 2); ++t) {
            int dir, first;
            sweep(t, updown, dir, first);
            const int n = dir == 0 ? nx : ny, nlines = ((dir == 0 ? ny : nx) - first + 2) / 2;
            const int ws = width(n), e = tid & ((1 << ws) - 1);
            const bool trans = dir == 1 && soT != nullptr;
            const T *sor = xy && dir ? d.sor1 : d.sor0;
            line_src<T> src = line_source<T>(trans ? soT : d.so, d.b, sor, d.ii, d.jj, dir, trans);
            if constexpr (MODE == 3)
                if (trans) src.b = bT;
            for (int wv = wave; wv << (6 - ws) < nlines; wv += NWAVE) {
                const int m = lane_line(wv, ws);
                const bool act = m < nlines;
                const int L = first + 2 * (act ? m : nlines - 1);
                line_ops<T> o[CH];
#pragma unroll
                for (int u = 0; u < CH; ++u) {
                    load_ops(o[u], src, L, u * WAVE + e, u * WAVE + (1 << ws) - 1 - e, n);
                    if constexpr (MODE == 2)
                        if (trans) o[u].qf = d.b[(min(u * WAVE + e, n - 1) + 1) * d.ii + L];
                }
                if (CH > 1 && n > WAVE)
                    solve_lines<T, CH>(o, d.x, d.ii, d.jj, dir, L, act, 6);
                else
                    solve_lines<T, 1>(reinterpret_cast<line_ops<T>(&)[1]>(o[0]), d.x, d.ii, d.jj, dir,
                                      L, act, ws);
            }
            x_barrier();
        }
    };
    // going down: residual and restriction to the next level's b, whose x becomes zero
    // (res of a MODE 3 first level is in memory)
    auto down = [&](const coarse_level<T> &F, const coarse_level<T> &C, bool first) {
        const int P = F.ii * F.jj, Pc = C.ii * C.jj;
        each(F.ii - 2, F.jj - 2, [&](int c, int r) {
            const int p = (r + 1) * F.ii + c + 1;
            const T co = F.so[p], x = F.x[p];
            const T v = apply_offdiag<T, true>(F.so, P, F.x, p, F.ii, F.b[p]);
            F.res[p] = v - co * x;
        });
        if (MODE == 3 && first)
            __syncthreads();
        else
            x_barrier();
        each(C.ii - 2, C.jj - 2, [&](int c, int r) {
            C.b[(r + 1) * C.ii + c + 1] = restrict_point<T>(C.ci, F.res, F.ii, C.ii, Pc, c + 1, r + 1);
        });
        for (int k = tid; k < Pc; k += NT) C.x[k] = T(0);
        x_barrier();
    };
    auto up = [&](const coarse_level<T> &F, const coarse_level<T> &C) {
        each(F.ii / 2, F.jj / 2, [&](int c, int r) {
            interp_block<T, false>(F.x, C.x, F.res, F.so, C.ci, C.ii, C.jj, F.ii, F.jj, c + 1, r + 1);
        });
        x_barrier();
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
            smooth_level(F, rise ? 1 : 0);
            if (!rise) {
                down(F, C, false);
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
            smooth_first(F, s);
            if (s == 0) {
                down(F, C, true);
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

std::size_t fused_cycle_lds_bytes(int wbytes, const int *ii, const int *jj, int nlev, int lds_mode,
                                  int relax) {
    std::size_t b = 0;
    const bool ci = !(lds_mode & kCiInMemory);
    for (int l = 0; l < nlev; ++l) {
        const int m = l == 0 ? lds_mode & ~kCiInMemory : 1;
        b += wbytes == 8 ? fused_level_bytes<double>(ii[l], jj[l], ci && l > 0, m, relax)
                         : fused_level_bytes<float>(ii[l], jj[l], ci && l > 0, m, relax);
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
    auto pick = [&](auto ch) {  // lines of at most ch chunks of 64 elements
        constexpr int CH = decltype(ch)::value;
        switch (mode) {
        case 0: return launch(coarse_cycle_k<T, CH, 0, false>);
        case 1: return launch(coarse_cycle_k<T, CH, 1, true>);
        case 2: return launch(coarse_cycle_k<T, CH, 2, true>);
        case 3: return launch(coarse_cycle_k<T, CH, 3, true>);
        case 1 | kCiInMemory: return launch(coarse_cycle_k<T, CH, 1, false>);
        case 2 | kCiInMemory: return launch(coarse_cycle_k<T, CH, 2, false>);
        default: return launch(coarse_cycle_k<T, CH, 3, false>);
        }
    };
    if (max_side <= 64)
        pick(std::integral_constant<int, 1>{});
    else
        pick(std::integral_constant<int, 2>{});
}

#define CDR_INST(T)                                                                               \
    template void coarse_cycle<T>(const coarse_level<T> *, int, int, int, int, int, const         \
        double *, double *, hipStream_t, int, int, std::size_t, int);
CDR_INST(double)
CDR_INST(float)
#undef CDR_INST

}  // namespace k2
}  // namespace cdr
