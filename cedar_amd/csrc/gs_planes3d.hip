// 7-point Gauss-Seidel, both colours of a sweep in one launch
// (src/3d/ftn/BMG3_SymStd_relax_GS.f90:127-181; colours and operation order as gs7_colour_k of
// bmg3_kernels.hip, built with -ffp-contract=off, so bitwise the same).
#include "bmg2_device.hpp"
#include "bmg3_launch.hpp"
#include "bmg3_stencil.hpp"
#include "row_pairs.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>

namespace cdr {
namespace k3 {

namespace {

constexpr int LANES = 64;  // pairs of a row per workgroup, the first and last a halo
constexpr int ROWS = 16;   // rows of a plane per workgroup, the first and last a halo

// One pair (2 t, 2 t + 1) of a row in one plane: what its two relaxations need besides the iterate.
template <typename T>
struct pair_ops {
    row_pair<T> w, s, sn, bn, rec, f;  // sn: s of the next row, bn: b of the next plane
    T we;                              // w east of the pair
    row_pair<T> qn;                    // iterate in the next plane
    T side, qs, qnr;                   // iterate beside the first colour's point, in the rows j -+ 1
};

// by value: a choice between two members of a struct would send it to memory
template <typename T>
__device__ inline T pick(int c, T a, T b) {
    return c ? a : b;
}

// The second colour's points neighbour only first-colour points, and those only old second-colour
// values.  So a workgroup marches through the planes k of its tile, relaxes the first colour in plane
// k + 1 on the tile and one row and pair around it, then the second colour in plane k, and writes both
// to another array (neighbouring tiles still read the old values).  A row is a wavefront, its lanes
// pairs of points; new first-colour values go to the neighbours through LDS, to the next planes in
// registers; the operands of plane k + 2 are on their way meanwhile.  Ghosts are read from g and
// never written.  Bound by HBM: a sweep reads the operator, its reciprocal diagonal, the right-hand
// side and the iterate once instead of once per colour, the halos (a quarter more) mostly from L2.
// 200^3 in FP64: 142 us against 2 x 109 (gs7_sweep_pays has the other sizes).
template <typename T>
__global__ __launch_bounds__(LANES *ROWS) void gs7_sweep_k(
    const T *__restrict__ so, const T *__restrict__ qf, const T *__restrict__ q,
    T *__restrict__ out, const T *__restrict__ g, const T *__restrict__ sor, int ii, int jj, int kk,
    int pts, int nchunk, int ntile, int tiles, int J, int K) {
    __shared__ T fresh[2][ROWS][LANES + 2];  // [plane parity][row][pair + 1]: first colour's values
    // consecutive tiles, which share their halos, on one XCD
    const int id = (int)(blockIdx.x % 8) * (int)(gridDim.x / 8) + (int)(blockIdx.x / 8);
    if (id >= tiles) return;
    const int lane = threadIdx.x % LANES, r = __builtin_amdgcn_readfirstlane(threadIdx.x / LANES);
    const int c = id % nchunk, j0 = 1 + (id / nchunk) % ntile * J, k0 = 1 + id / (nchunk * ntile) * K;
    const int k1 = min(k0 + K, kk - 1) - 1, tlast = (ii - 1) / 2;
    // lanes and rows past the grid repeat its last ones and store nothing
    const int t0 = c * (LANES - 2) + lane, t = min(t0, tlast), j = min(j0 + r - 1, jj - 1);
    const bool own = t0 <= tlast && (lane > 0 || c == 0) && (lane < LANES - 1 || c == nchunk - 1) &&
                     r >= 1 && r <= J && j0 + r - 1 <= jj - 2;
    const bool has2 = 2 * t + 1 <= ii - 1;
    const bool in_a = t > 0 && 2 * t <= ii - 2, in_b = 2 * t + 1 <= ii - 2;  // not ghosts of the row
    const bool row_in = j >= 1 && j <= jj - 2;
    const std::size_t A = (std::size_t)ii * jj, P = A * kk;
    const int row = j * ii, rs = max(j - 1, 0) * ii, rn = min(j + 1, jj - 1) * ii;
    const int ia = 2 * t, ie = min(ia + 2, ii - 1), iw = max(ia - 1, 0);
    const int ig = t == 0 ? 0 : ii - 1;  // the row's ghost in this pair, if it has one
    const bool has_g = t == 0 || ia == ii - 1 || ia + 1 == ii - 1;
    // rows start at a scalar address, a lane's place in them is a 32-bit offset
    const unsigned oa = (unsigned)(ia - (has2 ? 0 : 1)) * (unsigned)sizeof(T);
    auto lane_ptr = [](const T *row_start, unsigned bytes) {
        return reinterpret_cast<const T *>(reinterpret_cast<const char *>(row_start) + bytes);
    };
    auto pair = [=](const T *row_start) {  // the pair; past the row's end its first element twice
        row_pair<T> v = load2(lane_ptr(row_start, oa));
        if (!has2) v.a = v.b;
        return v;
    };
    auto old = [=](int z) {  // the pair's iterate in plane z
        const bool gz = !row_in || z == 0 || z == kk - 1;
        const T *src = pick(gz, g, q) + (z * A + row);
        row_pair<T> v = pair(src);
        const T e = pick(has_g, g + (z * A + row), src)[pick(has_g, ig, ia)];
        if (has_g && ig == ia) v.a = e;
        if (has_g && ig == ia + 1) v.b = e;
        return v;
    };
    // element 0 or 1 of a pair that the first colour takes in plane z
    auto parity = [=](int z) { return (j + z + pts + 1) & 1; };
    auto load = [=](pair_ops<T> &o, int z) {
        const int rho = parity(z), zn = min(z + 1, kk - 1);
        const std::size_t p = z * A + row, pn = z * A + rn, ps = z * A + rs;
        const bool gz = !row_in || z == 0 || z == kk - 1;
        const unsigned or_ = (unsigned)min(ia + rho, ii - 1) * (unsigned)sizeof(T);
        const int is = pick(rho, ie, iw);
        o.w = pair(so + (kpw - 1) * P + p);
        o.we = *lane_ptr(so + (kpw - 1) * P + p, (unsigned)ie * (unsigned)sizeof(T));
        o.s = pair(so + (kps - 1) * P + p);
        o.sn = pair(so + (kps - 1) * P + pn);
        o.bn = pair(so + (kb - 1) * P + (zn * A + row));
        o.rec = pair(sor + P + p);
        o.f = pair(qf + p);
        o.qn = old(zn);
        o.side = pick(gz || is == 0 || is == ii - 1, g, q)[p + is];
        o.qs = *lane_ptr(pick(gz || j <= 1, g, q) + ps, or_);
        o.qnr = *lane_ptr(pick(gz || j >= jj - 2, g, q) + pn, or_);
    };
    const int za = k0 - 1, zb = k1 + 1;
    row_pair<T> qm = old(max(za - 1, 0)), qz = old(za);
    row_pair<T> b = pair(so + (kb - 1) * P + (za * A + row));
    pair_ops<T> cur, nxt;
    load(cur, za);
    // of the plane before: the second colour's point, its operands
    T fp = T(0), recp = T(0), w0 = T(0), w1 = T(0), s0 = T(0), s1 = T(0), b0 = T(0), b1 = T(0);
    T first1 = T(0), first2 = T(0);  // the pair's first-colour values one and two planes before
    for (int z = za; z <= zb; ++z) {
        load(nxt, min(z + 1, zb));
        k2::loads_issued();
        const int rho = parity(z);
        auto sel = [rho](row_pair<T> v) { return pick(rho, v.b, v.a); };
        // the first colour in plane z
        T first = sel(qz);
        {
            T v = sel(cur.f);
            v = v + sel(cur.w) * pick(rho, qz.a, cur.side);
            v = v + sel(cur.sn) * cur.qnr;
            v = v + pick(rho, cur.we, cur.w.b) * pick(rho, cur.side, qz.b);
            v = v + sel(cur.s) * cur.qs;
            v = v + sel(b) * sel(qm);
            v = v + sel(cur.bn) * sel(cur.qn);
            v = v * sel(cur.rec);
            if (row_in && z >= 1 && z <= kk - 2 && pick(rho, (int)in_b, (int)in_a)) first = v;
        }
        fresh[z & 1][r][lane + 1] = first;
        // the second colour in plane z - 1, at the same element of the pair
        if (z - 1 >= k0) {
            const T(*pl)[LANES + 2] = fresh[(z - 1) & 1];
            const int rd = max(r - 1, 0), ru = min(r + 1, ROWS - 1);
            const T x = pl[r][rho ? lane + 2 : lane];
            T v = fp;
            v = v + w0 * pick(rho, first1, x);
            v = v + s1 * pl[ru][lane + 1];
            v = v + w1 * pick(rho, x, first1);
            v = v + s0 * pl[rd][lane + 1];
            v = v + b0 * first2;
            v = v + b1 * first;
            v = v * recp;
            T *dst = out + (z - 1) * A + row + ia;
            const T va = pick(rho, first1, v), vb = pick(rho, v, first1);
            if (own) {
                if (in_a && in_b)
                    store2(dst, va, vb);
                else if (in_a)
                    dst[0] = va;
                else if (in_b)
                    dst[1] = vb;
            }
        }
        k2::lds_barrier();
        // the second colour's element of plane z is the other one
        fp = pick(rho, cur.f.a, cur.f.b);
        recp = pick(rho, cur.rec.a, cur.rec.b);
        w0 = pick(rho, cur.w.a, cur.w.b);
        w1 = pick(rho, cur.w.b, cur.we);
        s0 = pick(rho, cur.s.a, cur.s.b);
        s1 = pick(rho, cur.sn.a, cur.sn.b);
        b0 = pick(rho, b.a, b.b);
        b1 = pick(rho, cur.bn.a, cur.bn.b);
        first2 = first1;
        first1 = first;
        qm = qz;
        qz = cur.qn;
        b = cur.bn;
        cur = nxt;
    }
}

struct sweep_shape {
    int nchunk, ntile, J, K;
    long tiles, steps;  // steps: planes that a CU marches through
};

// Slabs of planes such that the workgroups, one per CU, fill the chip's 256 a whole number of times
// as far as the two extra planes of a slab (and the latency of its start) allow.  rows, planes: J and K
// as given, where positive.
sweep_shape shape_of(int ii, int jj, int kk, int rows = 0, int planes = 0) {
    sweep_shape r{};
    r.nchunk = std::max(1, ((ii - 1) / 2 - 2) / (LANES - 2) + 1);
    r.ntile = (jj - 2 + ROWS - 3) / (ROWS - 2);
    r.J = (jj - 2 + r.ntile - 1) / r.ntile;
    if (rows > 0) {
        r.J = rows;
        r.ntile = (jj - 2 + rows - 1) / rows;
    }
    const long columns = (long)r.nchunk * r.ntile;
    for (int n = 1; n <= std::min(kk - 2, 64); ++n) {
        const int k = planes > 0 ? planes : (kk - 2 + n - 1) / n;
        const long tiles = columns * ((kk - 2 + k - 1) / k), steps = (tiles + 255) / 256 * (k + 4);
        if (n == 1 || steps < r.steps) r.steps = steps, r.K = k, r.tiles = tiles;
    }
    return r;
}
constexpr long kMaxTiles = 1L << 30;

}  // namespace

// The march takes 4.9 us per plane and CU in FP64 (200^3: 142 us) and less where its arrays stay in the
// last cache (120^3: 30 us for 9 planes), two launches of one colour 23 to 30 ps per point (200^3: 216
// us); FP32 about 0.6 of either.  Over 132 sizes of up to 25 million points, most of them about the
// line, what is taken is 0.99 to 2.4 times as fast, 1.6 in the middle.  Rows that leave most of a
// wavefront idle (128^3: 65 pairs on two) and small levels stay with the two launches; so do planes
// whose workgroups are a multiple of 8 up to 1.6 million points: each XCD then finds its rows of the
// plane before in its own cache, and the two launches take 17 ps per point (125 x 96 x 104: 22 us, the
// march 26; 122 x 157 x 77: 26 and 28).
bool gs7_sweep_pays(int ii, int jj, int kk) {
    const sweep_shape f = shape_of(ii, jj, kk);
    const double points = (double)ii * jj * kk;
    const int plane_groups = ((ii - 1) / 2 + 63) / 64 * ((jj - 2 + 3) / 4);  // of relax_gs
    if (plane_groups % 8 == 0 && points <= 1.6e6) return false;
    return (double)f.steps * 4.9 < points * 26e-6 && f.tiles < kMaxTiles;
}

bool gs7_shape_ok(int ii, int jj, int kk, int rows, int planes) {
    return rows >= 0 && rows <= ROWS - 2 && planes >= 0 && planes <= kk - 2 &&
           shape_of(ii, jj, kk, rows, planes).tiles < kMaxTiles;
}

template <typename T>
void relax_gs7_sweep(const T *so, const T *qf, const T *q, T *out, const T *g, const T *sor, int ii,
                     int jj, int kk, int updown, hipStream_t s, int rows, int planes) {
    const sweep_shape f = shape_of(ii, jj, kk, rows, planes);
    gs7_sweep_k<T><<<(unsigned)((f.tiles + 7) / 8 * 8), LANES * ROWS, 0, s>>>(
        so, qf, q, out, g, sor, ii, jj, kk, updown == 0 ? 1 : 0, f.nchunk, f.ntile, (int)f.tiles, f.J,
        f.K);
}

template void relax_gs7_sweep<double>(const double *, const double *, const double *, double *,
                                      const double *, const double *, int, int, int, int,
                                      hipStream_t, int, int);
template void relax_gs7_sweep<float>(const float *, const float *, const float *, float *,
                                     const float *, const float *, int, int, int, int, hipStream_t,
                                     int, int);

}  // namespace k3
}  // namespace cdr
