"""Kernels at the edges of their tiles, blocks and memory limits, against the oracle (bitwise: the
kernels keep its operation order)."""
import numpy as np
import pytest

from oracle import oracle as O
from oracle import oracle3 as O3
from tests.golden.gen3 import rand_so3
from tests.golden.make_golden_periodic import rand_periodic_so

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a, dtype=torch.float64):
    return torch.as_tensor(np.ascontiguousarray(a), dtype=dtype).cuda()


def host(t):
    return t.double().cpu().numpy()


# blocks of 8 points along a line with and without a remainder, groups of 4 lines with one to four
# in the last, odd and even seams; 5470 points do not fit LDS next to a wrap vector
@pytest.mark.parametrize("nx,ny", [(2, 2), (3, 2), (9, 4), (10, 9), (16, 7), (17, 8), (66, 3),
                                   (5470, 4), (4, 5470), (1500, 5), (5, 1500)])
@pytest.mark.parametrize("mask", [1, 2, 3])
@pytest.mark.parametrize("ns", [3, 5])
def test_periodic_lines(nx, ny, mask, ns):
    import cedar_amd as C
    print(f"\nperiodic lines {nx}x{ny} ns={ns} mask={mask}", flush=True)
    rng = np.random.default_rng(3 * nx + ny + mask + ns)
    jpn = O.bc_from_mask(mask)
    so = rand_periodic_so(rng, nx, ny, ns, mask)
    q = rng.standard_normal((ny + 2, nx + 2))
    qf = rng.standard_normal(q.shape)
    for d in ("x", "y"):
        sor, info = O.setup_lines_periodic(so, d, jpn)
        assert info == 0
        for ud in (O.DOWN, O.UP):
            g = C.relax_lines_periodic(dev(so), dev(qf), dev(q), dev(sor), ud, d, jpn)
            assert np.array_equal(host(g), O.relax_lines_periodic(so, qf, q, sor, ud, d, jpn)), (d, ud)


# short lines of which many share a workgroup: 64 up to 4 points, 16 up to 32, and up to 128 where there
# are four times as many; longer ones by themselves.  More of them than run at once otherwise (1024
# x-lines or 4096 y-lines of a colour), one less, and a last workgroup that is full or has one line; odd
# and even seams
@pytest.mark.parametrize("n,dr,nl", [(n, dr, nl) for n in (2, 3, 4, 5, 16, 31, 32, 33)
                                     for dr, nl in (("x", 2048), ("x", 2049), ("x", 2177), ("x", 2178),
                                                    ("y", 8192), ("y", 8194), ("y", 8321))] +
                         [(n, "x", nl) for n in (33, 128, 129) for nl in (8192, 8194, 8225)] +
                         [(n, "y", nl) for n in (33, 128, 129) for nl in (32768, 32770, 32801)])
@pytest.mark.parametrize("mask", [1, 2, 3])
def test_many_short_periodic_lines(n, dr, nl, mask):
    import cedar_amd as C
    nx, ny = (n, nl) if dr == "x" else (nl, n)
    ns = 3 + 2 * ((n + nl) % 2)
    print(f"\nshort periodic lines {dr} {nx}x{ny} ns={ns} mask={mask}", flush=True)
    rng = np.random.default_rng(3 * nx + ny + mask)
    jpn = O.bc_from_mask(mask)
    so = rand_periodic_so(rng, nx, ny, ns, mask)
    q = rng.standard_normal((ny + 2, nx + 2))
    qf = rng.standard_normal(q.shape)
    sor, info = O.setup_lines_periodic(so, dr, jpn)
    assert info == 0
    for ud in (O.DOWN, O.UP):
        g = C.relax_lines_periodic(dev(so), dev(qf), dev(q), dev(sor), ud, dr, jpn)
        assert np.array_equal(host(g), O.relax_lines_periodic(so, qf, q, sor, ud, dr, jpn)), ud


# A sweep of 2048 lines leaves the chip half empty; 32 times as many lines have 32 times the work and
# move 30 MB.  With a workgroup for each line they took 14 to 16 times as long, shared out 1.7 to 3.
@pytest.mark.parametrize("dr", ["x", "y"])
def test_short_periodic_lines_scale(dr):
    import cedar_amd as C
    jpn = C.bc_from_mask((dr == "x", dr == "y"))
    best = {}
    for nl in (2048, 65536):
        d = (8, nl) if dr == "x" else (nl, 8)
        so = torch.full((5, d[1] + 2, d[0] + 2), 0.5, dtype=torch.float64, device="cuda")
        so[0] = 9.0
        sor = torch.zeros((2,) + tuple(so.shape[1:]), dtype=torch.float64, device="cuda")
        C.setup_lines_periodic(so, sor, dr, jpn)
        f, q = torch.rand_like(so[0]), torch.rand_like(so[0])
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            C.relax_lines_periodic(so, f, q, sor, 0, dr, jpn)
            a.record()
            for _ in range(20):
                C.relax_lines_periodic(so, f, q, sor, 0, dr, jpn)
            b.record()
            b.synchronize()
            best[nl] = min(best.get(nl, 1e9), a.elapsed_time(b) / 20)
    print(f"\nshort periodic lines {dr}: {best}", flush=True)
    assert best[65536] < 6 * best[2048], best


# coarse rows of 64 points, one less and one more; the smallest grids; even extents, whose last
# fine points lie beyond the last coarse one; a level of more than 256 workgroups (one point's
# whole row per thread there, parts of it below)
@pytest.mark.parametrize("dims", [(3, 3, 3), (4, 3, 5), (125, 5, 4), (127, 6, 5), (128, 4, 9),
                                  (129, 9, 6), (131, 3, 3), (6, 129, 5), (6, 260, 66)])
@pytest.mark.parametrize("ns", [4, 14])
def test_galerkin3(dims, ns):
    import cedar_amd as C
    print(f"\ngalerkin {dims} ns={ns}", flush=True)
    so = rand_so3(np.random.default_rng(sum(dims) + ns), *dims, ns)
    ci = O3.setup_interp(so)
    soc = torch.full((14,) + ci.shape[1:], 7.0, dtype=torch.float64, device="cuda")
    C.cdr3.setup_galerkin(dev(so), dev(ci), soc)
    ref = O3.setup_galerkin(so, ci)
    inner = (slice(None),) + (slice(1, -1),) * 3
    assert np.array_equal(host(soc)[inner], ref[inner])
    assert (host(soc)[:, 0] == 7.0).all() and (host(soc)[:, :, :, -1] == 7.0).all()  # ghosts untouched


# a weight that is infinite or undefined enters exactly the sums that have a term with it: one such
# weight per case, in each of the 26 planes in turn; the parts of a row and, at the largest, whole rows
@pytest.mark.parametrize("dims", [(5, 4, 7), (6, 260, 66)])
@pytest.mark.parametrize("ns", [4, 14])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_galerkin3_keeps_undefined_weights_where_they_are(dims, ns, bad):
    import cedar_amd as C
    print(f"\ngalerkin, weight {bad} {dims} ns={ns}", flush=True)
    rng = np.random.default_rng(sum(dims) + ns)
    so = rand_so3(rng, *dims, ns)
    ci = O3.setup_interp(so)
    nc = ci.shape[1:]
    for p in range(26) if dims[1] < 100 else (0, 13, 25):
        c = ci.copy()
        at = tuple(int(rng.integers(1, n)) for n in nc)
        c[(p,) + at] = bad
        soc = torch.zeros((14,) + nc, dtype=torch.float64, device="cuda")
        C.cdr3.setup_galerkin(dev(so), dev(c), soc)
        ref = O3.setup_galerkin(so, c)
        inner = (slice(None),) + (slice(1, -1),) * 3
        assert np.array_equal(host(soc)[inner], ref[inner], equal_nan=True), (p, at)


def _so2(rng, nx, ny, ns):
    """Random couplings inside the grid, diagonally dominant, zero across the boundary."""
    so = np.zeros((ns, ny + 2, nx + 2))
    so[1, 1:-1, 2:-1] = rng.uniform(0.1, 1.0, (ny, nx - 1))
    so[2, 2:-1, 1:-1] = rng.uniform(0.1, 1.0, (ny - 1, nx))
    if ns == 5:
        so[3, 2:-1, 2:-1] = rng.uniform(0.1, 1.0, (ny - 1, nx - 1))
        so[4, 2:-1, 2:-1] = rng.uniform(0.1, 1.0, (ny - 1, nx - 1))
    so[0, 1:-1, 1:-1] = 9.0
    return so


# rows of 64, 128, ... points, one less and one more (thread classes), odd and even, up to the
# longest row of the fused kernel and beyond; boundary values that are not zero.  Extents of at
# least 2: with one the oracle's loops over the second colour run into the ghost layer.
@pytest.mark.parametrize("nx,ny", [(2, 2), (2, 3), (3, 2), (63, 9), (64, 8), (65, 17), (128, 5),
                                   (129, 4), (257, 6), (512, 3), (513, 3), (1025, 3), (2047, 4),
                                   (2049, 3), (4096, 2), (4097, 3)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_gs9_rows(nx, ny, dtype):
    import cedar_amd as C
    print(f"\ngs9 {nx}x{ny} {dtype}", flush=True)
    rng = np.random.default_rng(nx + ny)
    dt = torch.float64 if dtype == "f64" else torch.float32
    q, qf = rng.standard_normal((ny + 2, nx + 2)), rng.standard_normal((ny + 2, nx + 2))
    so = _so2(rng, nx, ny, 5)
    sor = O.setup_recip(so)
    for ud in (O.DOWN, O.UP):
        ref = O.relax_gs(so, qf, q, sor, ud)
        g = host(C.relax_gs(dev(so, dt), dev(qf, dt), dev(q, dt), dev(sor, dt), ud))
        if dtype == "f64":
            assert np.array_equal(g, ref), ud
        else:  # 9 products and sums of values of order 1 a point, two colours deep
            assert np.abs(g - ref).max() <= 20 * 2.0 ** -24 * np.abs(ref).max(), ud


def test_gs9_rows_batch_of_shared_operators():
    """Several right-hand sides per operator: each problem as if relaxed alone."""
    import cedar_amd as C
    rng = np.random.default_rng(3)
    nops, nrhs, nx, ny = 3, 4, 130, 70
    ops = np.stack([_so2(rng, nx, ny, 5) for _ in range(nops)])
    b = rng.standard_normal((nops * nrhs, ny + 2, nx + 2))
    kw = dict(relaxation="point", maxiter=3, tol=1e-30)
    x, _ = C.Solver(dev(ops), nrhs=nrhs, **kw).solve(dev(b))
    for k in range(nops * nrhs):
        one, _ = C.Solver(dev(ops[k // nrhs]), **kw).solve(dev(b[k]))
        assert torch.equal(x[k], one), k


@pytest.mark.parametrize("dims", [(2, 2, 2), (2, 3, 3), (15, 4, 5), (16, 5, 4), (17, 9, 3),
                                  (33, 6, 7), (64, 3, 4), (65, 7, 2), (129, 3, 3), (257, 3, 2),
                                  (512, 2, 3), (513, 3, 2)])
@pytest.mark.parametrize("dtype", ["f64", "f32"])
def test_gs27_rows(dims, dtype):
    import cedar_amd as C
    print(f"\ngs27 {dims} {dtype}", flush=True)
    nx, ny, nz = dims
    rng = np.random.default_rng(sum(dims))
    dt = torch.float64 if dtype == "f64" else torch.float32
    so = rand_so3(rng, nx, ny, nz, 14)
    shp = (nz + 2, ny + 2, nx + 2)
    q, qf = rng.standard_normal(shp), rng.standard_normal(shp)
    sor = O3.setup_recip(so)
    K = C.cdr3
    for ud in (K.DOWN, K.UP):
        ref = O3.relax_gs(so, qf, q, sor, ud)
        g = host(K.relax_gs(dev(so, dt), dev(qf, dt), dev(q, dt), dev(sor, dt), ud))
        if dtype == "f64":
            assert np.array_equal(g, ref), ud
        else:  # 27 products and sums a point, eight colours deep
            assert np.abs(g - ref).max() <= 100 * 2.0 ** -24 * np.abs(ref).max(), ud


# tiles of 64 elements and groups of 16 lines, one less, one more; two and three tiles; a pivot that
# is not positive in the first tile, at a tile's edge and in the last element
@pytest.mark.parametrize("nx,ny", [(2, 3), (63, 15), (64, 16), (65, 17), (129, 33), (193, 5), (7, 130)])
@pytest.mark.parametrize("ns", [3, 5])
def test_line_setup(nx, ny, ns):
    import cedar_amd as C
    print(f"\nline setup {nx}x{ny} ns={ns}", flush=True)
    so = _so2(np.random.default_rng(nx + ny + ns), nx, ny, ns)
    for d in ("x", "y"):
        sor = O.setup_lines(so, d)
        sor = sor[0] if isinstance(sor, tuple) else sor
        g = torch.zeros(sor.shape, dtype=torch.float64, device="cuda")
        assert np.array_equal(host(C.setup_lines(dev(so), g, d)), sor), d


# lines of at most 8 points, 64 to a workgroup, of at most 64, 16 to one, and longer: groups that are
# full, one short, one over; every pivot in turn not positive
@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 63, 64, 65])
@pytest.mark.parametrize("nl", [15, 16, 17, 63, 64, 65, 129])
@pytest.mark.parametrize("d", ["x", "y"])
def test_line_setup_of_short_lines(n, nl, d):
    import cedar_amd as C
    nx, ny = (n, nl) if d == "x" else (nl, n)
    print(f"\nshort line setup {d} {nx}x{ny}", flush=True)
    so = _so2(np.random.default_rng(n + nl), nx, ny, 5)
    sor = O.setup_lines(so, d)
    sor = sor[0] if isinstance(sor, tuple) else sor
    g = torch.zeros(sor.shape, dtype=torch.float64, device="cuda")
    assert np.array_equal(host(C.setup_lines(dev(so), g, d)), sor)
    for k in range(0, n, 7):
        bad = so.copy()
        bad[(0,) + ((nl, k + 1) if d == "x" else (k + 1, nl))] = -1.0
        with pytest.raises(C.CedarHipError):
            C.setup_lines(dev(bad), g, d)


# 200000 lines of 4 points move 20 MB, a few us beside a launch: three buffers for each group of 16 made
# them take 3 times as long as 2048 lines, one for 64 takes 1.2
@pytest.mark.parametrize("d", ["x", "y"])
def test_line_setup_of_short_lines_scales(d):
    import cedar_amd as C
    best = {}
    for nl in (2048, 200000):
        nx, ny = (4, nl) if d == "x" else (nl, 4)
        so = torch.full((5, ny + 2, nx + 2), 0.5, dtype=torch.float64, device="cuda")
        so[0] = 9.0
        sor = torch.zeros((2, ny + 2, nx + 2), dtype=torch.float64, device="cuda")
        C.setup_lines(so, sor, d)
        for _ in range(6):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            C.setup_lines(so, sor, d)
            a.record()
            for _ in range(20):
                C.setup_lines(so, sor, d)
            b.record()
            b.synchronize()
            best[nl] = min(best.get(nl, 1e9), a.elapsed_time(b) / 20)
    print(f"\nshort line setup {d}: {best}", flush=True)
    assert best[200000] < 2 * best[2048], best


@pytest.mark.parametrize("k", [0, 1, 63, 64, 128])
@pytest.mark.parametrize("d", ["x", "y"])
def test_line_setup_reports_the_failing_pivot(k, d):
    import cedar_amd as C
    n = 129
    so = _so2(np.random.default_rng(k), n, n, 5)
    so[(0,) + ((5, k + 1) if d == "x" else (k + 1, 5))] = -1.0
    g = torch.zeros((2, n + 2, n + 2), dtype=torch.float64, device="cuda")
    with pytest.raises(C.CedarHipError):
        C.setup_lines(dev(so), g, d)


# first levels of the fused coarse cycle that lie in LDS whole, but for the interpolation, for the
# operator, with the iterate alone, not at all, in both word sizes; lines of 16, 32, 64 points and
# more, several to a wavefront, odd and even.  num_levels = 3 leaves one level to start at.
@pytest.mark.parametrize("precision", ["f64", "mixed"])
@pytest.mark.parametrize("relax", ["point", "line-x", "line-y", "line-xy"])
@pytest.mark.parametrize("nx,ny", [(31, 33), (33, 18), (63, 64), (66, 61), (95, 90), (127, 128),
                                   (130, 60), (163, 150), (200, 199), (60, 250)])
def test_fused_cycle_memory_modes(nx, ny, relax, precision):
    import cedar_amd as C
    print(f"\nfused {nx}x{ny} {relax} {precision}", flush=True)
    rng = np.random.default_rng(nx + ny)
    so, b = dev(_so2(rng, nx, ny, 5)), dev(rng.standard_normal((ny + 2, nx + 2)))
    kw = dict(relaxation=relax, nrelax_pre=2, nrelax_post=1, num_levels=3, maxiter=3, tol=1e-30,
              precision=precision)
    x, h = C.Solver(so, **kw).solve(b)
    y, g = C.Solver(so, fused_coarse=False, **kw).solve(b)
    assert torch.equal(x, y) and np.array_equal(h, g)


# FP32 transfers move blocks inside the grid as pairs and those at its last points one by one: the
# smallest grids, odd and even extents, one tile of 64 x 16 coarse points and a remainder.  Every
# result is a sum of at most 9 products with one quotient, so at most 12 roundings of 2^-24 of the
# sum of its terms' sizes.
@pytest.mark.parametrize("nx,ny", [(3, 3), (4, 3), (3, 4), (5, 6), (31, 33), (127, 17), (128, 34),
                                   (129, 65), (130, 66)])
@pytest.mark.parametrize("ns", [3, 5])
def test_fp32_transfers(nx, ny, ns):
    import cedar_amd as C
    print(f"\nFP32 transfers {nx}x{ny} ns={ns}", flush=True)
    rng = np.random.default_rng(5 * nx + ny + ns)
    r32 = lambda a: np.asarray(a, dtype=np.float32).astype(np.float64)
    so = r32(_so2(rng, nx, ny, ns))
    ci = r32(O.setup_interp(so))
    q, res, qc = (r32(rng.standard_normal(s)) for s in (so.shape[1:], so.shape[1:], ci.shape[1:]))
    f = lambda a: dev(a, torch.float32)
    g, h = f(q), torch.zeros(ci.shape[1:], dtype=torch.float32, device="cuda")
    C.interp_add(g, f(qc), f(res), f(so), f(ci))
    C.restrict(f(ci), f(res), h)
    size = [O.interp_add(*map(np.abs, (q, qc, res, so, ci)))[0], O.restrict(abs(ci), abs(res))]
    want = [O.interp_add(q, qc, res, so, ci)[0], O.restrict(ci, res)]
    for got, w, s in zip((host(g), host(h)), want, size):
        assert (np.abs(got - w) <= 12 * 2.0 ** -24 * np.abs(s)).all()


def _cycle3(C, lv, abd, l, x, b, pre, post):
    """One V-cycle, every sweep in place, level by level."""
    so, ci, sor = lv[l]
    if l == len(lv) - 1:
        C.cdr3.solve_cg(x, b, abd)
        return
    for _ in range(pre):
        C.cdr3.relax_gs(so, b, x, sor, 0)
    res, ci = torch.zeros_like(x), lv[l + 1][1]
    C.cdr3.residual(so, b, x, res)
    xc, bc = torch.zeros_like(lv[l + 1][0][0]), torch.zeros_like(lv[l + 1][0][0])
    C.cdr3.restrict(ci, res, bc)
    _cycle3(C, lv, abd, l + 1, xc, bc, pre, post)
    C.cdr3.interp_add(x, xc, res, so, ci)
    for _ in range(post):
        C.cdr3.relax_gs(so, b, x, sor, 1)


def _op7(rand, shape):
    so = torch.zeros((4,) + shape, device="cuda", dtype=torch.float64)
    so[0, 1:-1, 1:-1, 1:-1] = 7.0
    so[1, 1:-1, 1:-1, 1:] = 0.1 + 0.9 * rand(shape[0] - 2, shape[1] - 2, shape[2] - 1)
    so[2, 1:-1, 1:, 1:-1] = 0.1 + 0.9 * rand(shape[0] - 2, shape[1] - 1, shape[2] - 2)
    so[3, 1:, 1:-1, 1:-1] = 0.1 + 0.9 * rand(shape[0] - 1, shape[1] - 2, shape[2] - 2)
    return so


# A five-point sweep moves 8 values a point where a nine-point one moves 12: it takes 0.57 of its time
# when it waits for memory alone, and took 1.07 of it when its factors were loaded one at a time.
def test_long_fp32_y_lines_load_their_factors_in_groups():
    import cedar_amd as C
    n, best = 4090, {}
    for ns in (3, 5):
        so = torch.full((ns, n + 2, n + 2), 0.5, device="cuda")
        so[0] = 9.0
        sor = torch.full((2, n + 2, n + 2), 0.1, device="cuda")
        sor[0] = 9.0
        f, q = torch.rand_like(so[0]), torch.rand_like(so[0])
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            C.relax_lines(so, f, q, sor, 0, "y")
            a.record()
            for _ in range(10):
                C.relax_lines(so, f, q, sor, 0, "y")
            b.record()
            b.synchronize()
            best[ns] = min(best.get(ns, 1e9), a.elapsed_time(b) / 10)
    print(f"\nFP32 y-lines of {n} points: {best}", flush=True)
    assert best[3] < 0.85 * best[5], best


# One 7-point sweep out of place against the one in place, every shape of the launch by itself: 1 to 4
# points a side; rows of one group of 62 pairs that is nearly full, full, one over, and of three; tiles
# of 1, 3, 13 and 14 rows with and without a remainder; slabs of one plane, of all, and of lengths that
# divide the planes and do not; a march of 25 and of 60 planes; 1, 255 to 257 and 1000 workgroups.
# Ghosts are those of a third array (those of q and out are NaN), the rest of out stays.
@pytest.mark.parametrize("dims,rows,planes", [
    ((1, 1, 1), 0, 0), ((2, 1, 1), 0, 0), ((1, 2, 3), 1, 1), ((3, 3, 3), 0, 0), ((4, 4, 4), 3, 2),
    ((4, 2, 3), 14, 3), ((3, 4, 1), 1, 1), ((121, 5, 4), 0, 0), ((122, 13, 9), 13, 3), ((123, 14, 9), 14, 4),
    ((124, 15, 9), 14, 1), ((125, 28, 7), 14, 7), ((126, 29, 10), 14, 5), ((127, 9, 6), 3, 6),
    ((247, 15, 4), 0, 0), ((371, 17, 5), 7, 2), ((200, 16, 50), 14, 25), ((130, 30, 60), 0, 60),
    ((30, 60, 52), 14, 20), ((20, 51, 15), 3, 1), ((20, 16, 128), 14, 1), ((20, 3, 257), 3, 1),
    ((140, 70, 100), 14, 1), ((200, 200, 200), 0, 0)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_gs7_sweep_shapes(dims, rows, planes, dtype):
    import cedar_amd as C
    print(f"\n7-point sweep {dims} rows {rows} planes {planes} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(sum(dims) + rows + planes)
    shape = tuple(n + 2 for n in dims[::-1])
    rand = lambda *s: torch.rand(*s, generator=gen, device="cuda", dtype=torch.float64)
    so = _op7(rand, shape)
    sor = torch.zeros((2,) + shape, device="cuda", dtype=torch.float64)
    C.cdr3.setup_recip(so, sor)
    so, sor, f, x = (t.to(dtype) for t in (so, sor, rand(*shape) - 0.5, rand(*shape) - 0.5))
    inner = (slice(1, -1),) * 3
    q = torch.full_like(x, float("nan"))
    q[inner] = x[inner]
    ghosts = torch.full_like(x, float("nan"))
    edge = torch.ones_like(x, dtype=torch.bool)
    edge[inner] = False
    ghosts[edge] = x[edge]
    for ud in (0, 1):
        want = C.cdr3.relax_gs(so, f, x.clone(), sor, ud)
        out = torch.full_like(x, 7.0)
        C.cdr3.relax_gs7_to(so, f, q, out, sor, ud, ghosts=ghosts, rows=rows, planes=planes)
        assert torch.equal(out[inner], want[inner]), ud
        assert bool((out[edge] == 7.0).all())


def test_gs7_sweep_refuses_what_it_cannot_launch():
    import cedar_amd as C
    x, so, sor = (torch.zeros(n + (5, 5, 5), dtype=torch.float64, device="cuda") for n in ((), (4,), (2,)))
    out = torch.zeros_like(x)
    for rows, planes in ((15, 1), (-1, 1), (1, 4), (1, -1)):
        with pytest.raises(C.CedarHipError):
            C.cdr3.relax_gs7_to(so, x, x, out, sor, 0, rows=rows, planes=planes)
    with pytest.raises(C.CedarHipError):
        C.cdr3.relax_gs7_to(so, x, x, x, sor, 0)


# the cycles of test_gs7_sweeps take the out-of-place form at their sizes; levels where the two launches
# are faster do not, among them planes of a multiple of 8 workgroups
@pytest.mark.parametrize("dims,taken", [((125, 97, 104), True), ((126, 167, 59), True),
                                        ((126, 65, 152), True), ((117, 70, 152), True),
                                        ((249, 70, 71), True), ((248, 97, 53), True),
                                        ((373, 53, 62), True), ((200, 200, 200), True),
                                        ((125, 96, 104), False), ((248, 94, 53), False),
                                        ((122, 157, 77), False), ((116, 63, 201), False),
                                        ((63, 63, 63), False), ((3, 3, 3), False)])
def test_gs7_sweep_sizes(dims, taken):
    import cedar_amd as C
    assert C.cdr3.relax_gs7_to_pays(*dims) == taken


def _fmg3(C, lv, abd, l, x, b, pre, post):
    """The F-cycle from the finest level down, every sweep in place."""
    so, ci, sor = lv[l]
    if l == len(lv) - 1:
        C.cdr3.solve_cg(x, b, abd)
        return
    ci = lv[l + 1][1]
    bc, xc = torch.zeros_like(lv[l + 1][0][0]), torch.zeros_like(lv[l + 1][0][0])
    C.cdr3.restrict(ci, b, bc)
    _fmg3(C, lv, abd, l + 1, xc, bc, pre, post)
    x.zero_()
    C.cdr3.interp_add(x, xc, torch.zeros_like(x), so, ci)
    _cycle3(C, lv, abd, l, x, b, pre, post)


# an F-cycle enters the V-cycle with the residual's array written; the sweeps borrow that array
@pytest.mark.parametrize("dims", [(125, 97, 104), (126, 167, 59)])
@pytest.mark.parametrize("pre,post", [(2, 1), (1, 2)])
def test_gs7_sweeps_in_f_cycles(dims, pre, post):
    import cedar_amd as C
    print(f"\nF-cycle, 7-point sweeps {dims} {pre},{post}", flush=True)
    assert C.cdr3.relax_gs7_to_pays(*dims)
    gen = torch.Generator(device="cuda").manual_seed(sum(dims) + pre)
    shape = tuple(n + 2 for n in dims[::-1])
    rand = lambda *s: torch.rand(*s, generator=gen, device="cuda", dtype=torch.float64)
    so = _op7(rand, shape)
    b = torch.zeros(shape, device="cuda", dtype=torch.float64)
    b[1:-1, 1:-1, 1:-1] = rand(*dims[::-1]) - 0.5
    s = C.Solver3(so, nrelax_pre=pre, nrelax_post=post, maxiter=1, tol=1e-30, cycle="f")
    lv = []
    for l in range(s.nlevels):
        a, ci = s.level_arrays(l)
        a = dev(a)
        sor = torch.zeros((2,) + tuple(a.shape[1:]), device="cuda", dtype=torch.float64)
        C.cdr3.setup_recip(a, sor)
        lv.append((a, None if ci is None else dev(ci), sor))
    abd = C.cdr3.setup_cg(lv[-1][0])
    want, got = torch.zeros_like(b), torch.zeros_like(b)
    for _ in range(2):  # the second one finds the arrays as the first one left them
        s.vcycle(got, b)
        _fmg3(C, lv, abd, 0, want, b, pre, post)
        assert torch.equal(got, want)


# 7-point sweeps that take both colours in one launch: one to three groups of 62 pairs along a row,
# the last one full, nearly full or short, odd and even; tiles of 14 rows with and without a
# remainder, slabs of three planes with one of two; couplings to the ghosts of a nonzero boundary; odd
# and even numbers of sweeps.  The sizes are about the smallest that take this path (asserted in
# test_gs7_sweep_sizes); test_gs7_sweep_shapes has the other slabs.
@pytest.mark.parametrize("dims", [(125, 96, 104), (126, 167, 59), (126, 65, 152), (117, 70, 152),
                                  (249, 70, 71), (248, 94, 53), (373, 53, 62), (125, 97, 104),
                                  (248, 97, 53)])
@pytest.mark.parametrize("pre,post", [(2, 1), (1, 2), (3, 0)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_gs7_sweeps(dims, pre, post, dtype):
    import cedar_amd as C
    print(f"\n7-point sweeps {dims} {pre},{post} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(sum(dims) + pre)
    shape = tuple(n + 2 for n in dims[::-1])
    rand = lambda *s: torch.rand(*s, generator=g, device="cuda", dtype=torch.float64)
    so = torch.zeros((4,) + shape, device="cuda", dtype=torch.float64)
    so[0, 1:-1, 1:-1, 1:-1] = 7.0
    so[1, 1:-1, 1:-1, 1:] = 0.1 + 0.9 * rand(shape[0] - 2, shape[1] - 2, shape[2] - 1)
    so[2, 1:-1, 1:, 1:-1] = 0.1 + 0.9 * rand(shape[0] - 2, shape[1] - 1, shape[2] - 2)
    so[3, 1:, 1:-1, 1:-1] = 0.1 + 0.9 * rand(shape[0] - 1, shape[1] - 2, shape[2] - 2)
    b, x = rand(*shape) - 0.5, rand(*shape) - 0.5
    f64 = dtype == torch.float64
    s = C.Solver3(so, nrelax_pre=pre, nrelax_post=post, maxiter=1, tol=1e-30,
                  precision="f64" if f64 else "mixed")
    lv = []
    for l in range(s.nlevels):
        a, ci = s.level_arrays(l)
        a = dev(a)
        sor = torch.zeros((2,) + tuple(a.shape[1:]), device="cuda", dtype=torch.float64)
        C.cdr3.setup_recip(a, sor)
        lv.append(tuple(None if v is None else v.to(dtype)
                        for v in (a, None if ci is None else dev(ci), sor)))
        abd = C.cdr3.setup_cg(a) if l == s.nlevels - 1 else None
    want, got = x.clone(), x.clone()
    if f64:
        s.vcycle(got, b)
        _cycle3(C, lv, abd, 0, want, b, pre, post)
    else:
        s.solve(b, got)
        r = torch.zeros_like(b)
        C.cdr3.residual(so, b, x, r)
        e = torch.zeros_like(r, dtype=dtype)
        _cycle3(C, lv, abd, 0, e, r.to(dtype), pre, post)
        inner = (slice(1, -1),) * 3  # the outer iterate's ghosts are those of its own arrays
        want, got = (want + e.double())[inner], got[inner]
    assert torch.equal(got, want)
