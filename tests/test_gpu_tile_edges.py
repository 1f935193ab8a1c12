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


# coarse rows of 64 points, one less and one more; the smallest grids; even extents, whose last
# fine points lie beyond the last coarse one
@pytest.mark.parametrize("dims", [(3, 3, 3), (4, 3, 5), (125, 5, 4), (127, 6, 5), (128, 4, 9),
                                  (129, 9, 6), (131, 3, 3), (6, 129, 5)])
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
