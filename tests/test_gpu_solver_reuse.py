"""Solvers built from the memory of destroyed ones, on one and on several threads and streams."""
import threading

import numpy as np
import pytest

from cedar_amd import gallery as G

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _problem(n, seed):
    so, b, _ = G.heterogeneous_9pt(n, seed=seed, block=8, sigma=1.0)
    return torch.as_tensor(so).cuda(), torch.as_tensor(b).cuda()


KW = dict(relaxation="line-xy", nrelax_pre=1, nrelax_post=1, maxiter=30, tol=1e-10)


@pytest.mark.parametrize("precision", ["f64", "mixed"])
def test_a_rebuilt_solver_gives_the_same_solution(precision):
    import cedar_amd as C
    first = {}
    for rnd in range(3):
        for n in (65, 96, 130):
            so, b = _problem(n, n)
            s = C.Solver(so, precision=precision, **KW)
            x, h = s.solve(b)
            s.close()
            if rnd == 0:
                first[n] = (x, h)
            else:
                assert torch.equal(x, first[n][0]) and np.array_equal(h, first[n][1])


def test_rebuilt_3d_solvers():
    import cedar_amd as C
    so, b, _ = G.poisson3_sine(33)
    so, b = torch.as_tensor(so).cuda(), torch.as_tensor(b).cuda()
    ref = None
    for relax in ("point", "plane-xy", "point", "plane-xy"):
        s = C.Solver3(so, relaxation=relax, maxiter=4)
        x, h = s.solve(b)
        s.close()
        ref = ref or {}
        if relax in ref:
            assert torch.equal(x, ref[relax][0]) and np.array_equal(h, ref[relax][1])
        ref[relax] = (x, h)


def test_threads_and_streams_that_build_and_destroy_solvers():
    import cedar_amd as C
    sizes = (65, 66, 96, 97)
    probs = {n: _problem(n, n) for n in sizes}
    ref = {n: C.Solver(probs[n][0], **KW).solve(probs[n][1]) for n in sizes}
    torch.cuda.synchronize()
    bad = []

    def work(k):
        try:
            st = torch.cuda.Stream()
            with torch.cuda.stream(st):
                for r in range(4):
                    n = sizes[(k + r) % len(sizes)]
                    s = C.Solver(probs[n][0], **KW)
                    x, h = s.solve(probs[n][1])
                    s.close()
                    if not (torch.equal(x, ref[n][0]) and np.array_equal(h, ref[n][1])):
                        bad.append((k, r, n))
                st.synchronize()
        except BaseException as exc:  # reported by the main thread
            bad.append(exc)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad, bad


def test_closed_solvers_give_their_memory_back():
    """memory_trim returns what closed solvers left, to the device and so to other libraries; with a
    limit of 0 they leave nothing; a limit between evicts, and solutions stay the same."""
    import cedar_amd as C
    so, b = _problem(700, 3)
    free = lambda: torch.cuda.mem_get_info()[0]

    def solve():
        s = C.Solver(so, **KW)
        x, h = s.solve(b)
        s.close()
        return x, h

    first = solve()
    torch.cuda.synchronize()
    C.memory_trim()
    base = free()
    prev = C.memory_limit(1 << 32)
    least = 5 * 702 * 702 * 8  # the factors of both line directions and the residual of the finest level
    try:
        solve()
        torch.cuda.synchronize()
        assert base - free() > least
        assert C.memory_trim() > least
        assert free() >= base - (4 << 20)
        assert C.memory_trim() == 0
        for limit in (0, 20 << 20):
            C.memory_limit(limit)
            for _ in range(2):
                x, h = solve()
                assert torch.equal(x, first[0]) and np.array_equal(h, first[1])
            torch.cuda.synchronize()
            assert C.memory_limit(limit) == limit
            assert C.memory_trim() <= limit
    finally:
        C.memory_limit(prev)


def test_recorded_fused_starts_are_listed_and_forgotten():
    """The first level of the fused cycle that a solver's setup chose is listed with its device, taken
    over by the next solver, and forgotten with the line shapes; none of it changes a solution."""
    import cedar_amd as C
    so, b = _problem(300, 5)
    prev = C.autotune(True)
    mine = lambda: [r for r in C.autotune_report() if r["dir"] == "f" and "300 x 300" in r["kernel"]]
    try:
        C.autotune_clear()
        assert C.autotune_report() == []
        ref = None
        for _ in range(6):  # disturbed timings are not recorded
            s = C.Solver(so, **KW)
            x, h = s.solve(b)
            s.close()
            ref = ref or (x, h)
            assert torch.equal(x, ref[0]) and np.array_equal(h, ref[1])
            if mine():
                break
        r, = mine()
        assert r["device"] == torch.cuda.current_device() and r["fp"] == 64 and r["nb"] == 1
        n = 300
        for _ in range(r["shape"]):
            n = (n - 1) // 2 + 1
        assert n <= 128 and (r["ii"], r["jj"]) == (n + 2, n + 2)
        s = C.Solver(so, **KW)
        x, h = s.solve(b)
        s.close()
        assert mine() == [r] and torch.equal(x, ref[0]) and np.array_equal(h, ref[1])
        C.autotune_clear()
        assert C.autotune_report() == []
    finally:
        C.autotune(prev)


# Solvers built, used and closed beside a capture of the caller's, in the modes that allow it: another
# thread's work beside a thread-local or relaxed capture, and a close inside a relaxed one
@pytest.mark.parametrize("mode,thread,what", [("thread_local", True, "close"), ("thread_local", True, "new"),
                                              ("relaxed", True, "close"), ("relaxed", True, "new"),
                                              ("relaxed", False, "close")])
@pytest.mark.parametrize("dim", [2, 3])
def test_solvers_beside_a_capture(mode, thread, what, dim):
    import cedar_amd as C
    print(f"\n{dim}D solver, {what} beside a {mode} capture, other thread: {thread}", flush=True)
    if dim == 2:
        so, b = _problem(96, 1)
        build = lambda: C.Solver(so, **KW)
    else:
        so, b, _ = G.poisson3_sine(17)
        so, b = torch.as_tensor(so).cuda(), torch.as_tensor(b).cuda()
        build = lambda: C.Solver3(so, relaxation="plane-xy", maxiter=3)
    held = build()
    ref = held.solve(b)
    x, y = torch.ones(1000, device="cuda"), torch.zeros(1000, device="cuda")
    torch.cuda.synchronize()
    g, got = torch.cuda.CUDAGraph(), []

    def act():
        try:
            if what == "close":
                held.close()
            else:
                s = build()
                got.append(s.solve(b))
                s.close()
        except Exception as exc:  # reported below
            got.append(exc)

    with torch.cuda.graph(g, stream=torch.cuda.Stream(), capture_error_mode=mode):
        y.add_(x)
        if thread:
            t = threading.Thread(target=act)
            t.start()
            t.join()
        else:
            act()
        y.add_(x)
    for _ in range(3):
        g.replay()
    torch.cuda.synchronize()
    assert bool((y == 6).all())
    if what == "close":
        assert got == []
    else:
        assert torch.equal(got[0][0], ref[0]) and np.array_equal(got[0][1], ref[1])


def test_threads_that_capture_while_others_close():
    """Every solver times and captures its cycles anew while three other threads close theirs."""
    import cedar_amd as C
    sizes = (65, 66, 96, 97)
    probs = {n: _problem(n, n) for n in sizes}
    ref = {n: C.Solver(probs[n][0], **KW).solve(probs[n][1]) for n in sizes}
    torch.cuda.synchronize()
    bad = []

    def work(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for r in range(4):
                    n = sizes[(k + r) % len(sizes)]
                    s = C.Solver(probs[n][0], **KW)
                    x, h = s.solve(probs[n][1])
                    s.close()
                    if not (torch.equal(x, ref[n][0]) and np.array_equal(h, ref[n][1])):
                        bad.append((k, r, n))
                torch.cuda.current_stream().synchronize()
        except BaseException as exc:  # reported by the main thread
            bad.append(exc)

    for _ in range(20):
        C.autotune_clear()
        ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        assert not bad, bad


def test_a_solver_whose_level_pointers_were_given_out_leaves_nothing():
    """Work of the caller's own on another stream may still use such a pointer after the solver is
    destroyed, so its blocks go back to the device and not to the next solver."""
    import cedar_amd as C
    so, b = _problem(200, 2)
    for give in (True, False):
        s = C.Solver(so, **KW)
        s.solve(b)
        if give:
            assert s.level(1)[2]
        C.memory_trim()  # what setup itself gave back
        s.close()
        left = C.memory_trim()
        assert left == 0 if give else left > 5 * 202 * 202 * 8


@pytest.mark.parametrize("dim", [2, 3])
@pytest.mark.parametrize("captured", [True, False])
def test_a_solver_recorded_into_a_graph_leaves_nothing(dim, captured):
    """A graph of the caller's may still run on another stream when its solver is destroyed: the
    solver's blocks, and those of its plane solvers, then go back to the device."""
    import cedar_amd as C
    side = torch.cuda.Stream()
    if dim == 2:
        so, b = _problem(200, 2)
        build = lambda: C.Solver(so, **KW)
    else:
        so, b, _ = G.poisson3_sine(33)
        so, b = torch.as_tensor(so).cuda(), torch.as_tensor(b).cuda()
        build = lambda: C.Solver3(so, relaxation="plane-xyz", maxiter=3)
    with torch.cuda.stream(side):
        s = build()
        want = torch.zeros_like(b)
        s.vcycle(want, b)
    torch.cuda.synchronize()
    x = torch.zeros_like(b)
    g = torch.cuda.CUDAGraph()
    if captured:
        with torch.cuda.graph(g, stream=side):
            s.vcycle(x, b)
        g.replay()  # on the current stream
    else:
        with torch.cuda.stream(side):
            s.vcycle(x, b)
    C.memory_trim()
    s.close()
    left = C.memory_trim()
    torch.cuda.synchronize()
    assert torch.equal(x, want)
    assert left == 0 if captured else left > 0
