"""Performance cases: what a program does with this framework, through its public entry points.

A case is a dict of plain values; `kind` names the entry point it goes through:

  solve2d     Solver(so).solve(b): 2D, one operator; `new` builds the solver in the pass too (a
              program whose coefficients change from step to step), else the handle is kept
  batch2d     BatchSet(operators).solve(rhs): many problems of mixed sizes, several right-hand sides
  gradient2d  adjoint.solve(theta, f), backward: differentiated diffusion solves
  solve3d     Solver3(so).solve(b): 3D, point or plane relaxation; `new` as above
  steps2d     the kernel calls of one two-grid step, as a host program that keeps its own cycle
              makes them: smoothing, residual, restriction, interpolation

Sizes follow the repository's benchmark workloads, the reference's tests and examples, and the
ranges between them; every side that is not of the form 2^k - 1 is there on purpose.
"""
import math

import numpy as np
import torch

import cedar_amd
from cedar_amd import adjoint, cdr2, cdr3, gallery
from cedar_amd.batch import BatchSet

CONTRAST = 1e4
MAXITER = 60


def listed():
    two = dict(kind="solve2d", periodic="", new=False, nrelax_pre=1, nrelax_post=1)
    three = dict(kind="solve3d", new=False, nrelax_pre=1, nrelax_post=1)
    return [
        # the smallest call: a small Poisson problem with Cedar's default settings, launch-bound
        dict(two, name="poisson2d_63", op="poisson", nx=63, ny=63, relaxation="point",
             nrelax_pre=2, precision="f64", tol=1e-8),
        # the benchmark's Poisson workload: 511^2, red-black Gauss-Seidel, V(2,1), FP64
        dict(two, name="poisson2d_511", op="poisson", nx=511, ny=511, relaxation="point",
             nrelax_pre=2, precision="f64", tol=1e-10),
        # the README's example: 1023^2 jumping coefficients, mixed precision
        dict(two, name="diffusion2d_1023_mixed", op="diffusion", nx=1023, ny=1023,
             relaxation="line-xy", precision="mixed", tol=1e-10),
        # the headline workload: 4095^2 jumping coefficients, mixed precision
        dict(two, name="diffusion2d_4095_mixed", op="diffusion", nx=4095, ny=4095,
             relaxation="line-xy", precision="mixed", tol=1e-10),
        # a time step whose coefficients changed: hierarchy and solve, FP64, even and ragged sides
        dict(two, name="diffusion2d_new_1500x1100", op="diffusion", nx=1500, ny=1100,
             relaxation="line-xy", precision="f64", tol=1e-10, new=True),
        # the periodic example's operator, periodic in x, with line smoothing (a channel)
        dict(two, name="periodic2d_512x511", op="poisson", nx=512, ny=511, periodic="x",
             relaxation="line-xy", precision="f64", tol=1e-10),
        # many problems of mixed sizes with 4 right-hand sides each (an eighth of the batch workload)
        dict(kind="batch2d", name="batch2d_12x4", sizes="257,513,1025", nprob=12, nrhs=4, tol=1e-10),
        # the training step of a coefficient field: solve, adjoint solve, gradient
        dict(kind="gradient2d", name="gradient2d_4x1025", nb=4, n=1025, tol=1e-10),
        # the kernel calls of a host program's own two-grid step on one level, FP64
        dict(kind="steps2d", name="steps2d_2047x1500", nx=2047, ny=1500, points=9, dtype="f64",
             relaxation="point"),
        # the reference's 3D Poisson test (200^3), from operator to solution, FP64
        dict(three, name="poisson3d_new_200", op="poisson", nx=200, ny=200, nz=200, new=True,
             relaxation="point", nrelax_pre=2, precision="f64", tol=1e-8),
        # 27-point finite elements in a box, kept handle, mixed precision
        dict(three, name="fe3d_127x127x95_mixed", op="fe", nx=127, ny=127, nz=95,
             relaxation="point", nrelax_pre=2, precision="mixed", tol=1e-10),
        # the benchmark's 3D workload: 255^3 anisotropic jumps, plane relaxation, mixed precision
        dict(three, name="plane3d_255_mixed", op="diffusion", nx=255, ny=255, nz=255,
             relaxation="plane-xy", precision="mixed", tol=1e-10),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["solve2d", "solve2d", "solve2d", "batch2d", "gradient2d", "steps2d",
                       "solve3d", "solve3d"])
    prec = rng.choice(["f64", "mixed"])
    if kind == "solve2d":
        nx = _log(rng, 31, 2600)
        ny = min(2600, max(31, int(nx * math.exp(rng.uniform(-1, 1)))))
        per = rng.choice(["", "", "", "x"])
        if per:  # periodic sides: powers of two, so that every coarsened level keeps an even period
            nx, ny = 2 ** rng.randint(5, 9), min(ny, 700)
        op = "poisson" if per else rng.choice(["poisson", "fe", "diffusion", "diffusion"])
        # point smoothing where the couplings of both directions are alike
        even = op == "fe" or 0.7 < nx / ny < 1.4
        relax = rng.choice(["point", "line-xy"]) if even and op != "diffusion" else "line-xy"
        return dict(kind=kind, op=op, nx=nx, ny=ny, periodic=per, relaxation=relax,
                    nrelax_pre=rng.randint(1, 2), nrelax_post=1, precision=prec, tol=1e-10,
                    new=rng.random() < 0.3)
    if kind == "batch2d":
        sizes = sorted({_log(rng, 33, 600) for _ in range(3)})
        return dict(kind=kind, sizes=",".join(map(str, sizes)), nprob=rng.randint(3, 16),
                    nrhs=rng.choice([1, 2, 4]), tol=1e-10)
    if kind == "gradient2d":
        return dict(kind=kind, nb=rng.randint(1, 6), n=_log(rng, 65, 900), tol=1e-10)
    if kind == "steps2d":
        nx = _log(rng, 65, 2500)
        ny = min(2500, max(65, int(nx * math.exp(rng.uniform(-1, 1)))))
        return dict(kind=kind, nx=nx, ny=ny, points=rng.choice([5, 9]),
                    dtype=rng.choice(["f64", "f32"]), relaxation=rng.choice(["point", "line-xy"]))
    op = rng.choice(["poisson", "fe", "diffusion"])
    top = 150 if op != "diffusion" else 130
    n = _log(rng, 17, top)
    n = [max(17, min(top, int(n * math.exp(rng.uniform(-0.3, 0.3))))) for _ in range(3)]
    if op == "diffusion":
        return dict(kind=kind, op=op, nx=n[0], ny=n[1], nz=n[2], relaxation="plane-xy",
                    nrelax_pre=1, nrelax_post=1, precision=prec, tol=1e-8, new=False)
    return dict(kind=kind, op=op, nx=n[0], ny=n[1], nz=n[2], relaxation="point",
                nrelax_pre=rng.randint(1, 2), nrelax_post=1, precision=prec, tol=1e-8,
                new=rng.random() < 0.4)


# ---- inputs ---------------------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _cells2(nx, ny, g, sigma=2.0, block=16):
    """k per cell, (1, ny+1, nx+1): lognormal on block x block cells, contrast <= CONTRAST."""
    nb = (-(-(ny + 1) // block), -(-(nx + 1) // block))
    t = sigma * torch.randn(nb, generator=g, device="cuda", dtype=torch.float64)
    lim = 0.5 * math.log(CONTRAST)
    k = torch.exp(t.clamp(-lim, lim))
    k = k.repeat_interleave(block, 0).repeat_interleave(block, 1)
    return k[:ny + 1, :nx + 1].contiguous()[None]


def _operator2(case, g):
    nx, ny = case["nx"], case["ny"]
    if case["op"] == "diffusion":
        return adjoint.assemble(_cells2(nx, ny, g))[0].contiguous()
    if case["op"] == "fe":
        return torch.as_tensor(gallery.fe(nx, ny)).cuda()
    if case["periodic"]:
        per = ("x" in case["periodic"], "y" in case["periodic"])
        return torch.as_tensor(gallery.periodic_problem(nx, ny, per)[0]).cuda()
    return torch.as_tensor(gallery.poisson(nx, ny)).cuda()


def _operator3(case, g):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["op"] == "poisson":
        return torch.as_tensor(gallery.poisson3(nx, ny, nz)).cuda()
    if case["op"] == "fe":
        return torch.as_tensor(gallery.fe3(nx, ny, nz)).cuda()
    nb = [-(-n // 8) for n in (nz, ny, nx)]
    k = torch.exp(1.5 * torch.randn(nb, generator=g, device="cuda", dtype=torch.float64))
    for d in range(3):
        k = k.repeat_interleave(8, d)
    k = k[:nz, :ny, :nx].cpu().numpy()
    return torch.as_tensor(gallery.fv7_diffusion(k, (1.0, 1.0, 1e-3))).cuda()


def _rhs(shape, g, periodic=""):
    """Interior values U[-1, 1], ghosts zero (or the periodic images)."""
    b = torch.zeros(shape, dtype=torch.float64, device="cuda")
    inner = (...,) + (slice(1, -1),) * (3 if len(shape) == 3 and not periodic else 2)
    b[inner] = 2 * torch.rand(b[inner].shape, generator=g, device="cuda", dtype=torch.float64) - 1
    if "x" in periodic:
        b[..., :, 0], b[..., :, -1] = b[..., :, -2].clone(), b[..., :, 1].clone()
    if "y" in periodic:
        b[..., 0, :], b[..., -1, :] = b[..., -2, :].clone(), b[..., 1, :].clone()
    return b


def _stack_rhs(m, shape, g):
    b = torch.zeros((m,) + shape, dtype=torch.float64, device="cuda")
    b[:, 1:-1, 1:-1] = 2 * torch.rand(b[:, 1:-1, 1:-1].shape, generator=g, device="cuda",
                                      dtype=torch.float64) - 1
    return b


def _keywords(case):
    kw = dict(relaxation=case["relaxation"], nrelax_pre=case["nrelax_pre"],
              nrelax_post=case["nrelax_post"], maxiter=MAXITER, tol=case["tol"],
              precision=case["precision"])
    if case["kind"] == "solve2d" and case["periodic"]:
        kw["periodic"] = ("x" in case["periodic"], "y" in case["periodic"])
    return kw


def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "solve2d":
        so = _operator2(case, g)
        s["so"], s["b"] = so, _rhs(tuple(so.shape[1:]), g, case["periodic"])
        s["solver"] = None if case["new"] else cedar_amd.Solver(so, **_keywords(case))
    elif kind == "solve3d":
        so = _operator3(case, g)
        s["so"], s["b"] = so, _rhs(tuple(so.shape[1:]), g)
        s["solver"] = None if case["new"] else cedar_amd.Solver3(so, **_keywords(case))
    elif kind == "batch2d":
        ns = _batch_sides(case)
        ops = [adjoint.assemble(_cells2(n, n, g))[0].contiguous() for n in ns]
        m = case["nrhs"]
        s["rhs"] = [_stack_rhs(m, (n + 2, n + 2), g) if m > 1
                    else _stack_rhs(1, (n + 2, n + 2), g)[0] for n in ns]
        s["ops"] = ops
        s["solver"] = BatchSet(ops, nrhs=m, relaxation="line-xy", nrelax_pre=1, nrelax_post=1,
                               maxiter=MAXITER, tol=case["tol"], precision="mixed")
    elif kind == "gradient2d":
        nb, n = case["nb"], case["n"]
        t = torch.randn((nb, 1, n + 5, n + 5), generator=g, device="cuda", dtype=torch.float64)
        s["theta"] = torch.nn.functional.avg_pool2d(t, 5, 1)[:, 0].contiguous()
        s["f"] = _stack_rhs(nb, (n + 2, n + 2), g)
        s["obs"] = 1e-3 * _stack_rhs(nb, (n + 2, n + 2), g)
    elif kind == "steps2d":
        so = _steps_operator(case, g)
        dt = torch.float64 if case["dtype"] == "f64" else torch.float32
        ny, nx = case["ny"], case["nx"]
        ii, jj = nx + 2, ny + 2
        iic, jjc = int((nx - 1) / 2.0 + 1) + 2, int((ny - 1) / 2.0 + 1) + 2
        ci = cdr2.setup_interp(so, torch.zeros((8, jjc, iic), dtype=torch.float64, device="cuda"))
        fac = torch.zeros((2, 2, jj * ii), dtype=torch.float64, device="cuda")
        if case["relaxation"] == "point":
            cdr2.setup_recip(so, fac[0].view(2, jj, ii))
        else:
            cdr2.setup_lines(so, fac[0].view(2, jj, ii), "x")
            cdr2.setup_lines(so, fac[1].view(2, jj, ii), "y")
        s.update(so=so.to(dt), ci=ci.to(dt), fac=fac.view(2, 2, jj, ii).to(dt),
                 f=_stack_rhs(1, (jj, ii), g)[0].to(dt), qc=_stack_rhs(1, (jjc, iic), g)[0].to(dt),
                 q=torch.zeros((jj, ii), dtype=dt, device="cuda"),
                 res=torch.zeros((jj, ii), dtype=dt, device="cuda"),
                 fc=torch.zeros((jjc, iic), dtype=dt, device="cuda"))
    return s


def _steps_operator(case, g):
    if case["points"] == 9:
        return adjoint.assemble(_cells2(case["nx"], case["ny"], g))[0].contiguous()
    return torch.as_tensor(gallery.poisson(case["nx"], case["ny"])).cuda()


def _batch_sides(case):
    sizes = [int(v) for v in case["sizes"].split(",")]
    return [sizes[k % len(sizes)] for k in range(case["nprob"])]


# ---- one pass -------------------------------------------------------------------------------
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind in ("solve2d", "solve3d"):
        solver = s["solver"]
        if solver is None:
            solver = (cedar_amd.Solver if kind == "solve2d" else cedar_amd.Solver3)(
                s["so"], **_keywords(case))
        x, rho = solver.solve(s["b"])
        # the residuals of an FP32 cycle follow its roundings, its cycle count and solution do not;
        # a history as long as the cycles allowed, so that its length does not depend on the inputs
        if case["precision"] == "mixed":
            return {"x": x, "cycles": len(rho)}
        return {"x": x, "rho": np.pad(rho, (0, MAXITER - len(rho)))}
    if kind == "batch2d":
        xs, hs = s["solver"].solve(s["rhs"])
        flat = hs if case["nrhs"] == 1 else [h for hk in hs for h in hk]
        return {"x": xs, "cycles": np.array([len(h) for h in flat])}
    if kind == "gradient2d":
        theta = s["theta"].detach().requires_grad_(True)
        u = adjoint.solve(theta, s["f"], tol=case["tol"])
        loss = 0.5 * (u - s["obs"]).square().sum()
        loss.backward()
        return {"u": u.detach(), "grad": theta.grad}
    so, q, f, res, fac = s["so"], s["q"], s["f"], s["res"], s["fac"]
    q.zero_()
    for updown in (cdr2.DOWN, cdr2.UP):
        if case["relaxation"] == "point":
            cdr2.relax_gs(so, f, q, fac[0], updown)
        else:
            cdr2.relax_lines_xy(so, f, q, fac[0], fac[1], updown)
        if updown == cdr2.DOWN:
            cdr2.residual(so, f, q, res)
            cdr2.restrict(s["ci"], res, s["fc"])
            cdr2.interp_add(q, s["qc"], res, so, s["ci"])
    return {"q": q, "res": res, "fc": s["fc"]}


# ---- work -----------------------------------------------------------------------------------
def work(case):
    """One pass with every array of the hierarchy read once a cycle and every iterate written once
    a cycle, in the precision of the cycle, for the number of cycles such a problem takes; a
    hierarchy built in the pass reads its operator once and writes its levels once."""
    kind = case["kind"]
    if kind == "steps2d":
        n = case["nx"] * case["ny"]
        w = 8 if case["dtype"] == "f64" else 4
        planes = (5 if case["points"] == 9 else 3) + (1 if case["relaxation"] == "point" else 4)
        return {"bytes": n * w * (planes + 8 / 4 + 1 + 1 + 1 + 0.5), "flops": n * 80}
    if kind == "batch2d":
        pts = [n * n for n in _batch_sides(case)]
        m = case["nrhs"]
        return {"bytes": 14 * 4 / 3 * 4 * sum(p * (11 + 4 * m) for p in pts),
                "flops": 14 * 4 / 3 * 100 * m * sum(pts)}
    if kind == "gradient2d":
        p = case["nb"] * case["n"] ** 2
        return {"bytes": p * (4 / 3 * 8 * 11 + 20 * 4 / 3 * 4 * 15 + 24),
                "flops": p * (4 / 3 * 400 + 20 * 4 / 3 * 100)}
    w = 8 if case["precision"] == "f64" else 4
    line = case["relaxation"] != "point"
    if kind == "solve2d":
        p = case["nx"] * case["ny"]
        cycles = 15 if case["op"] == "diffusion" else 10
        planes = (3 if case["op"] == "poisson" else 5) + (4 if line else 1) + 2
        return {"bytes": p * 4 / 3 * (cycles * w * (planes + 4) + (8 * planes if case["new"] else 0)),
                "flops": p * 4 / 3 * (cycles * (100 if line else 60) + (400 if case["new"] else 0))}
    p = case["nx"] * case["ny"] * case["nz"]
    planes = 14 if case["op"] == "fe" else 4
    cycles = 25 if line else 10
    per = (planes + 1) + 5 + 14 / 8 + (13 if line else 0)
    return {"bytes": p * (cycles * w * per + (8 * (planes + 8) if case["new"] else 0)),
            "flops": p * cycles * (400 if line else 200)}


def tolerance(case):
    # A solve ends where its residual passes tol, after the same cycles whatever the order of its
    # sums, so its iterates differ by roundings that the remaining cycles damp, never by tol.
    if case["kind"] == "steps2d":
        return {"rel": 1e-11} if case["dtype"] == "f64" else {"rel": 1e-4}
    if case["kind"] in ("batch2d", "gradient2d") or case["precision"] == "mixed":
        return {"rel": 1e-8}
    return {"rel": 1e-10}


# ---- 64-bit values without the framework ------------------------------------------------------
def exact(case, seed):
    kind = case["kind"]
    if kind == "steps2d":
        return _exact_steps(case, seed)
    if kind in ("solve2d", "solve3d"):
        if case["op"] == "diffusion":
            if kind == "solve3d" or _direct_cost([(case["nx"], case["ny"])]) > 1:
                return None
            g = _gen(seed)
            so = _assemble64(_cells2(case["nx"], case["ny"], g).cpu().numpy()[0])
            b = _rhs(so.shape[1:], g).cpu().numpy()
            x = _direct(so, b[None])[0]
        else:
            x = _exact_separable(case, seed)
        return {"x": x, "rho" if case["precision"] == "f64" else "cycles": None}
    if kind == "batch2d":
        ns, m = _batch_sides(case), case["nrhs"]
        if _direct_cost([(n, n) for n in ns]) > 1:
            return None
        g = _gen(seed)
        ops = [_assemble64(_cells2(n, n, g).cpu().numpy()[0]) for n in ns]
        rhs = [_stack_rhs(m, (n + 2, n + 2), g).cpu().numpy() for n in ns]
        xs = [_direct(so, b) for so, b in zip(ops, rhs)]
        return {"x": [x if m > 1 else x[0] for x in xs], "cycles": None}
    nb, n = case["nb"], case["n"]
    if _direct_cost([(n, n)] * 2 * nb) > 1:
        return None
    s = prepare(case, seed)
    th, f, obs = (s[k].cpu().numpy() for k in ("theta", "f", "obs"))
    us, gs = [], []
    for t in range(nb):
        k = np.exp(th[t])
        so = _assemble64(k)
        u = _direct(so, f[t][None])[0]
        d = u - obs[t]
        d[0], d[-1], d[:, 0], d[:, -1] = 0, 0, 0, 0
        lam = _direct(so, d[None])[0]
        us.append(u)
        gs.append(-k * _element_form(u, lam))
    return {"u": np.stack(us), "grad": np.stack(gs)}


def _direct_cost(sides):
    """Cost of _direct over operators of these sides, 1 being about ten seconds."""
    return sum(max(a, b) * min(a, b) ** 3 for a, b in sides) / 7e10


def _assemble64(k):
    """Bilinear finite elements of -div(k grad u), planes c, w, s, sw, nw as the solver stores them."""
    ny, nx = k.shape[0] - 1, k.shape[1] - 1
    so = np.zeros((5, ny + 2, nx + 2))
    a, b, c, d = k[:-1, :-1], k[:-1, 1:], k[1:, :-1], k[1:, 1:]
    so[0, 1:-1, 1:-1] = 2 / 3 * (a + b + c + d)
    so[1, 1:-1, 2:-1] = ((a + c) / 6)[:, 1:]
    so[2, 2:-1, 1:-1] = ((a + b) / 6)[1:]
    so[3, 2:-1, 2:-1] = so[4, 2:-1, 2:-1] = (a / 3)[1:, 1:]
    return so


def _element_form(u, lam):
    """lam_e^T K u_e of every cell, K the bilinear element matrix of unit coefficient."""
    c = [(slice(0, -1), slice(0, -1)), (slice(0, -1), slice(1, None)),
         (slice(1, None), slice(1, None)), (slice(1, None), slice(0, -1))]
    out = 0
    for p in range(4):
        for q in range(4):
            w = 4 if p == q else -1 if (p - q) % 2 else -2
            out = out + w / 6 * lam[c[p]] * u[c[q]]
    return out


def _direct(so, b):
    """Block elimination along the longer side; b and the result (m, ny+2, nx+2)."""
    if so.shape[1] < so.shape[2]:  # lines along the shorter side: the transposed grid
        st = np.ascontiguousarray(so[[0, 2, 1, 3, 4]].transpose(0, 2, 1))
        return np.ascontiguousarray(_direct(st, b.transpose(0, 2, 1)).transpose(0, 2, 1))
    so = torch.as_tensor(np.ascontiguousarray(so))
    rhs = torch.as_tensor(np.ascontiguousarray(b[:, 1:-1, 1:-1].transpose(1, 2, 0)))  # (ny, nx, m)
    ny, nx = so.shape[1] - 2, so.shape[2] - 2
    c, w, s, sw, nw = (so[k] for k in range(5))

    def below(j, v):  # (coupling of row j to row j - 1) v, v indexed along row j - 1
        out = s[j, 1:-1, None] * v
        out[1:] += sw[j, 2:-1, None] * v[:-1]
        out[:-1] += nw[j, 2:-1, None] * v[1:]
        return out

    def above(j, v):  # its transpose: from row j to row j - 1
        out = s[j, 1:-1, None] * v
        out[:-1] += sw[j, 2:-1, None] * v[1:]
        out[1:] += nw[j, 2:-1, None] * v[:-1]
        return out

    inv = torch.empty((ny, nx, nx), dtype=torch.float64)
    y = torch.empty_like(rhs)
    for j in range(1, ny + 1):
        d = torch.diag(c[j, 1:-1]) - torch.diag(w[j, 2:-1], 1) - torch.diag(w[j, 2:-1], -1)
        r = rhs[j - 1]
        if j > 1:
            t = below(j, inv[j - 2])
            d -= below(j, t.T.contiguous())
            r = r + below(j, y[j - 2])
        inv[j - 1] = torch.cholesky_inverse(torch.linalg.cholesky(0.5 * (d + d.T)))
        y[j - 1] = inv[j - 1] @ r
    x = torch.zeros((ny + 2, nx + 2, rhs.shape[2]), dtype=torch.float64)
    x[ny, 1:-1] = y[ny - 1]
    for j in range(ny, 1, -1):
        x[j - 1, 1:-1] = y[j - 2] + inv[j - 2] @ above(j, x[j, 1:-1])
    return x.permute(2, 0, 1).contiguous().numpy()


def _exact_separable(case, seed):
    """Constant stencils: eigenvectors of the one-dimensional second differences per direction."""
    g = _gen(seed)
    n = [case[k] for k in ("nx", "ny", "nz") if k in case]
    per = case.get("periodic", "")
    b = _rhs(tuple(m + 2 for m in reversed(n)), g, per)
    v = b[(slice(1, -1),) * len(n)].clone()
    mu, q = [], []
    for k, m in enumerate(n):
        e = torch.diag(torch.ones(m - 1, dtype=torch.float64), 1)
        e = e + e.T
        if "xyz"[k] in per:
            e[0, -1] = e[-1, 0] = 1.0
        lam, vec = torch.linalg.eigh(e)
        mu.append(lam.cuda())
        q.append(vec.cuda())
    dims = len(n)

    def apply(v, transpose):
        for k in range(dims):
            d = dims - 1 - k  # tensor dimension of direction k
            m = q[k].T if transpose else q[k]
            v = torch.movedim(torch.tensordot(m.contiguous(), v, ([1], [d])), 0, d)
        return v.contiguous()

    shape = lambda k: [-1 if d == dims - 1 - k else 1 for d in range(dims)]  # noqa: E731
    if case["op"] == "fe":  # 3^d - (product of 1 + neighbours)
        lam = torch.ones(1, dtype=torch.float64, device="cuda")
        for k in range(dims):
            lam = lam * (1 + mu[k]).reshape(shape(k))
        lam = 3.0 ** dims - lam
    else:
        h = [1.0 / (m + ("xyz"[k] not in per)) for k, m in enumerate(n)]
        lam = 0.0
        for k in range(dims):
            lam = lam + math.prod(h) / h[k] ** 2 * (2 - mu[k]).reshape(shape(k))
    x = torch.zeros_like(b)
    x[(slice(1, -1),) * dims] = apply(apply(v, True) / lam, False)
    if "x" in per:
        x[:, 0], x[:, -1] = x[:, -2].clone(), x[:, 1].clone()
    return x


def _exact_steps(case, seed):
    """The calls of run() in 64 bits, on the inputs as the precision of the case holds them."""
    s = {k: (v.double() if torch.is_tensor(v) else v) for k, v in prepare(case, seed).items()}
    so, f, fac, ci, qc = s["so"], s["f"], s["fac"], s["ci"], s["qc"]
    nine = case["points"] == 9
    q, res, fc = torch.zeros_like(f), torch.zeros_like(f), torch.zeros_like(qc)
    nx, ny = case["nx"], case["ny"]

    def off(q):  # f + the couplings to the neighbours, on the interior
        I, J = slice(1, -1), slice(1, -1)
        up, lo = slice(2, None), slice(0, -2)
        r = f[J, I] + so[1][J, I] * q[J, lo] + so[1][J, up] * q[J, up]
        r = r + so[2][J, I] * q[lo, I] + so[2][up, I] * q[up, I]
        if nine:
            r = r + so[3][J, I] * q[lo, lo] + so[4][J, up] * q[lo, up]
            r = r + so[4][up, I] * q[up, lo] + so[3][up, up] * q[up, up]
        return r

    j = torch.arange(1, ny + 1, device="cuda")[:, None]
    i = torch.arange(1, nx + 1, device="cuda")[None]

    def point(up):
        if nine:
            order = [(1, 1), (0, 1), (1, 0), (0, 0)]
            colours = [(i % 2 == a) & (j % 2 == b) for a, b in order]
        else:
            colours = [(i + j) % 2 == c for c in (0, 1)]
        for m in (reversed(colours) if up else colours):
            v = q[1:-1, 1:-1]
            q[1:-1, 1:-1] = torch.where(m, off(q) * fac[0][1][1:-1, 1:-1], v)

    def lines(d, up):
        for first in ((1, 2) if up else (2, 1)):
            # the couplings along the line are solved for, the others go to the right-hand side
            keep = so[1].clone(), so[2].clone()
            so[1 if d == "x" else 2] = 0
            r = off(q)
            so[1], so[2] = keep
            dia, cpl = so[0][1:-1, 1:-1], so[1 if d == "x" else 2][1:-1, 1:-1]
            if d == "y":
                r, dia, cpl = r.T, dia.T, cpl.T
            r, dia, cpl = r[first - 1::2], dia[first - 1::2], cpl[first - 1::2]
            n = r.shape[1]
            p, y = [dia[:, 0]], [r[:, 0]]
            for k in range(1, n):
                m = cpl[:, k] / p[-1]
                p.append(dia[:, k] - m * cpl[:, k])
                y.append(r[:, k] + m * y[-1])
            x = [y[-1] / p[-1]]
            for k in range(n - 2, -1, -1):
                x.append((y[k] + cpl[:, k + 1] * x[-1]) / p[k])
            x = torch.stack(x[::-1], 1)
            if d == "x":
                q[1:-1, 1:-1][first - 1::2] = x
            else:
                q[1:-1, 1:-1].T[first - 1::2] = x

    def smooth(up):
        if case["relaxation"] == "point":
            point(up)
        else:
            for d in ("yx" if up else "xy"):
                lines(d, up)

    smooth(False)
    res[1:-1, 1:-1] = off(q) - so[0][1:-1, 1:-1] * q[1:-1, 1:-1]
    # interpolation planes {L, R, A, B, SW, NW, NE, SE} on the coarse grid; coarse (jc, ic) lies at
    # fine (2 jc - 1, 2 ic - 1)
    L, R, A, B, SW, NW, NE, SE = ci
    jc, ic = fc.shape[0] - 2, fc.shape[1] - 2
    pad = torch.zeros((2 * jc + 3, 2 * ic + 3), dtype=torch.float64, device="cuda")
    pad[:res.shape[0], :res.shape[1]] = res[:pad.shape[0], :pad.shape[1]]
    pad[ny + 1:], pad[:, nx + 1:] = 0, 0

    def at(dj, di):
        return pad[1 + dj:1 + dj + 2 * jc:2, 1 + di:1 + di + 2 * ic:2]

    J, I, Jn, In = slice(1, jc + 1), slice(1, ic + 1), slice(2, jc + 2), slice(2, ic + 2)
    fc[J, I] = (NE[J, I] * at(-1, -1) + A[J, I] * at(-1, 0) + NW[J, In] * at(-1, 1)
                + R[J, I] * at(0, -1) + at(0, 0) + L[J, In] * at(0, 1)
                + SE[Jn, I] * at(1, -1) + B[Jn, I] * at(1, 0) + SW[Jn, In] * at(1, 1))
    # interpolation: coarse points, edges and cells, the fine residual over the diagonal added off
    # the coarse points
    q2 = q.clone()
    corr = torch.zeros((2 * jc + 3, 2 * ic + 3), dtype=torch.float64, device="cuda")
    J, I = slice(1, jc + 1), slice(1, ic + 1)
    corr[1:2 * jc:2, 1:2 * ic:2] = qc[J, I]
    Jm, Im = slice(1, jc + 1), slice(2, ic + 2)
    corr[1:2 * jc:2, 2:2 * ic + 1:2] = L[J, Im] * qc[J, I] + R[J, Im] * qc[J, Im]
    Jp = slice(2, jc + 2)
    corr[2:2 * jc + 1:2, 1:2 * ic:2] = A[Jp, I] * qc[Jp, I] + B[Jp, I] * qc[J, I]
    corr[2:2 * jc + 1:2, 2:2 * ic + 1:2] = (SW[Jp, Im] * qc[J, I] + NW[Jp, Im] * qc[Jp, I]
                                            + NE[Jp, Im] * qc[Jp, Im] + SE[Jp, Im] * qc[J, Im])
    off_c = (i % 2 == 0) | (j % 2 == 0)
    own = torch.where(off_c, res[1:-1, 1:-1] / so[0][1:-1, 1:-1], torch.zeros_like(f[1:-1, 1:-1]))
    q2[1:-1, 1:-1] += corr[1:ny + 1, 1:nx + 1] + own
    q = q2
    smooth(True)
    return {"q": q, "res": res, "fc": fc}
