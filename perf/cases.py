"""Workloads of the solve path, as the programs that use it run them.

Every case goes through the public entry points of pascal_poisson_fft_amd.api
on device buffers.  The kinds:

  solve    FFTPoisson.solve in FP64 (plan kept, one right-hand side a pass).
           tuned = the plan was tuned when it was made, as a long-running
           program does; otherwise the plan is used as created, as the Fortran
           module does (plan_create, initial, then solves).
  ir       FFTPoisson.solve of an FP32_IR plan: FP32 passes refined to a
           relative FP64 residual of 1e-10.
  noalloc  api.solve_noalloc: no plan, the workspace is static.
  batch    Batch.solve: many problems of uneven shapes, one hipGraph.
  tdma     TDMAPlanMany.solve / solve_cycle: the stand-alone batched Thomas,
           whose coefficient arrays the caller refills for every solve.

Boundary conditions of x and y are N (Neumann, DCT) or P (periodic, FFT); z
has Neumann walls and is uniform or tanh-stretched (gamma > 0).
"""
import math
import random

import torch

from pascal_poisson_fft_amd import api
from pascal_poisson_fft_amd.grid import make_axis

# x and y extents that the plans take
SIZES = [n for n in sorted({2 ** a * m for a in range(11) for m in (1, 3, 5, 7, 15)}) if 8 <= n <= 1024 and n % 2 == 0]
BATCH_SIZES = [32, 48, 64, 96, 128, 192, 256]


def listed():
    return [
        # the smallest ordinary calls, where launches and latency count: the
        # 64^3 manufactured problem of the reference's example, and a ragged
        # problem for a caller that may not allocate
        {"name": "solve_64cube_PP", "kind": "solve", "nx": 64, "ny": 64, "nz": 64, "bc": "PP", "gamma": 0.0, "tuned": False},
        {"name": "noalloc_60x48x50_PN", "kind": "noalloc", "nx": 60, "ny": 48, "nz": 50, "bc": "PN", "gamma": 1.4},
        # an ordinary single problem with ragged extents, plan as created
        {"name": "solve_320x224x200_NP", "kind": "solve", "nx": 320, "ny": 224, "nz": 200, "bc": "NP", "gamma": 1.2, "tuned": False},
        # a narrow, tall column: the longest z lines, few of them
        {"name": "solve_96x80x2050_NN", "kind": "solve", "nx": 96, "ny": 80, "nz": 2050, "bc": "NN", "gamma": 1.5, "tuned": False},
        # the headline problem, and the time-stepping (projection) problem,
        # the largest: a channel periodic in x with walls in y and z
        {"name": "solve_512cube_NN", "kind": "solve", "nx": 512, "ny": 512, "nz": 512, "bc": "NN", "gamma": 1.5, "tuned": True},
        {"name": "solve_1024x1024x768_PN", "kind": "solve", "nx": 1024, "ny": 1024, "nz": 768, "bc": "PN", "gamma": 1.8, "tuned": True},
        # FP32 storage with FP64 refinement to 1e-10: ordinary and headline
        {"name": "ir_112x96x130_PP", "kind": "ir", "nx": 112, "ny": 96, "nz": 130, "bc": "PP", "gamma": 1.5, "tuned": False},
        {"name": "ir_512cube_NN", "kind": "ir", "nx": 512, "ny": 512, "nz": 512, "bc": "NN", "gamma": 1.5, "tuned": True},
        # many independent problems of uneven shapes in one call: the FP64
        # batch, and a smaller one whose problems mix FP64 and FP32_IR
        {"name": "batch_96_fp64", "kind": "batch", "problems": 96, "shapes": 4, "mixed": False},
        {"name": "batch_24_mixed", "kind": "batch", "problems": 24, "shapes": 11, "mixed": True},
        # the stand-alone Thomas: one system per (x, y) column of a field, and
        # the cyclic form on a smaller ragged field
        {"name": "tdma_256x256x256", "kind": "tdma", "nx": 256, "ny": 256, "nz": 256, "cyclic": False},
        {"name": "tdma_cyclic_100x60x90", "kind": "tdma", "nx": 100, "ny": 60, "nz": 90, "cyclic": True},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _near(v):
    return min(SIZES, key=lambda n: abs(math.log(n / v)))


def draw(rng):
    """One more case: extents log-uniform over what the entry point takes."""
    kind = rng.choice(["solve", "solve", "solve", "ir", "noalloc", "batch", "tdma"])
    if kind == "batch":
        return {"kind": kind, "problems": rng.randint(4, 48), "shapes": rng.randrange(1000, 1 << 20),
                "mixed": rng.random() < 0.5}
    if kind == "tdma":
        while True:
            nx, ny, nz = (int(_log(rng, 12, 700)) for _ in range(3))
            if nx * ny * nz <= 2 ** 26:
                return {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "cyclic": rng.random() < 0.4}
    while True:
        nx, ny = _near(_log(rng, 16, 1024)), _near(_log(rng, 16, 1024))
        nz = 2 * int(_log(rng, 8, 512 if rng.random() < 0.85 else 1536))
        if nx * ny * nz <= (2 * 10 ** 6 if kind == "noalloc" else 2 ** 27):
            break
    case = {"kind": kind, "nx": nx, "ny": ny, "nz": nz, "bc": rng.choice("NP") + rng.choice("NP"),
            "gamma": rng.choice([0.0, round(rng.uniform(1.0, 2.0), 2)])}
    if kind != "noalloc":
        case["tuned"] = rng.random() < 0.4
    return case


# ---- inputs -----------------------------------------------------------------


class _Buffer:
    """A device buffer as the entry points take it: an object with .ptr."""

    def __init__(self, t):
        self.t, self.ptr = t, t.data_ptr()


class _Problem:
    """Inputs and solution buffer of one problem."""


def _dev(a):
    return torch.from_numpy(a).cuda()


def _box(f, axis, periodic):
    """3-point mean along an axis, mirrored at walls."""
    m, p = torch.roll(f, 1, axis), torch.roll(f, -1, axis)
    if not periodic:
        n = f.shape[axis]
        m.narrow(axis, 0, 1).copy_(f.narrow(axis, 0, 1))
        p.narrow(axis, n - 1, 1).copy_(f.narrow(axis, n - 1, 1))
    m += f
    m += p
    return m.div_(3.0)


def _axes(nx, ny, nz, bc, gamma, L):
    return (make_axis(nx, L, bc[0] == "P"), make_axis(ny, L, bc[1] == "P"),
            make_axis(nz, L, False, uniform=gamma == 0, gamma=gamma))


def _rhs(nx, ny, nz, bc, az, gen):
    """Smoothed N(0,1) field whose volume-weighted mean is zero, so that the
    zero-flux problem has a solution."""
    f = torch.randn((nz, ny, nx), dtype=torch.float64, device="cuda", generator=gen)
    f = _box(f, 2, bc[0] == "P")
    f = _box(f, 1, bc[1] == "P")
    f = _box(f, 0, False)
    w = _dev(az.dx[1:nz + 1].copy())
    f -= (f.sum((1, 2)) * w).sum() / (w.sum() * nx * ny)
    return f


def _problem(nx, ny, nz, bc, gamma, L, gen, out=None):
    ax, ay, az = _axes(nx, ny, nz, bc, gamma, L)
    q = _Problem()
    if out is None:
        out = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.float64, device="cuda")
    q.rhs, q.p = _Buffer(_rhs(nx, ny, nz, bc, az, gen)), _Buffer(out)
    q.dmx1, q.dmx2, q.dmx3, q.dx3 = (_Buffer(_dev(a)) for a in (ax.dmx, ay.dmx, az.dmx, az.dx))
    q.args = (q.rhs, q.p, q.dmx1, q.dmx2, q.dmx3, q.dx3)
    return q


def _shapes(case):
    """The problems of a batch: extents, boundaries and stretching."""
    rng = random.Random(case["shapes"])
    got = []
    for i in range(case["problems"]):
        gamma = 0.0 if rng.random() < 0.5 else rng.uniform(1.0, 2.0)
        got.append({"nx": rng.choice(BATCH_SIZES), "ny": rng.choice(BATCH_SIZES), "nz": 2 * rng.randint(16, 192),
                    "bc": "PP" if i < case["problems"] // 2 else "NN", "gamma": gamma,
                    "fp32": case["mixed"] and i % 2 == 1})
    return got


def _padded(d):
    """Doubles of one problem's P inside the batch's buffer (256-byte steps)."""
    return -(-(d["nx"] + 2) * (d["ny"] + 2) * (d["nz"] + 2) // 32) * 32


def _tdma_arrays(case, gen):
    shape = (case["nz"], case["ny"], case["nx"])
    u = [torch.rand(shape, dtype=torch.float64, device="cuda", generator=gen) for _ in range(4)]
    a, c, d = -0.5 - u[0], -0.5 - u[1], u[3] - 0.5
    return a, 0.5 + u[2] - a - c, c, d  # diagonally dominant, as the z rows are


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    s = {"case": case}
    if kind == "tdma":
        a, b, c0, d0 = _tdma_arrays(case, gen)
        s["a"], s["b"], s["c"], s["d"] = (_Buffer(t) for t in (a, b, torch.empty_like(c0), torch.empty_like(d0)))
        s["c0"], s["d0"] = c0, d0
        s["plan"] = api.TDMAPlanMany(case["nx"], case["ny"], case["nz"])
        return s
    if kind == "batch":
        shapes = _shapes(case)
        flat = s["out"] = torch.zeros(sum(_padded(d) for d in shapes), dtype=torch.float64, device="cuda")
        s["problems"], at = [], 0
        for d in shapes:
            q = _problem(d["nx"], d["ny"], d["nz"], d["bc"], d["gamma"], 1.0, gen, out=flat[at:])
            s["problems"].append((dict(n1m=d["nx"], n2m=d["ny"], n3m=d["nz"], L=(1.0, 1.0, 1.0),
                                       pbc=(d["bc"][0] == "P", d["bc"][1] == "P", False), tol=1e-10,
                                       precision=api.PPF_PREC_FP32_IR if d["fp32"] else api.PPF_PREC_FP64), q))
            at += _padded(d)
        s["batch"] = api.Batch(s["problems"])
        return s
    s["q"] = q = _problem(case["nx"], case["ny"], case["nz"], case["bc"], case["gamma"], 2.0, gen)
    s["pbc"] = (case["bc"][0] == "P", case["bc"][1] == "P", False)
    if kind != "noalloc":
        s["plan"] = api.FFTPoisson(case["nx"], case["ny"], case["nz"], (2.0, 2.0, 2.0), s["pbc"], tol=1e-10,
                                   precision=api.PPF_PREC_FP32_IR if kind == "ir" else api.PPF_PREC_FP64)
        if case["tuned"]:
            s["plan"].tune(*q.args)
    return s


def run(s):
    kind = s["case"]["kind"]
    if kind == "tdma":
        # c and d are overwritten by a solve: the caller fills them each time
        s["c"].t.copy_(s["c0"])
        s["d"].t.copy_(s["d0"])
        args = (s["a"], s["b"], s["c"], s["d"])
        if s["case"]["cyclic"]:
            s["plan"].solve_cycle(*args)
        else:
            s["plan"].solve(*args)
        return s["d"].t
    if kind == "batch":
        s["batch"].solve()
        return s["out"]
    if kind == "noalloc":
        c = s["case"]
        api.solve_noalloc(c["nx"], c["ny"], c["nz"], (2.0, 2.0, 2.0), s["pbc"], *s["q"].args)
    else:
        s["plan"].solve(*s["q"].args)
    return s["q"].p.t


# ---- what a pass cannot do without -------------------------------------------


def _solve_work(nx, ny, nz):
    """The right-hand side read once, the ghosted solution written once; line
    transforms (5 n/2 log2 n for a real line) both ways and the z solves."""
    n = nx * ny * nz
    return {"bytes": 8 * (n + (nx + 2) * (ny + 2) * (nz + 2)), "flops": n * (5 * math.log2(nx * ny) + 14)}


def work(case):
    if case["kind"] == "tdma":
        n = case["nx"] * case["ny"] * case["nz"]
        # refill (c, d read and written), then a, b, c, d read, c, d written
        return {"bytes": 8 * n * (4 + 6), "flops": n * (15 if case["cyclic"] else 9)}
    if case["kind"] == "batch":
        w = [_solve_work(d["nx"], d["ny"], d["nz"]) for d in _shapes(case)]
        return {k: sum(v[k] for v in w) for k in ("bytes", "flops")}
    return _solve_work(case["nx"], case["ny"], case["nz"])


def tolerance(case):
    if case["kind"] == "tdma":
        return "exact"  # the operation order is part of the entry point's contract
    # measured against exact(): 2e-11 for FP32_IR (it stops at a relative
    # residual of 1e-10), 6e-13 for FP64 (lines over 1024 rows in z are worse
    # conditioned: the FP64 tests allow 1e-11 there)
    if case["kind"] == "ir" or case.get("mixed"):
        return {"rel": 1e-10}
    return {"rel": 1e-11} if case.get("nz", 0) > 1024 else {"rel": 3e-12}


# ---- the answers in 64 bits, by torch alone ------------------------------------


def _along(v, axis, shape=3):
    return v.reshape([-1 if k == axis else 1 for k in range(shape)])


def _dct(f, axis, inverse):
    """Unnormalised DCT-II along an axis, or its inverse, through an FFT of the
    even samples followed by the odd ones backwards."""
    n = f.shape[axis]
    k = torch.arange(n, device=f.device)
    order = torch.cat([torch.arange(0, n, 2, device=f.device), torch.arange(n - 1, 0, -2, device=f.device)])
    q = _along(torch.exp(-0.5j * math.pi * k.double() / n), axis)
    if not inverse:
        v = torch.fft.fft(f.index_select(axis, order), dim=axis) * q
        if not f.is_complex():
            return v.real * 2.0
        m = torch.fft.fft(f.index_select(axis, order).conj().resolve_conj(), dim=axis) * q
        return v + m.conj()
    back = torch.roll(torch.flip(f, (axis,)), 1, axis)
    back.narrow(axis, 0, 1).zero_()
    v = torch.fft.ifft((f - 1j * back) * q.conj() * 0.5, dim=axis)
    v = v if f.is_complex() else v.real
    out = torch.empty_like(v)
    out.index_copy_(axis, order, v)
    return out


def _eigenvalues(n, h, periodic):
    k = torch.arange(n, dtype=torch.float64, device="cuda")
    s = torch.sin(k * (math.pi / n) * (1.0 if periodic else 0.5))
    return 4.0 * s * s / (h * h)


def _solution(f, nx, ny, nz, bc, gamma, L):
    """The ghosted solution of the 7-point problem, zero mean."""
    ax, ay, az = _axes(nx, ny, nz, bc, gamma, L)
    for axis, p in ((2, bc[0]), (1, bc[1])):
        f = torch.fft.fft(f, dim=axis) if p == "P" else _dct(f, axis, False)
    lam = _eigenvalues(ny, L / ny, bc[1] == "P")[:, None] + _eigenvalues(nx, L / nx, bc[0] == "P")[None, :]
    dx, dmx = az.dx, az.dmx
    am = [0.0] + [1.0 / dx[k] / dmx[k] for k in range(2, nz + 1)]
    ap = [1.0 / dx[k] / dmx[k + 1] for k in range(1, nz)] + [0.0]
    # Thomas along z; the (0,0) mode's first row is x = 0
    e = torch.empty((nz, ny, nx), dtype=torch.float64, device=f.device)
    b = -am[0] - ap[0] - lam
    b[0, 0] = 1.0
    f[0, 0, 0] = 0.0
    e[0] = ap[0] / b
    e[0, 0, 0] = 0.0
    f[0] /= b
    for k in range(1, nz):
        r = 1.0 / (-am[k] - ap[k] - lam - am[k] * e[k - 1])
        f[k] = (f[k] - am[k] * f[k - 1]) * r
        e[k] = ap[k] * r
    for k in range(nz - 2, -1, -1):
        f[k] -= e[k] * f[k + 1]
    del e
    for axis, p in ((1, bc[1]), (2, bc[0])):
        f = torch.fft.ifft(f, dim=axis) if p == "P" else _dct(f, axis, True)
    f = f.real if f.is_complex() else f
    out = torch.zeros((nz + 2, ny + 2, nx + 2), dtype=torch.float64, device=f.device)
    out[1:-1, 1:-1, 1:-1] = f - f.mean()
    # ghost layers: wall extrapolation along x, y, z, then the periodic wraps
    for wrap in (False, True):
        for axis, a in ((2, ax), (1, ay), (0, az)):
            if a.pbc != wrap:
                continue
            at = lambda i: out.narrow(axis, i, 1)  # noqa: E731
            n, d = a.nm, a.dmx
            if wrap:
                at(0).copy_(at(n))
                at(n + 1).copy_(at(1))
                continue
            for ghost, one, two, p, q in ((0, 1, 2, d[1], d[2]), (n + 1, n, n - 1, d[n + 1], d[n])):
                s = (p + q) ** 2
                at(ghost).copy_((s * at(one) - p * p * at(two)) / (s - p * p))
    return out


def _thomas(a, b, c, d, cyclic):
    """Systems along the first axis; cyclic ones as a rank-one correction."""
    n = d.shape[0]
    if cyclic:
        g = -b[0]
        b = b.clone()
        u = torch.zeros_like(d)
        u[0], u[-1] = g, c[-1]
        corner = a[0]
        b[0] = b[0] - g
        b[-1] = b[-1] - c[-1] * corner / g
        x, y = _thomas(a, b, c, d, False), _thomas(a, b, c, u, False)
        return x - y * ((x[0] + corner * x[-1] / g) / (1.0 + y[0] + corner * y[-1] / g))
    e, x = torch.empty_like(d), d.clone()
    e[0] = c[0] / b[0]
    x[0] = d[0] / b[0]
    for k in range(1, n):
        r = 1.0 / (b[k] - a[k] * e[k - 1])
        e[k] = c[k] * r
        x[k] = (x[k] - a[k] * x[k - 1]) * r
    for k in range(n - 2, -1, -1):
        x[k] -= e[k] * x[k + 1]
    return x


def exact(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(int(seed))
    kind = case["kind"]
    if kind == "tdma":
        return _thomas(*_tdma_arrays(case, gen), case["cyclic"])
    if kind == "batch":
        shapes = _shapes(case)
        flat, at = torch.zeros(sum(_padded(d) for d in shapes), dtype=torch.float64, device="cuda"), 0
        for d in shapes:
            az = _axes(d["nx"], d["ny"], d["nz"], d["bc"], d["gamma"], 1.0)[2]
            p = _solution(_rhs(d["nx"], d["ny"], d["nz"], d["bc"], az, gen), d["nx"], d["ny"], d["nz"], d["bc"],
                          d["gamma"], 1.0)
            flat[at:at + p.numel()] = p.reshape(-1)
            at += _padded(d)
        return flat
    az = _axes(case["nx"], case["ny"], case["nz"], case["bc"], case["gamma"], 2.0)[2]
    return _solution(_rhs(case["nx"], case["ny"], case["nz"], case["bc"], az, gen), case["nx"], case["ny"], case["nz"],
                     case["bc"], case["gamma"], 2.0)
