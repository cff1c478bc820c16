"""The work that programs have this framework do, as cases that can be timed.

A case is a plain dict: what is called (``kind``), the grid, and the options.
``prepare`` builds what a program holds before the call (context, fields on
the GPU), ``run`` is one pass through the public entry points of
``x3div_amd``, ``exact`` gives the same outputs in 64 bits from torch's FFTs
and dense solves, without the framework: with periodic boundaries every
compact operator is a circulant, so it is its symbol in Fourier space.

Kinds
  step       one Euler step (``X3D.step``), eager or as a captured HIP graph
  pieces     the step as the reference-shaped driver calls it: momentum right-
             hand side, Euler update, solve_poisson, velocity correction
  step_f32   one step of the FP32 form from a snapshot
  step_bfp   one step of the BFP32 form: FP64 fields encoded, stepped, decoded
  batch      one step of a batch of uneven grids, captured in a HIP graph
  ops        the periodic operators one by one, FP64, FP32 or on the matrix cores
  np         the non-periodic first derivatives, lines of any length
"""
import math

import numpy as np
import torch

from x3div_amd import X3D, X3DBatch

TWO_PI = 2.0 * math.pi
# a time step well inside the explicit Euler limit of the grids below
GDT = 5.0e-4
OPS = ["derx", "dery", "derz", "derxvp", "deryvp", "derzvp", "derxpv", "derypv", "derzpv",
       "intxvp", "intyvp", "intzvp", "intxpv", "intypv", "intzpv", "derxx", "deryy", "derzz"]
# line lengths that the periodic line kernels tile
LENGTHS = [16, 24, 32, 40, 48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512]
# dimensions of the batching form's grids
BATCH_SIZES = [32, 48, 64, 96, 128, 160]
# largest grid of a drawn case, in points
MOST = 512 ** 3


def listed():
    return [
        # the configuration of the reference's own test: a single small grid,
        # called eagerly, where launches and host work count
        {"name": "step_64", "kind": "step", "nx": 64, "ny": 64, "nz": 64, "graph": False, "stretch": False},
        # a mid-size cube stepped through its captured graph
        {"name": "step_256_graph", "kind": "step", "nx": 256, "ny": 256, "nz": 256, "graph": True, "stretch": False},
        # the headline size
        {"name": "step_512", "kind": "step", "nx": 512, "ny": 512, "nz": 512, "graph": False, "stretch": False},
        # a non-cubic grid with 3- and 5-smooth lengths and stretched y, driven
        # through the reference's four calls per step
        {"name": "pieces_320x96x160", "kind": "pieces", "nx": 320, "ny": 96, "nz": 160, "stretch": True},
        # a large single grid of the FP32 form (768-point lines, 1.6 GB a field)
        {"name": "step_f32_1024x768x512", "kind": "step_f32", "nx": 1024, "ny": 768, "nz": 512},
        # FP32 at the headline size
        {"name": "step_f32_512", "kind": "step_f32", "nx": 512, "ny": 512, "nz": 512},
        # block floating point at the headline size
        {"name": "step_bfp_512", "kind": "step_bfp", "nx": 512, "ny": 512, "nz": 512},
        # 96 independent uneven grids, both precisions
        {"name": "batch96_f64", "kind": "batch", "precision": 8, "ngrids": 96, "dims_seed": 2024},
        {"name": "batch96_f32", "kind": "batch", "precision": 4, "ngrids": 96, "dims_seed": 2024},
        # single operators as a program with its own step calls them
        {"name": "ops_f64_512", "kind": "ops", "form": "f64", "nx": 512, "ny": 512, "nz": 512},
        # the dense-circulant variant on the matrix cores
        {"name": "ops_mfma_512", "kind": "ops", "form": "mfma", "nx": 512, "ny": 512, "nz": 512},
        # wall-bounded grids have 2^k + 1 points per direction
        {"name": "np_513x257x129", "kind": "np", "nx": 513, "ny": 257, "nz": 129, "first": 2, "last": 2},
    ]


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["step", "step", "pieces", "step_f32", "step_bfp", "batch", "ops", "ops", "np"])
    if kind == "batch":
        return {"kind": "batch", "precision": rng.choice([8, 4]), "ngrids": int(round(math.exp(rng.uniform(0, math.log(96))))),
                "dims_seed": rng.randrange(1 << 20)}
    if kind == "np":
        n = [int(round(math.exp(rng.uniform(math.log(17), math.log(513))))) for _ in range(3)]
        first, last = rng.choice([(1, 1), (1, 2), (2, 1), (2, 2)])
        return {"kind": "np", "nx": n[0], "ny": n[1], "nz": n[2], "first": first, "last": last}
    form = rng.choice(["f64", "f32", "mfma", "bfp"]) if kind == "ops" else ""
    while True:
        nx, ny, nz = (rng.choice([128, 256, 384, 512] if form == "mfma" else LENGTHS) for _ in range(3))
        bfp = kind == "step_bfp" or form == "bfp"
        if nx * ny * nz <= MOST and not (bfp and nx % 16):
            break
    case = {"kind": kind, "nx": nx, "ny": ny, "nz": nz}
    if kind == "ops":
        case["form"] = form
    if kind == "step":
        case["graph"] = rng.random() < 0.5
    if kind in ("step", "pieces"):
        case["stretch"] = rng.random() < 0.25
    return case


# ---- inputs ------------------------------------------------------------------
def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _lengths(case):
    """Unequal box lengths, so that the three directions differ."""
    return (TWO_PI, TWO_PI * 0.75, TWO_PI * 1.25)


def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _phase(n, k, shape):
    return (TWO_PI * k / n * torch.arange(n, dtype=torch.float64, device="cuda")).reshape(shape)


def _smooth(dims, seed, modes=8):
    """Sum of seeded Fourier modes with wavenumbers up to 4, amplitude 1/8 each."""
    nx, ny, nz = dims
    rng = np.random.default_rng(seed)
    out = torch.zeros((nz, ny, nx), dtype=torch.float64, device="cuda")
    for _ in range(modes):
        kx, ky, kz = (int(v) for v in rng.integers(-4, 5, 3))
        if not (kx or ky or kz):
            kx = 1
        p = float(rng.uniform(0, TWO_PI))
        a = _phase(nx, kx, (1, 1, nx)) + _phase(ny, ky, (1, ny, 1)) + p
        b = _phase(nz, kz, (nz, 1, 1))
        # sin(a + b) from the plane and the line
        out += 0.125 * (torch.cos(b) * torch.sin(a) + torch.sin(b) * torch.cos(a))
    return out


def _velocity(case, seed):
    """Taylor-Green plus 1e-3 uniform noise for the FP64 steps; for the 32-bit
    forms uniform random fields, which hold all wavenumbers alike (on smooth
    fields an FP32 pressure gradient is the difference of nearly equal values)."""
    dims = _dims(case)
    if case["kind"] in ("step", "pieces"):
        nx, ny, nz = dims
        x, y, z = _phase(nx, 1, (1, 1, nx)), _phase(ny, 1, (1, ny, 1)), _phase(nz, 1, (nz, 1, 1))
        u = [torch.sin(x) * torch.cos(y) * torch.cos(z), -torch.cos(x) * torch.sin(y) * torch.cos(z),
             torch.zeros((nz, ny, nx), dtype=torch.float64, device="cuda")]
        g = _generator(seed)
        return [c + 1e-3 * (2.0 * torch.rand((nz, ny, nx), dtype=torch.float64, device="cuda", generator=g) - 1.0)
                for c in u]
    return _random3(dims[0] * dims[1] * dims[2], seed, (dims[2], dims[1], dims[0]))


def _random3(count, seed, shape):
    """Three uniform random components in [-1, 1)."""
    g = _generator(seed)
    return [(2.0 * torch.rand(count, dtype=torch.float64, device="cuda", generator=g) - 1.0).reshape(shape)
            for _ in range(3)]


def _scalar(case, seed):
    """One field for the single operators: smooth plus a little noise."""
    nx, ny, nz = _dims(case)
    noise = torch.rand((nz, ny, nx), dtype=torch.float64, device="cuda", generator=_generator(seed))
    return _smooth((nx, ny, nz), [seed, 7]) + 1e-3 * (2.0 * noise - 1.0)


def _stretching(case):
    """Vectors of a mildly stretched y grid: ppy at the points, ppyi between them."""
    if not case.get("stretch"):
        return None
    t = np.arange(case["ny"]) * (TWO_PI / case["ny"])
    h = 0.5 * TWO_PI / case["ny"]
    return 1.0 / (1.0 + 0.3 * np.cos(t)), 1.0 / (1.0 + 0.3 * np.cos(t + h))


def _batch_dims(case):
    rng = np.random.default_rng(case["dims_seed"])
    return [tuple(int(v) for v in rng.choice(BATCH_SIZES, 3)) for _ in range(case["ngrids"])]


class _Device:
    """A run of the batch's device memory for torch; keeps the batch alive."""

    def __init__(self, owner, ptr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr, "data": (ptr, False), "version": 2}


def _batch_fields(b, dims, precision):
    """Each field of the batch as one tensor over all grids, grid after grid."""
    sizes = [nx * ny * nz for nx, ny, nz in dims]
    out = []
    for name in b.FIELDS:
        ptr = [b._ptr(i, name).value for i in range(len(dims))]
        for i in range(1, len(dims)):
            if ptr[i] != ptr[i - 1] + precision * sizes[i - 1]:
                raise RuntimeError("the batch's grids do not follow each other in memory")
        out.append(torch.as_tensor(_Device(b, ptr[0], sum(sizes), "<f%d" % precision), device="cuda"))
    return out


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "batch":
        dims, prec = _batch_dims(case), case["precision"]
        b = X3DBatch(dims, precision=prec)
        f = _batch_fields(b, dims, prec)
        dt = torch.float64 if prec == 8 else torch.float32
        s["u0"] = [a.to(dt) for a in _random3(f[0].numel(), seed, (-1,))]
        for a in f[3:]:
            a.zero_()
        b.graph_capture(gdt=GDT)
        return {**s, "b": b, "f": f}
    if kind == "np":
        ctx = X3D(*_dims(case), 1.0, 2.0, 3.0, ncl1=(case["first"],) * 3, ncln=(case["last"],) * 3)
        s["in"] = _scalar(case, seed)
        s["out"] = [ctx.field() for _ in range(6)]
        return {**s, "ctx": ctx}
    ctx = X3D(*_dims(case), *_lengths(case))
    s["ctx"] = ctx
    if kind == "ops":
        form = s["form"] = case["form"]
        names = s["names"] = OPS[:15] if form == "mfma" else OPS
        u = _scalar(case, seed)
        if form == "f64":
            s["in"], s["out"] = u, [ctx.field() for _ in names]
        elif form == "bfp":
            s["in"], s["q"] = ctx.bfp_empty(), ctx.bfp_empty()
            ctx.bfp_encode(s["in"], u)
            s["out"] = [ctx.field() for _ in names]
        else:
            s["in"], s["out"] = u.float(), [ctx.field32() for _ in names]
        return s
    u = _velocity(case, seed)
    if kind in ("step", "pieces"):
        if case["stretch"]:
            ctx.set_stretching(1, *_stretching(case))
        s["f"] = u + [ctx.field() for _ in range(7)]
        s["graph"] = case.get("graph", False)
        if s["graph"]:
            ctx.graph_capture_step(*s["f"], gdt=GDT)
    elif kind == "step_f32":
        s["u0"] = [a.float() for a in u]
        del u
        s["f"] = [ctx.field32() for _ in range(10)]
    else:
        s["u0"] = u
        s["f"] = [ctx.bfp_empty() for _ in range(10)]
        s["out"] = [ctx.field() for _ in range(4)]
    return s


def run(s):
    kind = s["kind"]
    if kind == "step":
        if s["graph"]:
            s["ctx"].graph_launch()
        else:
            s["ctx"].step(*s["f"], gdt=GDT)
        return s["f"]
    if kind == "pieces":
        ctx, f = s["ctx"], s["f"]
        u, du, pp, g = f[:3], f[3:6], f[6], f[7:]
        ctx.calculate_transeq_rhs(*du, *u)
        ctx.int_time(*u, *du, gdt=GDT)
        ctx.solve_poisson(pp, *g, *u)
        ctx.cor_vel(*u, *g)
        return f
    if kind == "step_f32":
        # each pass steps the snapshot
        for a, b in zip(s["f"], s["u0"]):
            a.copy_(b)
        s["ctx"].step_f32(*s["f"], gdt=GDT)
        return s["f"]
    if kind == "step_bfp":
        ctx, f = s["ctx"], s["f"]
        for a, b in zip(f, s["u0"]):
            ctx.bfp_encode(a, b)
        ctx.step_bfp(*f, gdt=GDT)
        for a, b in zip(s["out"], f[:3] + [f[6]]):
            ctx.bfp_decode(a, b)
        return s["out"]
    if kind == "batch":
        for a, b in zip(s["f"], s["u0"]):
            a.copy_(b)
        s["b"].graph_launch()
        return s["f"]
    ctx = s["ctx"]
    if kind == "np":
        o, u = s["out"], s["in"]
        ctx.derx(o[0], u, "derx")
        ctx.derx(o[1], u, "derxp")
        ctx.dery(o[2], u, "dery")
        ctx.dery(o[3], u, "deryp")
        ctx.derz(o[4], u, "derz")
        ctx.derz(o[5], u, "derzp")
        return o
    if s["form"] == "bfp":
        for name, o in zip(s["names"], s["out"]):
            ctx.apply_bfp(name, s["q"], s["in"])
            ctx.bfp_decode(o, s["q"])
        return s["out"]
    fn = {"f64": ctx.apply, "f32": ctx.apply_f32, "mfma": ctx.apply_circ_mfma}[s["form"]]
    for name, o in zip(s["names"], s["out"]):
        fn(name, o, s["in"])
    return s["out"]


def work(case):
    """Inputs read once, outputs written once; multiplications and additions
    of the stencils, the line solves and the transforms."""
    kind = case["kind"]
    if kind == "batch":
        pts = sum(a * b * c for a, b, c in _batch_dims(case))
    else:
        pts = case["nx"] * case["ny"] * case["nz"]
    if kind == "np":
        return {"bytes": 7.0 * 8 * pts, "flops": 6.0 * 14 * pts}
    if kind == "ops":
        n, size = (15 if case["form"] == "mfma" else 18), (8 if case["form"] == "f64" else 4)
        out = 8 if case["form"] == "bfp" else size
        return {"bytes": float(size + n * out) * pts, "flops": n * 15.0 * pts}
    flops = (18 * 15.0 + 17 * 15.0 + 2 * 2.5 * math.log2(max(pts, 2)) + 20) * pts
    if kind == "step_bfp":
        return {"bytes": (3 * 8.0 + 4 * 8.0) * pts, "flops": flops}
    size = 4 if kind == "step_f32" or case.get("precision") == 4 else 8
    return {"bytes": 13.0 * size * pts, "flops": flops}


# ---- the same in 64 bits -----------------------------------------------------
def _symbols(n, L, kind):
    """Symbol of one periodic operator over the half spectrum of an axis, as
    complex numbers: the stencil's over that of the tridiagonal matrix."""
    w = TWO_PI / n * torch.arange(n // 2 + 1, dtype=torch.float64, device="cuda")
    h = L / n

    def e(k):
        return torch.polar(torch.ones_like(w), k * w)

    if kind == "d":
        al, top = 1.0 / 3.0, 7.0 / 9.0 / h * (e(1) - e(-1)) + 1.0 / 36.0 / h * (e(2) - e(-2))
    elif kind == "dd":
        al = 2.0 / 11.0
        top = 12.0 / 11.0 / h ** 2 * (e(1) - 2.0 + e(-1)) + 3.0 / 44.0 / h ** 2 * (e(2) - 2.0 + e(-2))
    elif kind in ("dvp", "dpv"):
        al, a, b = 9.0 / 62.0, 63.0 / 62.0 / h, 17.0 / 62.0 / 3.0 / h
        top = a * (e(1) - e(0)) + b * (e(2) - e(-1)) if kind == "dvp" else a * (e(0) - e(-1)) + b * (e(1) - e(-2))
    else:
        al = 0.49
        a, b, c = (75.0 + 70.0 * al) / 128.0, (126.0 * al - 25.0) / 256.0, (-10.0 * al + 3.0) / 256.0
        if kind == "ivp":
            top = a * (e(1) + e(0)) + b * (e(2) + e(-1)) + c * (e(3) + e(-2))
        else:
            top = a * (e(0) + e(-1)) + b * (e(1) + e(-2)) + c * (e(2) + e(-3))
    return top / (1.0 + 2.0 * al * torch.cos(w))


class _Exact:
    """The operators of one grid by their symbols."""

    def __init__(self, dims, L, stretch=None):
        self.n, self.L = dims, L
        self.sy = None
        if stretch is not None:
            self.sy = [torch.from_numpy(v).cuda().reshape(1, -1, 1) for v in stretch]

    def op(self, u, axis, kind):
        n, dim = self.n[axis], 2 - axis
        shape = [1, 1, 1]
        shape[dim] = n // 2 + 1
        f = torch.fft.rfft(u, dim=dim)
        f *= _symbols(n, self.L[axis], kind).reshape(shape)
        r = torch.fft.irfft(f, n=n, dim=dim)
        if self.sy is not None and axis == 1 and kind in ("d", "dvp", "dpv"):
            r *= self.sy[1 if kind == "dvp" else 0]
        return r

    def rhs(self, u):
        return [sum(self.op(u[d] * u[c], d, "d") + u[d] * self.op(u[c], d, "d") for d in range(3)) for c in range(3)]

    def divergence(self, u):
        a, b, c = self.op(u[0], 0, "dvp"), self.op(u[1], 0, "ivp"), self.op(u[2], 0, "ivp")
        t = self.op(a, 1, "ivp") + self.op(b, 1, "dvp")
        c = self.op(c, 1, "ivp")
        return self.op(t, 2, "ivp") + self.op(c, 2, "dvp")

    def poisson(self, r):
        nx, ny, nz = self.n
        k2, t = [], []
        for axis in range(3):
            n = self.n[axis]
            d, i = (_symbols(n, self.L[axis], k).abs() for k in ("dvp", "ivp"))
            if axis:  # mirrored above n / 2
                d, i = (torch.cat([v, v[1:n - n // 2].flip(0)]) for v in (d, i))
            shape = [1, 1, 1]
            shape[2 - axis] = d.numel()
            k2.append((d ** 2).reshape(shape))
            t.append(i.reshape(shape))
        K = k2[0] * (t[1] * t[2]) ** 2 + k2[1] * (t[0] * t[2]) ** 2 + k2[2] * (t[0] * t[1]) ** 2
        f = torch.fft.rfftn(r)
        f *= torch.where(K < 1e-16, torch.zeros_like(K), -1.0 / K)
        return torch.fft.irfftn(f, s=(nz, ny, nx))

    def gradp(self, p):
        a, b = self.op(p, 2, "ipv"), self.op(p, 2, "dpv")
        c, d, e = self.op(a, 1, "ipv"), self.op(a, 1, "dpv"), self.op(b, 1, "ipv")
        return [self.op(c, 0, "dpv"), self.op(d, 0, "ipv"), self.op(e, 0, "ipv")]

    def step(self, u):
        du = self.rhs(u)
        u = [a + GDT * b for a, b in zip(u, du)]
        p = self.poisson(self.divergence(u))
        g = self.gradp(p)
        return [a - b for a, b in zip(u, g)] + du + [p] + g


def _np_matrix(n, h, first, last, paire):
    """Dense matrix of a non-periodic first derivative: sixth-order compact
    rows inside, at an end the even (paire = 1) or odd extension of a free-slip
    boundary (code 1) or the one-sided closures of a Dirichlet one (code 2)."""
    A, B = np.zeros((n, n)), np.zeros((n, n))
    a, b = 7.0 / 9.0 / h, 1.0 / 36.0 / h
    for i in range(n):
        A[i, i] = 1.0
        if 2 <= i <= n - 3 or (i < 2 and first == 1) or (i > n - 3 and last == 1):
            for k, v in ((1, a), (-1, -a), (2, b), (-2, -b)):
                j, sign = i + k, 1.0
                if j < 0:
                    j, sign = -j, (1.0 if paire else -1.0)
                elif j > n - 1:
                    j, sign = 2 * (n - 1) - j, (1.0 if paire else -1.0)
                B[i, j] += sign * v
            # the derivative of an even field is odd, and the other way round
            for k in (1, -1):
                j, sign = i + k, 1.0
                if j < 0 or j > n - 1:
                    j, sign = (-j if j < 0 else 2 * (n - 1) - j), (-1.0 if paire else 1.0)
                A[i, j] += sign / 3.0
        elif i in (0, n - 1):
            d = 1 if i == 0 else -1
            A[i, i + d] = 2.0
            B[i, i], B[i, i + d], B[i, i + 2 * d] = -d * 2.5 / h, d * 2.0 / h, d * 0.5 / h
        else:
            A[i, i - 1] = A[i, i + 1] = 0.25
            B[i, i + 1], B[i, i - 1] = 0.75 / h, -0.75 / h
    return torch.from_numpy(np.linalg.solve(A, B)).cuda()


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        dt = torch.float64 if case["precision"] == 8 else torch.float32
        dims = _batch_dims(case)
        sizes = [nx * ny * nz for nx, ny, nz in dims]
        all3 = [a.to(dt).double().split(sizes) for a in _random3(sum(sizes), seed, (-1,))]
        got = []
        for i, (nx, ny, nz) in enumerate(dims):
            got.append(_Exact(dims[i], (TWO_PI,) * 3).step([a[i].reshape(nz, ny, nx) for a in all3]))
        return [torch.cat([g[k].reshape(-1) for g in got]) for k in range(10)]
    if kind == "np":
        u, out = _scalar(case, seed), []
        for dim, n, L in ((2, case["nx"], 1.0), (1, case["ny"], 2.0), (0, case["nz"], 3.0)):
            for paire in (0, 1):
                m = _np_matrix(n, L / (n - 1), case["first"], case["last"], paire)
                out.append(torch.movedim(torch.movedim(u, dim, -1).reshape(-1, n).matmul(m.t().contiguous()).reshape(
                    *[k for q, k in enumerate(u.shape) if q != dim], n), -1, dim).contiguous())
        return out
    e = _Exact(_dims(case), _lengths(case), _stretching(case))
    if kind == "ops":
        u = _scalar(case, seed)
        if case["form"] in ("f32", "mfma"):
            u = u.float().double()
        out = []
        for name in OPS[:15] if case["form"] == "mfma" else OPS:
            what = name[0] + name[4:] if name[4:] in ("vp", "pv") else ("dd" if name[:3] == "der" and len(name) == 5 else "d")
            out.append(e.op(u, "xyz".index(name[3]), what))
        return out
    u = _velocity(case, seed)
    if kind == "step_f32":
        u = [a.float().double() for a in u]
    r = e.step(u)
    return r[:3] + [r[6]] if kind == "step_bfp" else r
