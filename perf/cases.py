"""Performance cases of the Newton-CG framework.

Each case is one pass through public entry points: the Python package
(`Cell`, `material`, `solvers.newton_cg`, `serving.RVEServer`) or the C-ABI
of include/mugpu.h on device memory, as a program does that keeps its fields
on the GPU.  Sizes follow the benchmark workloads, the tests and the odd grids
that the reference's projections ask for.

kind     one pass
newton   a whole newton_cg load step through the Python package, the strain
         and stress fields read back
cg       one Newton iteration on the device: stress and tangent, the
         right-hand side -G:P and `iters` iterations of SolverCG in FP64
mixed    the same with the FP32 operator and FP64 refinement, solved to the
         relative residual of the benchmark workloads
op       the projected directional stiffness G:(K:dF) of an evaluated cell
proj     the projection G:f of a field, in place
fft      the engine's r2c alone, or r2c followed by c2r
serve    a stream of small-strain solves of uneven resolution through RVEServer

Moduli are in GPa.  `mat`: le1 two phases of MaterialLinearElastic1 (stiffness
contrast 10), le4 MaterialLinearElastic4 with lognormal moduli per voxel,
hep1 two phases of HyperElastoPlastic1 with the consistent tangent.
"""
import ctypes
import math

import numpy as np
import torch

import muspectre_amd as mu
from muspectre_amd import _capi
from muspectre_amd.serving import RVEServer

COMPILED = (16, 32, 48, 64, 96, 128, 256, 512)
CG_TOL, NEWTON_TOL, EQUIL_TOL = 1e-8, 1e-5, 1e-4
SERVE_TOL = 1e-6  # RVEServer's default
CHUNK = 8  # CG iterations queued per call, as SolverCG does
_vp = ctypes.c_void_p


# ------------------------------------------------------------------- cases
def _case(name, kind, res, **more):
    c = {"name": name, "kind": kind, "dim": len(res)}
    c.update(zip(("nx", "ny", "nz"), res))
    c.update(more)
    return c


def listed():
    return [
        # the smallest call: the reference's 2D demonstration script
        _case("newton_51x51", "newton", (51, 51), form="small", mat="le1", prec="fp64"),
        # a laptop-sized 3D cell on an odd grid, geometrically nonlinear
        _case("newton_33x27x35_finite", "newton", (33, 27, 35), form="finite", mat="le1", prec="fp64"),
        # a random medium on an odd grid, read back as a script does
        _case("newton_63x63x63_small", "newton", (63, 63, 63), form="small", mat="le4", prec="fp64"),
        # a particle composite at the benchmark's middle size
        _case("cg_128x128x128_small", "cg", (128, 128, 128), form="small", mat="le1", iters=32),
        # the same on the odd grid next to it, which the reference asks for
        _case("cg_125x125x125_small", "cg", (125, 125, 125), form="small", mat="le4", iters=32),
        # a ragged odd cell, finite strain, full symmetric tangent
        _case("cg_175x147x99_finite", "cg", (175, 147, 99), form="finite", mat="le1", iters=24),
        # the flagship benchmark: 256^3 elasto-plastic finite strain
        _case("cg_256x256x256_hep1", "cg", (256, 256, 256), form="finite", mat="hep1", iters=32),
        # a ragged 2D section
        _case("cg_255x243_small", "cg", (255, 243), form="small", mat="le1", iters=32),
        # the FP32-refined solve of a random medium
        _case("mixed_128x128x128_small", "mixed", (128, 128, 128), form="small", mat="le4"),
        # the projection alone, FP32, a large 2D section (finite strain)
        _case("proj_512x512_fp32", "proj", (512, 512), form="finite", prec="fp32"),
        # the engine's transforms on an odd 3D grid, both directions
        _case("fft_135x105x77_round", "fft", (135, 105, 77), prec="fp64", way="round"),
        # a burst of requests of uneven resolution
        _case("serve_12", "serve", (32, 64), requests=12),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, odd=0.6):
    """An axis length: odd, any, or one of the powers of two and their like."""
    u = rng.random()
    if u < odd:
        return min(hi, _log(rng, lo, hi) | 1)
    if u < odd + 0.1:
        return _log(rng, lo, hi)
    return rng.choice([n for n in COMPILED if lo <= n <= hi] or [lo])


def draw(rng):
    kind = rng.choice(["newton", "newton", "cg", "cg", "cg", "cg", "mixed", "op", "proj", "fft", "serve"])
    if kind == "serve":
        return {k: v for k, v in _case("", "serve", (rng.choice([32, 48]), rng.choice([64, 128])),
                                       requests=rng.randrange(4, 17)).items() if k != "name"}
    dim = 2 if rng.random() < 0.3 else 3
    most = {"newton": 200_000, "cg": 3_000_000, "mixed": 2_500_000, "op": 4_000_000, "proj": 4_000_000,
            "fft": 4_000_000}[kind]
    hi = {2: 151 if kind == "newton" else 512, 3: 63 if kind == "newton" else 256}[dim]
    while True:
        res = tuple(_size(rng, 11, hi) for _ in range(dim))
        if math.prod(res) <= most:
            break
    c = _case("", kind, res)
    form = rng.choice(["small", "finite"])
    if kind in ("newton", "cg", "mixed", "op", "proj"):
        c["form"] = "small" if kind == "mixed" else form
    if kind in ("newton", "cg", "op", "mixed"):
        c["mat"] = rng.choice(["le1", "le4"])
    if kind == "newton":
        c["prec"] = "fp32" if c["form"] == "small" and rng.random() < 0.25 else "fp64"
    if kind in ("proj", "fft"):
        c["prec"] = rng.choice(["fp64", "fp64", "fp32"])
    if kind == "fft":
        c["way"] = rng.choice(["r2c", "round"])
    if kind == "cg":
        c["iters"] = rng.choice([8, 16, 24, 32])
    del c["name"]
    return c


def _res(case):
    return [int(case[k]) for k in ("nx", "ny", "nz")[:case["dim"]]]


# ---------------------------------------------------------- what a cell holds
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _smooth(res, g):
    """A smooth periodic random field of unit variance on the grid."""
    out = torch.zeros(res, dtype=torch.float64, device="cuda")
    waves = 24
    k = torch.randint(-4, 5, (waves, len(res)), generator=g, device="cuda").double()
    ph = 2 * math.pi * torch.rand(waves, generator=g, device="cuda", dtype=torch.float64)
    for w in range(waves):
        arg = ph[w]
        for d, n in enumerate(res):
            x = 2 * math.pi * torch.arange(n, device="cuda", dtype=torch.float64) / n * k[w, d]
            arg = arg + x.reshape([-1 if e == d else 1 for e in range(len(res))])
        out += torch.cos(arg)
    return out.mul_(math.sqrt(2.0 / waves))


def _macro(case):
    """Macroscopic strain (small strain) or displacement gradient."""
    d = case["dim"]
    m = np.zeros((d, d))
    if case.get("mat") == "hep1":
        m[d - 1, d - 1] = 0.005
    else:
        m[0, 0], m[0, 1], m[1, 0] = 0.004, 0.01, 0.01
    return m


def _medium(case, seed):
    """The microstructure: a phase mask, or (E, nu) per voxel."""
    res, g = _res(case), _gen(seed)
    if case["mat"] == "le4":
        n = math.prod(res)
        E = 50.0 * torch.exp(0.3 * torch.randn(n, generator=g, device="cuda", dtype=torch.float64))
        nu = 0.2 + 0.2 * torch.rand(n, generator=g, device="cuda", dtype=torch.float64)
        return torch.stack([E, nu], 1)
    return (_smooth(res, g) > 0.3).reshape(-1)


LE1 = ((100.0, 0.3), (10.0, 0.3))  # inclusion, matrix
HEP1 = ((210.0, 0.33, 0.8, 1.0), (70.0, 0.33, 0.2, 1.0))  # E, nu, tau_y0, H


def _strain(case, seed):
    """The strain of a cell inside a Newton loop: macroscopic plus a smooth
    fluctuation; AoS, component i + dim j."""
    res, d = _res(case), case["dim"]
    g = _gen(seed + 7919)
    m = _macro(case)
    F = torch.empty(res + [d, d], dtype=torch.float64, device="cuda")  # [..., j, i]
    fine = case["form"] == "finite"
    amp = 0.1 * float(np.abs(m).max())
    for j in range(d):
        for i in range(d):
            if not fine and i < j:
                F[..., j, i] = F[..., i, j]
                continue
            F[..., j, i] = amp * _smooth(res, g) + float(m[i, j]) + (1.0 if fine and i == j else 0.0)
    return F.reshape(-1, d * d)


class _Cell:
    """A cell held through the C-ABI; freed with its last reference."""

    def __init__(self, case, seed, precision):
        self.lib = lib = _capi.load()
        _capi.check(lib.mugpu_init(0))
        res, d = _res(case), case["dim"]
        self.n = math.prod(res) * d * d
        h = _vp()
        _capi.check(lib.mugpu_cell_create(
            d, (ctypes.c_int * d)(*res), (ctypes.c_double * d)(*[1.0 + 0.1 * k for k in range(d)]),
            _capi.SMALL_STRAIN if case["form"] == "small" else _capi.FINITE_STRAIN, precision,
            1 if any(r % 2 == 0 for r in res) else 0, ctypes.byref(h)))
        self.h = h
        med = _medium(case, seed)
        if case["mat"] == "le4":
            self._add(_capi.LE4, (0.0, 0.0, 0.0, 0.0), np.arange(math.prod(res), dtype=np.int64), med.cpu().numpy())
        else:
            mask = med.cpu().numpy()
            fam, pars = (_capi.HEP1_CT, HEP1) if case["mat"] == "hep1" else (_capi.LE1, LE1)
            for par, idx in zip(pars, (np.flatnonzero(mask), np.flatnonzero(~mask))):
                self._add(fam, tuple(par) + (0.0,) * (4 - len(par)), idx.astype(np.int64), None)
        _capi.check(lib.mugpu_cell_initialise(h))
        F = _strain(case, seed)
        p = _vp()
        _capi.check(lib.mugpu_cell_strain(h, ctypes.byref(p)))
        torch.cuda.synchronize()
        _capi.check(lib.mugpu_scale_copy(1.0, F.data_ptr(), p, self.n))
        _capi.check(lib.mugpu_cell_stress(h, ctypes.byref(p)))
        self.P = p
        _capi.check(lib.mugpu_synchronize())

    def _add(self, family, par, idx, params):
        m = ctypes.c_int()
        _capi.check(self.lib.mugpu_cell_add_material(self.h, family, *par, ctypes.byref(m)))
        pp = None if params is None else np.ascontiguousarray(params).ctypes.data_as(ctypes.POINTER(ctypes.c_double))
        _capi.check(self.lib.mugpu_material_add_pixels(
            self.h, m, len(idx), idx.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), pp))

    def __del__(self):
        if getattr(self, "h", None):
            self.lib.mugpu_cell_destroy(self.h)
            self.h = None


def _dev(n, dtype=torch.float64):
    return torch.zeros(n, dtype=dtype, device="cuda")


def _requests(case, seed):
    """The burst: resolutions in turn, a smooth two-phase medium each."""
    a, b = int(case["nx"]), int(case["ny"])
    sizes = [(a, a, a), (b, b), (2 * a, a, a), (2 * b, b)]
    out = []
    for i in range(int(case["requests"])):
        res = list(sizes[i % 4])
        g = _gen(seed * 1000 + i)
        mask = (_smooth(res, g) > 0.3).reshape(-1).cpu().numpy()
        con, nu = (10.0 ** torch.rand(1, generator=g, device="cuda", dtype=torch.float64)).item(), 0.2 + 0.01 * i
        d = len(res)
        e = (0.02 * torch.rand(d, d, generator=g, device="cuda", dtype=torch.float64) - 0.01).cpu().numpy()
        out.append((res, np.where(mask, con, 1.0), np.full(mask.size, nu), 0.5 * (e + e.T)))
    return out


def prepare(case, seed):
    kind, d = case["kind"], case["dim"]
    st = {"case": case}
    if kind == "serve":
        st["requests"] = _requests(case, seed)
        st["server"] = RVEServer(hbm_budget=2 << 30, cg_tol=SERVE_TOL)
        return st
    res = _res(case)
    n = math.prod(res) * d * d
    even = any(r % 2 == 0 for r in res)
    if kind == "newton":
        form = mu.Formulation.small_strain if case["form"] == "small" else mu.Formulation.finite_strain
        cell = mu.Cell(res, [1.0 + 0.1 * k for k in range(d)], form, precision=case["prec"], allow_even=even)
        med = _medium(case, seed).cpu().numpy()
        make = getattr(mu.material, "MaterialLinearElastic%s_%dd" % (case["mat"][2], d)).make
        if case["mat"] == "le4":
            make(cell, "medium").add_pixels_by_index(np.arange(len(med)), med)
        else:
            for (E, nu), name, idx in zip(LE1, ("inclusion", "matrix"), (np.flatnonzero(med), np.flatnonzero(~med))):
                make(cell, name, E, nu).add_pixels_by_index(idx)
        cell.initialise()
        st.update(cell=cell, load=_macro(case))
    elif kind in ("cg", "mixed", "op"):
        st["cell"] = c = _Cell(case, seed, _capi.FP32 if kind == "mixed" else _capi.FP64)
        st["lib"], st["n"] = c.lib, n
        if kind == "op":
            _capi.check(c.lib.mugpu_cell_evaluate_stress_tangent(c.h))
            st["in"] = torch.randn(n, generator=_gen(seed + 1), device="cuda", dtype=torch.float64)
            st["out"] = _dev(n)
        else:
            st["rhs"], st["x"] = _dev(n), _dev(n)
            if kind == "cg":
                st["work"] = [_dev(n) for _ in range(3)]
    else:
        st["lib"] = lib = _capi.load()
        _capi.check(lib.mugpu_init(0))
        real = torch.float64 if case["prec"] == "fp64" else torch.float32
        plan = _vp()
        _capi.check(lib.mugpu_fft_create(d, (ctypes.c_int * d)(*res), d * d,
                                         _capi.FP64 if case["prec"] == "fp64" else _capi.FP32, ctypes.byref(plan)))
        st["field"] = torch.randn(n, generator=_gen(seed + 1), device="cuda", dtype=torch.float64).to(real)
        if kind == "proj":
            h = _vp()
            _capi.check(lib.mugpu_projection_create(
                plan, _capi.PROJ_SMALL_STRAIN if case["form"] == "small" else _capi.PROJ_FINITE_STRAIN_FAST,
                (ctypes.c_double * d)(*[1.0 + 0.1 * k for k in range(d)]), 1 if even else 0, ctypes.byref(h)))
            st["owner"] = _Owner(lib.mugpu_projection_destroy, h)
        else:
            st["owner"] = _Owner(lib.mugpu_fft_destroy, plan)
            st["spec"] = _dev(2 * n // res[-1] * (res[-1] // 2 + 1), real)
            st["back"] = _dev(n, real)
    torch.cuda.synchronize()
    return st


class _Owner:
    def __init__(self, free, h):
        self.free, self.h = free, h

    def __del__(self):
        if self.h:
            self.free(self.h)
            self.h = None


# --------------------------------------------------------------------- a pass
def _run_newton(st):
    solver = mu.solvers.SolverCG(st["cell"], CG_TOL, 2000, False)
    r = mu.solvers.newton_cg(st["cell"], [st["load"]], solver, NEWTON_TOL, EQUIL_TOL, 0)[0]
    return {"grad": r.grad, "stress": r.stress}


def _rhs(st):
    """Stress and tangent at the cell's strain, and rhs = -G:P."""
    lib, c = st["lib"], st["cell"]
    _capi.check(lib.mugpu_cell_evaluate_stress_tangent(c.h))
    _capi.check(lib.mugpu_scale_copy(-1.0, c.P, st["rhs"].data_ptr(), st["n"]))
    _capi.check(lib.mugpu_cell_apply_projection(c.h, st["rhs"].data_ptr()))


def _run_cg(st):
    lib, h = st["lib"], st["cell"].h
    _rhs(st)
    x, (r, p, Ap) = st["x"].data_ptr(), [w.data_ptr() for w in st["work"]]
    rr, bb, done = ctypes.c_double(), ctypes.c_double(), ctypes.c_int()
    _capi.check(lib.mugpu_cg_start(h, st["rhs"].data_ptr(), x, r, p, Ap, ctypes.byref(rr), ctypes.byref(bb)))
    for it in range(0, int(st["case"]["iters"]), CHUNK):
        _capi.check(lib.mugpu_cg_steps(h, 1 if it else 0, x, r, p, Ap, 0.0, CHUNK, ctypes.byref(done),
                                       ctypes.byref(rr)))
    _capi.check(lib.mugpu_cg_finish(h))
    return {"rhs": st["rhs"], "x": st["x"]}


def _run_mixed(st):
    lib, h = st["lib"], st["cell"].h
    _rhs(st)
    its, refs, rel = ctypes.c_int64(), ctypes.c_int(), ctypes.c_double()
    _capi.check(lib.mugpu_cg_solve_mixed(h, st["rhs"].data_ptr(), st["x"].data_ptr(), CG_TOL, 2000, 1e-4,
                                         ctypes.byref(its), ctypes.byref(refs), ctypes.byref(rel)))
    return {"rhs": st["rhs"], "x": st["x"]}


def _run_serve(st):
    srv = st["server"]
    ids = [srv.submit(res, E, nu, eps) for res, E, nu, eps in st["requests"]]
    srv.run()
    srv.poll()
    out = [srv.result(i)["mean_stress"] for i in ids]
    for i in ids:
        srv.release(i)
    return out


def run(st):
    kind = st["case"]["kind"]
    if kind == "newton":
        return _run_newton(st)
    if kind == "cg":
        return _run_cg(st)
    if kind == "mixed":
        return _run_mixed(st)
    if kind == "serve":
        return _run_serve(st)
    lib = st["lib"]
    if kind == "op":
        _capi.check(lib.mugpu_cell_directional_stiffness(st["cell"].h, st["in"].data_ptr(), st["out"].data_ptr()))
        return st["out"]
    if kind == "proj":
        _capi.check(lib.mugpu_projection_apply(st["owner"].h, st["field"].data_ptr()))
        return st["field"]
    _capi.check(lib.mugpu_fft_r2c(st["owner"].h, st["field"].data_ptr(), st["spec"].data_ptr()))
    if st["case"]["way"] == "r2c":
        return st["spec"]
    _capi.check(lib.mugpu_fft_c2r(st["owner"].h, st["spec"].data_ptr(), st["back"].data_ptr()))
    return st["back"]


# ----------------------------------------------------------- what it must move
def _operator_work(N, d, comp, size, tan):
    """G:(K:p): p in, the spectrum of `comp` components between the axes, and
    the result out."""
    sweeps = 2 * d if d > 1 else 2
    return N * (2 * comp * size + sweeps * 2 * comp * size // 2 + tan), N * comp * 2 * 2.5 * math.log2(N)


def work(case):
    kind, d = case["kind"], case["dim"]
    if kind == "serve":
        its, total = 50, {"bytes": 0.0, "flops": 0.0}
        a, b = case["nx"], case["ny"]
        for i in range(int(case["requests"])):
            N, dd = ((a ** 3, 3), (b ** 2, 2), (2 * a ** 3, 3), (2 * b ** 2, 2))[i % 4]
            by, fl = _operator_work(N, dd, dd * (dd + 1) // 2, 4, 8)
            total["bytes"] += 16 * N + its * (by + N * 5 * dd * (dd + 1) // 2 * 4)
            total["flops"] += its * fl
        return total
    N = math.prod(_res(case))
    full = d * d
    if kind == "fft":
        s = 8 if case["prec"] == "fp64" else 4
        ways = 1 if case["way"] == "r2c" else 2
        return {"bytes": ways * N * full * s * 2 * d, "flops": ways * N * full * 2.5 * math.log2(N)}
    comp = full if case["form"] == "finite" else d * (d + 1) // 2
    if kind == "proj":
        s = 8 if case["prec"] == "fp64" else 4
        by, fl = _operator_work(N, d, comp, s, 0)
        return {"bytes": by, "flops": fl}
    f32 = kind == "mixed" or case.get("prec") == "fp32"
    s = 4 if f32 else 8
    tan = (full * (full + 1) // 2 if case["form"] == "finite" else 2) * s
    by, fl = _operator_work(N, d, comp, s, tan)
    if kind == "op":
        return {"bytes": by, "flops": fl}
    its = case.get("iters", 60)
    # x, r and p are read and written once per iteration besides the operator's p
    per = by + N * comp * s * 4
    return {"bytes": its * per + N * full * 8 * 4, "flops": its * fl}


# ------------------------------------------------- the same in 64 bits, plainly
def _freqs(res, lengths):
    ks = [torch.fft.fftfreq(n, 1.0 / n, device="cuda", dtype=torch.float64) for n in res]
    ks[-1] = torch.arange(res[-1] // 2 + 1, device="cuda", dtype=torch.float64)
    if res[-1] % 2 == 0:
        ks[-1][-1] = -(res[-1] // 2)
    d = len(res)
    q = [(k / L).reshape([-1 if e == a else 1 for e in range(d)]) for a, (k, L) in enumerate(zip(ks, lengths))]
    keep = torch.ones([len(k) for k in ks], dtype=torch.float64, device="cuda")
    keep[(0,) * d] = 0.0
    for a, n in enumerate(res):
        if n % 2 == 0:
            keep.select(a, n // 2).zero_()
    n2 = sum(x * x for x in q)
    n2[(0,) * d] = 1.0
    inv = 1.0 / torch.sqrt(n2)
    return [x * inv for x in q], keep


class _Plain:
    """G, K and the solvers over fields f[j][i] (tensor component i, j) as
    plain grids in FP64."""

    def __init__(self, res, form, lengths=None):
        self.res, self.d, self.small = list(res), len(res), form == "small"
        self.xi, self.keep = _freqs(self.res, lengths or [1.0 + 0.1 * k for k in range(self.d)])

    def split(self, f):
        """AoS (n, dim*dim) -> list over components of grids."""
        return [f.reshape(self.res + [-1])[..., c].contiguous() for c in range(self.d ** 2)]

    def join(self, f):
        return torch.stack([x.reshape(-1) for x in f], 1).reshape(-1)

    def G(self, f):
        d, xi = self.d, self.xi
        h = [torch.fft.rfftn(x) * self.keep for x in f]
        at = lambda i, j: h[i + d * j]
        if self.small:
            a = [sum((at(i, m) + at(m, i)) * 0.5 * xi[m] for m in range(d)) for i in range(d)]
            s = sum(xi[i] * a[i] for i in range(d))
            g = [xi[i] * a[j] + xi[j] * a[i] - xi[i] * xi[j] * s for j in range(d) for i in range(d)]
        else:
            a = [sum(at(i, m) * xi[m] for m in range(d)) for i in range(d)]
            g = [a[i] * xi[j] for j in range(d) for i in range(d)]
        return [torch.fft.irfftn(x, s=self.res, dim=tuple(range(d))) for x in g]

    def elastic(self, lam, mu_):
        self.lam, self.mu = lam, mu_

    def hooke(self, E):
        d = self.d
        tr = sum(E[i + d * i] for i in range(d))
        return [(self.lam * tr if i == j else 0.0) + self.mu * (E[i + d * j] + E[j + d * i])
                for j in range(d) for i in range(d)]

    def mm(self, A, B, ta=False):
        d = self.d
        return [sum((A[k + d * i] if ta else A[i + d * k]) * B[k + d * j] for k in range(d))
                for j in range(d) for i in range(d)]

    def stress(self, F):
        """P at F; keeps what K needs."""
        if self.small:
            return self.hooke(F)
        d = self.d
        E = self.mm(F, F, ta=True)
        E = [0.5 * (e - (1.0 if c % (d + 1) == 0 else 0.0)) for c, e in enumerate(E)]
        self.F, self.S = F, self.hooke(E)
        return self.mm(F, self.S)

    def K(self, dF):
        if self.small:
            return self.hooke(dF)
        d = self.d
        dE = self.mm(self.F, dF, ta=True)
        dE = [0.5 * (dE[i + d * j] + dE[j + d * i]) for j in range(d) for i in range(d)]
        return [a + b for a, b in zip(self.mm(dF, self.S), self.mm(self.F, self.hooke(dE)))]

    @staticmethod
    def dot(a, b):
        return sum((x * y).sum() for x, y in zip(a, b)).item()

    def cg(self, b, iters, tol=0.0):
        x = [torch.zeros_like(v) for v in b]
        r = [-v for v in b]
        p = [v.clone() for v in b]
        rr = bb = self.dot(b, b)
        for _ in range(iters):
            Ap = self.G(self.K(p))
            al = rr / self.dot(p, Ap)
            for k in range(len(b)):
                x[k] += al * p[k]
                r[k] += al * Ap[k]
            new = self.dot(r, r)
            p = [-v + (new / rr) * w for v, w in zip(r, p)]
            rr = new
            if not rr > tol * tol * bb:
                break
        return x


def _plain_cell(case, seed):
    q = _Plain(_res(case), case["form"])
    med = _medium(case, seed)
    if case["mat"] == "le4":
        E, nu = med[:, 0], med[:, 1]
    else:
        E = torch.where(med, LE1[0][0], LE1[1][0]).double()
        nu = torch.full_like(E, LE1[0][1])
    E, nu = E.reshape(q.res), nu.reshape(q.res)
    q.elastic(E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu)))
    return q


def _plain_newton(q, load, tol):
    d = q.d
    F = [torch.full(q.res, float(load[c % d, c // d]) + (0.0 if q.small or c % (d + 1) else 1.0),
                    dtype=torch.float64, device="cuda") for c in range(d * d)]
    incr, grad, P = 2 * NEWTON_TOL, 1.0, None
    for _ in range(50):
        P = q.stress(F)
        b = q.G([-v for v in P])
        if math.sqrt(q.dot(b, b)) < EQUIL_TOL:
            break
        x = q.cg(b, 2000, tol)
        F = [a + v for a, v in zip(F, x)]
        incr, grad = math.sqrt(q.dot(x, x)), math.sqrt(q.dot(F, F))
        if incr / grad <= NEWTON_TOL:
            break
    return F, P


def exact(case, seed):
    kind, d = case["kind"], case["dim"]
    if kind == "serve":
        out = []
        for res, E, nu, eps in _requests(case, seed):
            q = _Plain(res, "small", [1.0] * len(res))
            E, nu = (torch.as_tensor(v, device="cuda").reshape(res) for v in (E, nu))
            q.elastic(E * nu / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu)))
            _, P = _plain_newton(q, eps, 1e-12)
            out.append(np.array([v.mean().item() for v in P]))
        return out
    if kind == "fft":
        res = _res(case)
        f = torch.randn(math.prod(res) * d * d, generator=_gen(seed + 1), device="cuda", dtype=torch.float64)
        f = f.to(torch.float64 if case["prec"] == "fp64" else torch.float32).double()
        if case["way"] == "round":
            return f * float(math.prod(res))
        return torch.view_as_real(torch.fft.rfftn(f.reshape(res + [-1]), dim=tuple(range(d))).contiguous()).reshape(-1)
    if kind == "proj":
        q = _Plain(_res(case), case["form"])
        f = torch.randn(math.prod(q.res) * d * d, generator=_gen(seed + 1), device="cuda", dtype=torch.float64)
        f = f.to(torch.float64 if case["prec"] == "fp64" else torch.float32).double()
        return q.join(q.G(q.split(f)))
    if case["mat"] == "hep1":
        return None  # 3x3 eigenproblems of every voxel: minutes in plain torch
    q = _plain_cell(case, seed)
    if kind == "newton":
        F, P = _plain_newton(q, _macro(case), 1e-12 if case["prec"] == "fp32" else CG_TOL)
        return {"grad": q.join(F).cpu().numpy().reshape(-1, 1), "stress": q.join(P).cpu().numpy().reshape(-1, 1)}
    P = q.stress(q.split(_strain(case, seed)))
    if kind == "op":
        f = torch.randn(math.prod(q.res) * d * d, generator=_gen(seed + 1), device="cuda", dtype=torch.float64)
        return q.join(q.G(q.K(q.split(f))))
    b = q.G([-v for v in P])
    x = q.cg(b, int(case["iters"])) if kind == "cg" else q.cg(b, 2000, 1e-13)
    return {"rhs": q.join(b), "x": q.join(x)}
