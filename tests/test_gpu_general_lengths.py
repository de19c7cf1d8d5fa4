"""Passes along axes of run-time length, at the lengths where they can go
wrong: every compiled radix alone and with a span before it, primes without a
compiled butterfly (one and two of them, one or two tasks per thread), the
lengths whose workgroups just fit and the next ones that fall back, and grids
whose tiles of rows, lines or k-points end in a remainder.

Oracle: numpy's FFT in FP64.  Tolerance: a pass of radix R rounds a sum of R
terms, so the relative 2-norm error of a transform is at most about
eps * sum over the passes of sqrt(R), with a factor 8 for the twiddles, the
separation of the paired rows and numpy's own error; FP32 (the engine's
transforms and the projections) likewise with its own eps.
"""
import ctypes

import numpy as np
import pytest

from muspectre_amd._device import DeviceBuffer

pytestmark = pytest.mark.gpu

SIZES = [
    # each radix as the only pass, and after another one
    [2, 3], [5, 7], [9, 8], [11, 13], [17, 4], [34, 22], [26, 51], [63, 45], [72, 99], [121, 15],
    # primes without a compiled butterfly: 19, 23 and 31 small, 127 and 251 long, two in one length
    [19, 23], [46, 57], [31, 62], [127, 19], [6, 251], [251, 5], [437, 3], [4, 437],
    # long axes: the last that fit a workgroup, and beyond (2D last axis, first axis)
    [3, 1000], [3, 1100], [1050, 3], [1280, 2], [2000, 1],
    # 3D: the three roles, remainders in every tile, a single point on an axis
    [23, 10, 14], [10, 29, 21], [7, 33, 37], [50, 18, 3], [1, 13, 25], [25, 1, 13], [13, 25, 1], [80, 40, 20],
    [3, 5, 660], [3, 5, 700], [600, 3, 2], [2, 600, 3],
]


def _passes(n):
    out = []
    for r in (17, 13, 11, 9, 8, 7, 5, 4, 3, 2):
        while n % r == 0:
            out.append(r)
            n //= r
    r = 19
    while n > 1:
        while n % r == 0:
            out.append(r)
            n //= r
        r += 2
    return out


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("res", SIZES, ids=lambda r: "x".join(map(str, r)))
def test_transforms_vs_numpy(capi, res, prec):
    dt, ct = (np.float64, np.complex128) if prec == 0 else (np.float32, np.complex64)
    lib = capi.load()
    d, N = len(res), int(np.prod(res))
    nc = d * d
    rng = np.random.default_rng(N)
    h = ctypes.c_void_p()
    capi.check(lib.mugpu_fft_create(d, (ctypes.c_int * d)(*res), nc, prec, ctypes.byref(h)))
    tol = 8 * np.finfo(dt).eps * (1 + sum(np.sqrt(r) for n in res for r in _passes(n)))
    try:
        kp = lib.mugpu_fft_nb_fourier_points(h)
        herm = [*res[:-1], res[-1] // 2 + 1]
        x = rng.standard_normal([*res, nc]).astype(dt)
        din = DeviceBuffer.from_array(x)
        dspec = DeviceBuffer(kp * nc * np.dtype(ct).itemsize)
        capi.check(lib.mugpu_fft_r2c(h, din.ptr, dspec.ptr))
        spec = dspec.download((*herm, nc), ct)
        ref = np.fft.rfftn(x.astype(np.float64), axes=tuple(range(d)))
        assert np.linalg.norm(spec - ref) <= tol * np.linalg.norm(ref)
        dout = DeviceBuffer(x.nbytes)
        capi.check(lib.mugpu_fft_c2r(h, dspec.ptr, dout.ptr))
        out = dout.download((*res, nc), dt).astype(np.float64) / N
        assert np.linalg.norm(out - x) <= 2 * tol * np.linalg.norm(x)
    finally:
        lib.mugpu_fft_destroy(h)


@pytest.mark.parametrize("form", [0, 1], ids=["finite", "small"])
@pytest.mark.parametrize("res", [[51, 38], [23, 7], [15, 22, 9], [9, 26, 13], [19, 6, 17],
                                 # compiled last axis under an odd number of rows
                                 [5, 7, 16], [3, 5, 96], [9, 512], [7, 256]],
                         ids=lambda r: "x".join(map(str, r)))
def test_operator_vs_oracle(capi, oracle, res, form):
    """G:(K:dF) through every pass of a cell (small strain: packed symmetric
    lines, of a dF that is not symmetric); the bound of the other operator
    tests, 1e-12 of the largest value."""
    from test_gpu_abi_cell import GpuCell
    d, N = len(res), int(np.prod(res))
    even = int(any(r % 2 == 0 for r in res))
    L = [1.0, 1.3, 0.7][:d]
    oc = oracle.Cell(res, L, form, allow_even=bool(even))
    gc = GpuCell(capi, res, L, form, allow_even=even)
    mo, mg = oc.add_material(1, 70.0, .3), gc.add_material(1, 70.0, .3)
    for i in range(N):
        oc.add_pixel(mo, i)
    gc.add_pixels(mg, np.arange(N))
    oc.initialise()
    capi.check(gc.lib.mugpu_cell_initialise(gc.h))
    rng = np.random.default_rng(7)
    F = 0.01 * rng.standard_normal((N, d * d)) + (np.eye(d).ravel() if form == 0 else 0.0)
    oc.F[:] = F
    gc.set_F(F)
    oc.evaluate_stress_tangent()
    capi.check(gc.lib.mugpu_cell_evaluate_stress_tangent(gc.h))
    dF = rng.standard_normal((N, d * d))
    ref = oc.directional_stiffness(dF)
    bi, bo = DeviceBuffer.from_array(dF), DeviceBuffer(dF.nbytes)
    capi.check(gc.lib.mugpu_cell_directional_stiffness(gc.h, bi.ptr, bo.ptr))
    assert np.abs(bo.download(dF.shape) - ref).max() <= 1e-12 * np.abs(ref).max()
    # the projection alone
    refG = oc.apply_projection(dF.copy())
    capi.check(gc.lib.mugpu_cell_apply_projection(gc.h, bi.ptr))
    assert np.abs(bi.download(dF.shape) - refG).max() <= 1e-12 * np.abs(refG).max()


@pytest.mark.parametrize("kind", [0, 1, 2], ids=["small", "finite_fast", "finite"])
@pytest.mark.parametrize("res", [[51, 38], [23, 7], [15, 22, 9], [9, 26, 13], [16, 9, 48]],
                         ids=lambda r: "x".join(map(str, r)))
def test_fp32_projection_vs_fp64(capi, res, kind):
    """The FP32 projection against the FP64 one of the same field: the two
    transforms and the projection round like one more pass of radix dim^2."""
    lib, d, N = capi.load(), len(res), int(np.prod(res))
    f = np.random.default_rng(3).standard_normal((N, d * d)).astype(np.float32)
    out = []
    for prec, dt in ((0, np.float64), (1, np.float32)):
        plan, proj = ctypes.c_void_p(), ctypes.c_void_p()
        capi.check(lib.mugpu_fft_create(d, (ctypes.c_int * d)(*res), d * d, prec, ctypes.byref(plan)))
        capi.check(lib.mugpu_projection_create(plan, kind, (ctypes.c_double * d)(*[1.0, 1.3, 0.7][:d]), 1,
                                               ctypes.byref(proj)))
        buf = DeviceBuffer.from_array(f.astype(dt))
        capi.check(lib.mugpu_projection_apply(proj, buf.ptr))
        out.append(buf.download(f.shape, dt).astype(np.float64))
        lib.mugpu_projection_destroy(proj)
    tol = 16 * np.finfo(np.float32).eps * (1 + d + sum(np.sqrt(r) for n in res for r in _passes(n)))
    assert np.linalg.norm(out[1] - out[0]) <= tol * np.linalg.norm(f)
