"""FP64 CG whose alpha comes from p.(K:p) before the inverse transform (a
right-hand side in the range of the projector G), against the oracle and
against the plain schedule that any other right-hand side takes.

Tolerances: iteration counts and fields as in test_gpu_abi_cell.py (equal
counts, 1e-10 relative); at cg_tol 1e-12 the last iterations work near the
rounding of the projection, so the count may differ by one.
"""
import ctypes

import numpy as np
import pytest

from muspectre_amd._device import DeviceBuffer
from test_gpu_abi_cell import GpuCell, _arr, _gpu_cg, _gpu_cg_chunked, _sphere_mask, _two_phase  # noqa: F401

pytestmark = pytest.mark.gpu

# compiled last axis, run-time last axis (odd and even number of rows), a last
# axis beyond both (plain schedule), one row pair less than a workgroup's
CASES = [([16, 32, 16], 0), ([32, 16, 64], 1), ([9, 13, 15], 0), ([7, 11, 19], 1), ([13, 25], 0), ([64, 51], 1),
         ([3, 1203], 1)]


def _cells(capi, oracle, res, form):
    d = len(res)
    even = int(any(n % 2 == 0 for n in res))
    oc = oracle.Cell(res, [1.0] * d, form, allow_even=bool(even))
    gc = GpuCell(capi, res, [1.0] * d, form, allow_even=even)
    _two_phase(oc, gc, _sphere_mask(res, max(2, min(res) / 3)), 1, 1, 100.0, 10.0, .3)
    oc.initialise()
    capi.check(gc.lib.mugpu_cell_initialise(gc.h))
    F = np.zeros((gc.N, d * d)) + (np.eye(d).ravel() if form == 0 else 0.0)
    F[:, 1] += 0.01
    F[:, d] += 0.01
    oc.F[:] = F
    gc.set_F(F)
    oc.evaluate_stress_tangent()
    capi.check(gc.lib.mugpu_cell_evaluate_stress_tangent(gc.h))
    return oc, gc, -oc.apply_projection(oc.P.copy())


@pytest.mark.parametrize("res,form", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else str(v))
def test_projected_rhs_vs_oracle(capi, oracle, res, form):
    oc, gc, rhs = _cells(capi, oracle, res, form)
    for tol, slack in ((1e-8, 0), (1e-12, 1)):
        c0 = oc.counter.value
        ref = oc.cg_solve(rhs, tol, 400)
        count = oc.counter.value - c0
        x, it, conv = _gpu_cg(gc, rhs, tol, 400)
        assert conv and abs(it - count) <= slack
        if it == count:
            assert np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref)
        # queued on the device: the same iterates bit for bit
        x2, _, it2, _, _ = _gpu_cg_chunked(gc, rhs, tol, 400, 8)
        assert it2 == it
        np.testing.assert_array_equal(x2, x)


@pytest.mark.parametrize("res,form", CASES[:6], ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else str(v))
def test_rhs_off_the_range_takes_the_plain_schedule(capi, oracle, res, form):
    """A constant added to the right-hand side (in the null space of G): the
    first iterates are those of SolverCG's loop (solver_cg.cc:62-96) over the
    oracle's operator, whose p.Ap leaves the constant out; p.(K:p) would not.
    (Such a solve has no solution to converge to.)"""
    oc, gc, rhs = _cells(capi, oracle, res, form)
    b = rhs + 1e-3 * np.abs(rhs).max()
    ref, r = np.zeros_like(b), -b
    p, rr = b.copy(), np.sum(b * b)
    for _ in range(3):
        Ap = oc.directional_stiffness(p)
        al = rr / np.sum(p * Ap)
        ref += al * p
        r += al * Ap
        new = np.sum(r * r)
        p, rr = -r + new / rr * p, new
    x, it, _ = _gpu_cg(gc, b, 0.0, 3)
    assert it == 3 and np.linalg.norm(x - ref) <= 1e-10 * np.linalg.norm(ref)
    np.testing.assert_array_equal(_gpu_cg_chunked(gc, b, 0.0, 3, 3)[0], x)


@pytest.mark.parametrize("res,form", [CASES[0], CASES[3]], ids=["compiled", "run-time"])
def test_step_writes_Ap_and_steps_apply_x(capi, oracle, res, form):
    """mugpu_cg_step leaves A p in Ap; where the last axis has no compiled
    passes, x is complete after mugpu_cg_steps without mugpu_cg_finish."""
    _, gc, rhs = _cells(capi, oracle, res, form)
    lib, n = gc.lib, gc.N * gc.nc
    b = DeviceBuffer.from_array(rhs)
    x, r, p, Ap, ref = (DeviceBuffer(8 * n) for _ in range(5))
    rr, bb, done = ctypes.c_double(), ctypes.c_double(), ctypes.c_int()
    capi.check(lib.mugpu_cg_start(gc.h, b.ptr, x.ptr, r.ptr, p.ptr, Ap.ptr, ctypes.byref(rr), ctypes.byref(bb)))
    capi.check(lib.mugpu_cg_step(gc.h, 0, x.ptr, r.ptr, p.ptr, Ap.ptr, ctypes.byref(rr)))
    capi.check(lib.mugpu_cell_directional_stiffness(gc.h, p.ptr, ref.ptr))
    np.testing.assert_array_equal(Ap.download(n), ref.download(n))
    capi.check(lib.mugpu_cg_steps(gc.h, 1, x.ptr, r.ptr, p.ptr, Ap.ptr, 0.0, 5, ctypes.byref(done), ctypes.byref(rr)))
    if res[-1] == 19:
        before = x.download(n)
        capi.check(lib.mugpu_cg_finish(gc.h))
        np.testing.assert_array_equal(x.download(n), before)
    else:
        capi.check(lib.mugpu_cg_finish(gc.h))
    np.testing.assert_array_equal(x.download((gc.N, gc.nc)), _gpu_cg(gc, rhs, 1e-30, 6)[0])
