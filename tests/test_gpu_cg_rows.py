"""Small-strain CG on grids whose last workgroup of the run-time-length r2c pass
misses rows beyond its first row pair (test_stage_bounds.py has the index
arithmetic): the first iterations against SolverCG's loop (solver_cg.cc:62-96)
over the oracle's operator, and chunks against single steps bit for bit.

Tolerance: 1e-10 of the norm, as in test_gpu_cg_early_alpha.py.
"""
import numpy as np
import pytest

from test_gpu_abi_cell import _sphere_mask
from test_gpu_cg_ring import _cell, _Solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("res", [[67, 67, 67], [65, 66, 63], [101, 101, 35], [99, 75, 63]],
                         ids=lambda r: "x".join(map(str, r)))
def test_missing_row_pairs(capi, oracle, res):
    gc, rhs = _cell(capi, res, 1)
    oc = oracle.Cell(res, [1.0] * 3, 1, allow_even=bool(any(n % 2 == 0 for n in res)))
    mask = _sphere_mask(res, max(2, min(res) / 3)).ravel()
    mi, mo = oc.add_material(1, 100.0, .3), oc.add_material(1, 10.0, .3)
    for i in range(mask.size):
        oc.add_pixel(mi if mask[i] else mo, i)
    oc.initialise()
    oc.evaluate_stress_tangent()
    b = rhs.download((gc.N, gc.nc))
    x, r = np.zeros_like(b), -b
    p, rr = b.copy(), np.sum(b * b)
    s = _Solve(capi, gc, rhs)
    assert s.steps(3, 0.0) == 3
    for it in range(3):
        p = p if it == 0 else -r + beta * p  # noqa: F821
        Ap = oc.directional_stiffness(p)
        al = rr / np.sum(p * Ap)
        x += al * p
        r += al * Ap
        new = np.sum(r * r)
        beta, rr = new / rr, new  # noqa: F841
    for got, want in zip(s.vectors(), (x, r, p)):
        assert np.linalg.norm(got - want.ravel()) <= 1e-10 * np.linalg.norm(want)
    t = _Solve(capi, gc, rhs)
    for _ in range(3):
        t.step()
    for got, want in zip(t.vectors(), s.vectors()):
        np.testing.assert_array_equal(got, want)
