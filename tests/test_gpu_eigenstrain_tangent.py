"""Finite-strain tangents of MaterialLinearElastic2 with eigenstrains that are not
symmetric: the PK2 stress is then not symmetric either, nor is the tangent
(dP = dF S + F dS takes S itself), so neither the factors of LE1-4 nor a
triangle of the matrix can stand for it.

Tolerance: 1e-12 of the largest entry, as in test_gpu_tangent_factors.py.
"""
import numpy as np
import pytest

from test_gpu_abi_cell import GpuCell
from test_gpu_tangent_factors import _check, _rotation

pytestmark = pytest.mark.gpu


def _cells(capi, oracle, res, prec=0):
    """LE2 on every other voxel, one eigenstrain in three nonsymmetric, LE1 between."""
    d, N = len(res), int(np.prod(res))
    even = int(any(n % 2 == 0 for n in res))
    oc = oracle.Cell(res, [1.0] * d, 0, allow_even=bool(even))
    gc = GpuCell(capi, res, [1.0] * d, 0, prec, allow_even=even)
    rng = np.random.default_rng(N)
    for fam in (1, 2):
        mo, mg = oc.add_material(fam, 100.0, 0.3), gc.add_material(fam, 100.0, 0.3)
        idx = np.arange(fam - 1, N, 2)
        par = None
        if fam == 2:
            t = 0.02 * rng.standard_normal((len(idx), d, d))
            t[np.arange(len(idx)) % 3 > 0] += t[np.arange(len(idx)) % 3 > 0].transpose(0, 2, 1)
            par = np.ascontiguousarray(t.reshape(len(idx), -1))
        for k, i in enumerate(idx):
            oc.add_pixel(mo, int(i)) if par is None else oc.add_pixel(mo, int(i), par[k])
        gc.add_pixels(mg, idx, par)
    F = np.stack([(_rotation(rng, d) @ (np.eye(d) + 0.1 * rng.standard_normal((d, d)))).ravel(order="F")
                  for _ in range(N)])
    return oc, gc, F


@pytest.mark.parametrize("res", [[7, 9], [32, 16]], ids=lambda r: "x".join(map(str, r)))
def test_nonsymmetric_eigenstrain_2d(capi, oracle, res):
    oc, gc, F = _cells(capi, oracle, res)
    _check(capi, oc, gc, F, 1)


@pytest.mark.parametrize("prec", [0, 1], ids=["fp64", "fp32"])
@pytest.mark.parametrize("res", [[5, 3, 7], [3, 5, 16]], ids=lambda r: "x".join(map(str, r)))
def test_nonsymmetric_eigenstrain_3d(capi, oracle, res, prec):
    """(an FP32 cell's material stage, tangent and FP64 operator)"""
    oc, gc, F = _cells(capi, oracle, res, prec)
    _check(capi, oc, gc, F, 1)
