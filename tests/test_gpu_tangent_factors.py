"""Tangents kept as factors (FP64 finite strain: cells of LE1-4 alone, 3D cells
of the consistent HyperElastoPlastic1 alone) against the oracle's matrices:
every law in one cell, large rotations (each branch of the rotation's
quaternion), stretches whose principal values coincide or nearly do, elastic
and plastic voxels, and a voxel count that ends inside a tangent block of 64.

Tolerance: 1e-12 of the largest entry, as in test_gpu_abi_cell.py.
"""
import numpy as np
import pytest

from muspectre_amd._device import DeviceBuffer
from test_gpu_abi_cell import GpuCell, _arr

pytestmark = pytest.mark.gpu


def _rotation(rng, d):
    q, r = np.linalg.qr(rng.standard_normal((d, d)))
    q = q * np.sign(np.diag(r))
    if np.linalg.det(q) < 0:
        q[:, 0] *= -1
    return q


def _check(capi, oc, gc, F, seed):
    N, nc = gc.N, gc.nc
    oc.initialise()
    capi.check(gc.lib.mugpu_cell_initialise(gc.h))
    oc.F[:] = F
    gc.set_F(F)
    oc.evaluate_stress_tangent()
    capi.check(gc.lib.mugpu_cell_evaluate_stress_tangent(gc.h))
    assert np.abs(gc.get("P") - oc.P).max() <= 1e-12 * np.abs(oc.P).max()
    K = np.zeros((N, nc * nc))
    capi.check(gc.lib.mugpu_cell_get_tangent(gc.h, _arr(K)))
    assert np.abs(K - oc.K).max() <= 1e-12 * np.abs(oc.K).max()
    dF = np.random.default_rng(seed).standard_normal((N, nc))
    bi, bo = DeviceBuffer.from_array(dF), DeviceBuffer(dF.nbytes)
    capi.check(gc.lib.mugpu_cell_tangent_product(gc.h, bi.ptr, bo.ptr))
    # K(r, c) at r + nc c
    ref = np.einsum("vcr,vc->vr", oc.K.reshape(N, nc, nc), dF)
    assert np.abs(bo.download(dF.shape) - ref).max() <= 1e-12 * np.abs(ref).max()
    ref = oc.directional_stiffness(dF)
    capi.check(gc.lib.mugpu_cell_directional_stiffness(gc.h, bi.ptr, bo.ptr))
    assert np.abs(bo.download(dF.shape) - ref).max() <= 1e-12 * np.abs(ref).max()


@pytest.mark.parametrize("res", [[7, 9], [32, 16], [5, 3, 7], [3, 5, 16]], ids=lambda r: "x".join(map(str, r)))
def test_linear_elastic_factors(capi, oracle, res):
    d, N = len(res), int(np.prod(res))
    even = int(any(n % 2 == 0 for n in res))
    oc = oracle.Cell(res, [1.0] * d, 0, allow_even=bool(even))
    gc = GpuCell(capi, res, [1.0] * d, 0, allow_even=even)
    rng = np.random.default_rng(N)
    for fam in (1, 2, 3, 4):
        E, nu = (100.0 + fam, 0.3) if fam < 3 else (0.0, 0.0)
        mo, mg = oc.add_material(fam, E, nu), gc.add_material(fam, E, nu)
        idx = np.arange(fam - 1, N, 4)
        par = (None if fam == 1 else 0.01 * rng.standard_normal((len(idx), d * d)) if fam == 2
               else np.stack([rng.uniform(50, 200, len(idx)), rng.uniform(0.1, 0.4, len(idx))], 1))
        if fam == 2:  # symmetric eigenstrains
            t = par.reshape(-1, d, d)
            par = np.ascontiguousarray((t + t.transpose(0, 2, 1)).reshape(len(idx), -1))
        for k, i in enumerate(idx):
            oc.add_pixel(mo, int(i)) if par is None else oc.add_pixel(mo, int(i), par[k])
        gc.add_pixels(mg, idx, par)
    F = np.stack([(_rotation(rng, d) @ (np.eye(d) + 0.1 * rng.standard_normal((d, d)))).ravel(order="F")
                  for _ in range(N)])
    _check(capi, oc, gc, F, 1)


@pytest.mark.parametrize("res", [[5, 3, 7], [3, 5, 16]], ids=lambda r: "x".join(map(str, r)))
def test_consistent_hep1_factors(capi, oracle, res):
    N = int(np.prod(res))
    even = int(any(n % 2 == 0 for n in res))
    oc = oracle.Cell(res, [1.0] * 3, 0, allow_even=bool(even))
    gc = GpuCell(capi, res, [1.0] * 3, 0, allow_even=even)
    rng = np.random.default_rng(N)
    mo = oc.add_material(6, 210.0, 0.33, 0.8, 1.0)
    mg = gc.add_material(6, 210.0, 0.33, 0.8, 1.0)
    for i in range(N):
        oc.add_pixel(mo, i)
    gc.add_pixels(mg, np.arange(N))
    F = []
    for i in range(N):
        kind = i % 4
        if kind == 0:    # plastic, distinct stretches
            lam = 1.0 + np.array([0.02, -0.01, 0.005]) * rng.uniform(0.5, 2, 3)
        elif kind == 1:  # elastic
            lam = 1.0 + 1e-3 * rng.standard_normal(3)
        elif kind == 2:  # two equal
            lam = np.array([1.02, 0.99, 0.99])
        else:            # nearly equal
            lam = 1.01 + np.array([0.02, 1e-9, 2e-9])
        R, V = _rotation(rng, 3), _rotation(rng, 3)
        F.append((R @ V @ np.diag(lam[rng.permutation(3)]) @ V.T).ravel(order="F"))
    _check(capi, oc, gc, np.stack(F), 2)
