"""mugpu_cg_steps with a right-hand side in the range of the projector: the
directions of a chunk are kept until x is updated, and small-strain solves keep
the packed components of p and r inside a chunk.

x, r and p after every call equal those of the loop over mugpu_cg_step bit for
bit (the same arithmetic in the same order), at chunk lengths around the number
of directions kept and where the loop test stops inside a chunk.
"""
import ctypes

import numpy as np
import pytest

from muspectre_amd._device import DeviceBuffer
from test_gpu_abi_cell import GpuCell, _sphere_mask

pytestmark = pytest.mark.gpu

# grids just above the sizes from which the directions are kept, with compiled
# and run-time last axes and rows left over in a workgroup, and one below
CASES = [([48, 44, 45], 1), ([41, 48, 48], 1), ([80, 77, 76], 0), ([61, 60, 128], 0), ([1201, 1180], 1),
         ([1050, 1000], 0), ([9, 13, 15], 1)]


def _cell(capi, res, form):
    d = len(res)
    gc = GpuCell(capi, res, [1.0] * d, form, allow_even=int(any(n % 2 == 0 for n in res)))
    mask = _sphere_mask(res, max(2, min(res) / 3))
    mi, mo = gc.add_material(1, 100.0, .3), gc.add_material(1, 10.0, .3)
    idx = np.arange(mask.size)
    gc.add_pixels(mi, idx[mask.ravel()])
    gc.add_pixels(mo, idx[~mask.ravel()])
    capi.check(gc.lib.mugpu_cell_initialise(gc.h))
    F = np.zeros((gc.N, d * d)) + (np.eye(d).ravel() if form == 0 else 0.0)
    F[:, 1] += 0.01
    F[:, d] += 0.01
    gc.set_F(F)
    capi.check(gc.lib.mugpu_cell_evaluate_stress_tangent(gc.h))
    rhs = DeviceBuffer.from_array(np.random.default_rng(2).standard_normal((gc.N, gc.nc)))
    capi.check(gc.lib.mugpu_cell_apply_projection(gc.h, rhs.ptr))
    return gc, rhs


class _Solve:
    def __init__(self, capi, gc, rhs):
        self.capi, self.gc, self.n = capi, gc, gc.N * gc.nc
        self.v = [DeviceBuffer(8 * self.n) for _ in range(4)]  # x, r, p, Ap
        rr, bb = ctypes.c_double(), ctypes.c_double()
        x, r, p, Ap = (b.ptr for b in self.v)
        capi.check(gc.lib.mugpu_cg_start(gc.h, rhs.ptr, x, r, p, Ap, ctypes.byref(rr), ctypes.byref(bb)))
        self.it, self.rr = 0, rr.value

    def step(self):
        nr = ctypes.c_double()
        x, r, p, Ap = (b.ptr for b in self.v)
        self.capi.check(self.gc.lib.mugpu_cg_step(self.gc.h, int(self.it > 0), x, r, p, Ap, ctypes.byref(nr)))
        self.it, self.rr = self.it + 1, nr.value

    def steps(self, k, tol2):
        nr, done = ctypes.c_double(), ctypes.c_int()
        x, r, p, Ap = (b.ptr for b in self.v)
        self.capi.check(self.gc.lib.mugpu_cg_steps(self.gc.h, int(self.it > 0), x, r, p, Ap, tol2, k,
                                                   ctypes.byref(done), ctypes.byref(nr)))
        self.capi.check(self.gc.lib.mugpu_cg_finish(self.gc.h))
        self.it, self.rr = self.it + done.value, nr.value
        return done.value

    def vectors(self):
        return [b.download(self.n) for b in self.v[:3]]


@pytest.mark.parametrize("graphs", [0, 1], ids=["direct", "graph"])
@pytest.mark.parametrize("res,form", CASES, ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else str(v))
def test_chunks_equal_steps(capi, res, form, graphs):
    gc, rhs = _cell(capi, res, form)
    chunks = (1, 2, 8, 3, 9)
    ref, sol = _Solve(capi, gc, rhs), []
    rr = []
    for k in chunks:
        for _ in range(k):
            ref.step()
            rr.append(ref.rr)
        sol.append(ref.vectors())
    try:
        capi.check(gc.lib.mugpu_cg_graphs(graphs))
        for _ in range(2):
            s = _Solve(capi, gc, rhs)
            for k, want in zip(chunks, sol):
                assert s.steps(k, 0.0) == k
                for a, b in zip(s.vectors(), want):
                    np.testing.assert_array_equal(a, b)
            assert s.rr == rr[-1]
        # a stop inside the chunk, in each group of directions
        for stop in (1, 4, 8, 11):
            low = min(rr[:stop])
            if rr[stop - 1] != low or (stop > 1 and min(rr[:stop - 1]) == low):
                continue  # (r . r is not monotonic: the loop test stops earlier)
            t, want = _Solve(capi, gc, rhs), []
            for k in (stop, 5):
                for _ in range(k):
                    t.step()
                want.append(t.vectors())
            # (a cell runs one solve at a time)
            s = _Solve(capi, gc, rhs)
            assert s.steps(20, low) == stop
            for a, b in zip(s.vectors(), want[0]):
                np.testing.assert_array_equal(a, b)
            # and goes on from there
            s.steps(5, 0.0)
            for a, b in zip(s.vectors(), want[1]):
                np.testing.assert_array_equal(a, b)
    finally:
        capi.check(gc.lib.mugpu_cg_graphs(1))


@pytest.mark.parametrize("form", [0, 1], ids=["finite", "small"])
def test_ring_given_back(capi, form):
    """The directions' memory is given back on request between two calls; the
    solve goes on (without it, in full fields) to the same result within the
    rounding of 16 iterations' sums at a condition number near 10 (1e-12 of |x|;
    of |b| for r and p)."""
    gc, rhs = _cell(capi, [61, 96, 80] if form == 0 else [41, 48, 48], form)
    ref = _Solve(capi, gc, rhs)
    ref.steps(8, 0.0)
    ref.steps(8, 0.0)
    s = _Solve(capi, gc, rhs)
    s.steps(8, 0.0)
    capi.check(gc.lib.mugpu_release_cached())
    s.steps(8, 0.0)
    want, nb = ref.vectors(), np.linalg.norm(rhs.download(gc.N * gc.nc))
    for a, b, scale in zip(s.vectors(), want, (np.linalg.norm(want[0]), nb, nb)):
        assert np.linalg.norm(a - b) <= 1e-12 * scale
    # the next solve has its own again
    t = _Solve(capi, gc, rhs)
    t.steps(8, 0.0)
    t.steps(8, 0.0)
    for a, b in zip(t.vectors(), want):
        np.testing.assert_array_equal(a, b)
