"""Chunks of CG iterations where the device has room for four directions instead of
eight, or for none (x then rides on the next iteration's first pass, also in a
solve that starts so): x, r and p equal those of single steps bit for bit, at
chunk lengths around the four and where the loop test stops at the end of a
group of directions and inside one.
"""
import ctypes

import numpy as np
import pytest

from test_gpu_cg_ring import _cell, _Solve

pytestmark = pytest.mark.gpu


def _kept(capi, gc):
    n, k = ctypes.c_int(), ctypes.c_int()
    capi.check(gc.lib.mugpu_cell_kept_directions(gc.h, ctypes.byref(n), ctypes.byref(k)))
    return n.value, k.value


@pytest.mark.parametrize("graphs", [0, 1], ids=["direct", "graph"])
@pytest.mark.parametrize("most", [8, 4, 0])
@pytest.mark.parametrize("res,form", [([48, 44, 45], 1), ([41, 48, 48], 1), ([80, 77, 76], 0), ([61, 60, 128], 0),
                                      ([1470, 952], 1)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else str(v))
def test_fewer_directions(capi, res, form, most, graphs):
    gc, rhs = _cell(capi, res, form)
    d = len(res)
    chunks = (3, 4, 5, 8, 9)
    try:
        capi.check(gc.lib.mugpu_debug_kept_directions(most))
        capi.check(gc.lib.mugpu_cg_graphs(graphs))
        ref, rr, sol = _Solve(capi, gc, rhs), [], []
        assert _kept(capi, gc) == (most, d * (d + 1) // 2 if form == 1 and most else d * d)
        for _ in range(sum(chunks)):
            ref.step()
            rr.append(ref.rr)
            sol.append(ref.vectors())
        s = _Solve(capi, gc, rhs)
        done = 0
        for k in chunks:
            assert s.steps(k, 0.0) == k
            done += k
            assert s.rr == rr[done - 1]
            for got, want in zip(s.vectors(), sol[done - 1]):
                np.testing.assert_array_equal(got, want)
        for stop in (1, 3, 4, 5, 8, 9):
            if stop > 1 and rr[stop - 1] >= min(rr[:stop - 1]):
                continue  # (r . r is not monotonic: the loop test stops earlier)
            s = _Solve(capi, gc, rhs)
            assert s.steps(12, rr[stop - 1]) == stop and s.rr == rr[stop - 1]
            for got, want in zip(s.vectors(), sol[stop - 1]):
                np.testing.assert_array_equal(got, want)
            s.steps(5, 0.0)
            for got, want in zip(s.vectors(), sol[stop + 4]):
                np.testing.assert_array_equal(got, want)
    finally:
        capi.check(gc.lib.mugpu_cg_graphs(1))
        capi.check(gc.lib.mugpu_debug_kept_directions(8))
