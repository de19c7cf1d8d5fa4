"""The memory of kept CG directions is bounded over all cells: a solve that needs
more takes it from the cells whose latest solve began first, and a cell that
lost its directions takes them anew for its next solve, with the same result.
"""
import numpy as np
import pytest

from test_gpu_cg_ring import _cell, _Solve
from test_gpu_cg_ring_length import _kept

pytestmark = pytest.mark.gpu


def test_total_is_bounded(capi):
    res = [48, 48, 48]
    one = 8 * int(np.prod(res)) * 6 * 9  # eight directions and r, packed
    cells = [_cell(capi, res, 1) for _ in range(3)]
    lib = cells[0][0].lib

    def solve(i):
        s = _Solve(capi, *cells[i])
        s.steps(8, 0.0)
        s.steps(3, 0.0)
        return s.vectors()

    def kept():
        return [_kept(capi, gc)[0] for gc, _ in cells]

    try:
        capi.check(lib.mugpu_debug_kept_bytes(2 * one + 1000))
        first = [solve(0), solve(1)]
        assert kept() == [8, 8, 0]
        solve(0)
        solve(2)  # cell 1 has been idle longest
        assert kept() == [8, 0, 8]
        for got, want in zip(solve(1), first[1]):
            np.testing.assert_array_equal(got, want)
        assert kept() == [0, 8, 8]
        # room for half as many only, then for none
        for total, n in ((one - 1000, 4), (1000, 0)):
            capi.check(lib.mugpu_debug_kept_bytes(total))
            assert kept() == [0, 0, 0]
            got = solve(0)
            assert kept() == [n, 0, 0]
            if n:
                for a, b in zip(got, first[0]):
                    np.testing.assert_array_equal(a, b)
    finally:
        capi.check(lib.mugpu_debug_kept_bytes(0))
