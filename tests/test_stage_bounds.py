"""CPU check of the index arithmetic of the r2c pass over packed small-strain CG
vectors (sym_stage in op_stages.hpp): on grids with every number of rows per
workgroup and every remainder of rows in the last one, what a chunk's first
iteration reads from p and r lies inside the fields, and reaches their ends.
"""
import ctypes

import numpy as np
import pytest


def _reads(res):
    from muspectre_amd import _capi
    lo, hi, rb = ctypes.c_int64(), ctypes.c_int64(), ctypes.c_int()
    _capi.check(_capi.load().mugpu_debug_stage_reads(
        len(res), (ctypes.c_int * len(res))(*res), ctypes.byref(lo), ctypes.byref(hi), ctypes.byref(rb)))
    return lo.value, hi.value, rb.value


def _check(res):
    d, n = len(res), res[-1]
    N = int(np.prod(res))
    lo, hi, rb = _reads(res)
    rows = N // n
    assert lo == (rows - 1) // rb * rb * n * d * d, res
    assert hi == N * d * d - 1, res
    return rb, rows % rb


@pytest.mark.parametrize("res", [[65, 65, 63], [67, 67, 67], [75, 75, 75], [81, 81, 81], [99, 99, 99], [111, 111, 111],
                                 [65, 66, 63], [99, 75, 63], [101, 101, 35], [105, 135, 77], [255, 255, 21],
                                 [128, 256, 40], [48, 44, 45], [41, 48, 48], [7, 9, 16], [51, 51], [4001, 255],
                                 [4099, 7]], ids=lambda r: "x".join(map(str, r)))
def test_reads_inside_the_fields(res):
    _check(res)


def test_every_remainder_of_rows():
    seen = set()
    for n in list(range(3, 120, 2)) + [16, 20, 24, 32, 40, 48, 60, 64, 72, 80, 96, 100, 125, 128, 175, 256, 512]:
        for rows in (1, 2, 3, 5, 63, 1023, *range(4096, 4113), *range(16384, 16401)):
            for res in ([rows, n], [rows, 1, n]):
                seen.add(_check(res))
    for rb in (2, 4, 6, 8, 10, 12, 16):
        assert all((rb, m) in seen for m in range(rb)), rb
