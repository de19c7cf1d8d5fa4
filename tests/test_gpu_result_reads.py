"""A result field is downloaded once or twice and then read from the host: its
values are the same at every read, a write replaces them, and a read after that
costs less than downloading the field (the ratio is 0.02 for the small field and
about 0.35 for the large one).
"""
import ctypes
import time

import numpy as np
import pytest

from muspectre_amd._device import DeviceBuffer

pytestmark = pytest.mark.gpu


def _median(f, reps=31):
    t = []
    for _ in range(reps):
        t0 = time.perf_counter()
        f()
        t.append(time.perf_counter() - t0)
    return float(np.median(t))


@pytest.mark.parametrize("res", [[51, 51], [41, 41, 41]], ids=lambda r: "x".join(map(str, r)))
def test_repeated_reads(capi, res):
    import muspectre_amd as mu
    d, N = len(res), int(np.prod(res))
    cell = mu.Cell(res, [1.0] * d, mu.Formulation.small_strain)
    make = getattr(mu.material, "MaterialLinearElastic1_{}d".format(d)).make
    a, b = make(cell, "a", 100.0, .3), make(cell, "b", 10.0, .3)
    idx = np.arange(N)
    a.add_pixels_by_index(idx[::3])
    b.add_pixels_by_index(idx[idx % 3 > 0])
    load = np.zeros((d, d))
    load[0, 1] = load[1, 0] = .01
    r = mu.solvers.newton_cg(cell, load, mu.solvers.SolverCG(cell, 1e-6, 500, False), 1e-5, 1e-10, 0)
    first = r.stress
    for _ in range(3):
        np.testing.assert_array_equal(r.stress, first)
    buf, out = DeviceBuffer.from_array(first), np.empty_like(first)
    down = _median(lambda: capi.check(capi.load().mugpu_download(
        out.ctypes.data_as(ctypes.c_void_p), buf.ptr, out.nbytes)))
    assert _median(lambda: r.stress) < 0.7 * down
    r.stress = 2 * first
    np.testing.assert_array_equal(r.stress, 2 * first)
