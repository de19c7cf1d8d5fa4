"""Downloads around the sizes at which the pinned ring takes over: below it, at
it, a last block that is short, exactly the ring's 16 blocks and several times
round it; twice in a row, and again after the ring was given back.  The values
are those uploaded, bit for bit."""
import numpy as np
import pytest

from muspectre_amd._device import DeviceBuffer

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("nbytes", [8, 2 * MB - 8, 2 * MB, 3 * MB + 8, 16 * MB, 16 * MB + 8, 67 * MB - 8])
def test_download_sizes(capi, nbytes):
    a = np.random.default_rng(nbytes).integers(0, 2 ** 63, nbytes // 8)
    buf = DeviceBuffer.from_array(a)
    for _ in range(2):
        np.testing.assert_array_equal(buf.download(a.shape, a.dtype), a)
    capi.check(capi.load().mugpu_release_cached())
    np.testing.assert_array_equal(buf.download(a.shape, a.dtype), a)


def test_result_fields_are_fresh_arrays(capi):
    """Every read of a result field is an array of its own; an assigned one is
    read back."""
    import muspectre_amd as mu
    cell = mu.Cell([15, 13], [1.0, 1.0], mu.Formulation.small_strain)
    m = mu.material.MaterialLinearElastic1_2d.make(cell, "m", 10.0, 0.3)
    m.add_pixels_by_index(np.arange(15 * 13))
    solver = mu.solvers.SolverCG(cell, 1e-8, 50, False)
    r = mu.solvers.newton_cg(cell, [np.array([[0.01, 0.0], [0.0, 0.0]])], solver, 1e-5, 1e-10, 0)[0]
    a, b = r.grad, r.grad
    assert a.shape == (15 * 13 * 4, 1) and a is not b
    np.testing.assert_array_equal(a, b)
    a[:] = 7.0
    np.testing.assert_array_equal(r.grad, b)
    r.stress = a
    np.testing.assert_array_equal(r.stress, a)
