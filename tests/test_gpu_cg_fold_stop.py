"""CG chunks whose scalars are folded into the passes, stopped by the loop test at
every iteration of a chunk, on compiled last axes and up to the largest number of
workgroups that fold (the launch that finds the loop over also clears the flag
which its own workgroups start from): x, r and p equal those of single steps bit
for bit, and the solve goes on from there.
"""
import numpy as np
import pytest

from test_gpu_cg_ring import _cell, _Solve

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graphs", [0, 1], ids=["direct", "graph"])
@pytest.mark.parametrize("res,form", [([64, 64, 64], 0), ([64, 64, 64], 1), ([32, 16, 32], 1), ([512, 512], 1),
                                      ([256, 256], 0), ([16, 64], 0), ([45, 32, 64], 1)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, list) else str(v))
def test_every_stop(capi, res, form, graphs):
    gc, rhs = _cell(capi, res, form)
    ref, rr, sol = _Solve(capi, gc, rhs), [], []
    for _ in range(11):
        ref.step()
        rr.append(ref.rr)
        sol.append(ref.vectors())
    try:
        capi.check(gc.lib.mugpu_cg_graphs(graphs))
        stops = 0
        for k in range(1, 10):
            if k > 1 and rr[k - 1] >= min(rr[:k - 1]):
                continue  # (r . r is not monotonic: the loop test stops earlier)
            stops += 1
            s = _Solve(capi, gc, rhs)
            assert s.steps(10, rr[k - 1]) == k and s.rr == rr[k - 1]
            for got, want in zip(s.vectors(), sol[k - 1]):
                np.testing.assert_array_equal(got, want)
            assert s.steps(2, 0.0) == 2 and s.rr == rr[k + 1]
            for got, want in zip(s.vectors(), sol[k + 1]):
                np.testing.assert_array_equal(got, want)
        assert stops >= 3
    finally:
        capi.check(gc.lib.mugpu_cg_graphs(1))
