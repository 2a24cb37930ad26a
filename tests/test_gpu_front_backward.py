"""The fronts' backward substitution in one launch a level (front_bwd_kernel, chosen
where (own blocks - 1) x update blocks <= 8) beside the two-launch form: Newton
increments of plates whose plans hold single blocks, roots of 1 to 6 blocks without
an update part, fronts of one own block, and levels on both sides of the rule, in
FP64 and with FP32 factors refined in FP64, against the band LU.

The equilibrated condition is below 1e7 here: both solves agree to 1e7 eps times a
growth of a few, 1e-8."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [abi.GF_PREC_FP64, abi.GF_PREC_MIXED])
@pytest.mark.parametrize("nq", [1, 2, 3, 4, 6, 12, 24, 40])
def test_backward_matches_band(nq, precision):
    m, _, _ = M.shell_plate(nq=nq, seed=nq)
    xs = []
    for solver, prec in ((abi.GF_SOLVER_FRONTS, precision), (abi.GF_SOLVER_BAND, abi.GF_PREC_FP64)):
        dm = runtime.DeviceModel(m, solver=solver, precision=prec)
        dm.set_window(0.0, 1.0)
        dm.begin_step(0.0, 0.2)
        dm.assemble()
        assert dm.solve() == 0
        xs.append(dm.increment())
        dm.close()
    assert np.abs(xs[0] - xs[1]).max() <= 1e-8 * np.abs(xs[1]).max()
