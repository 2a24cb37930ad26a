"""The multifrontal step kernel's items against the band LU: one Newton increment of
plates whose launches take each form of item -- update items of one tile row and
of up to four (from about 2,304 tiles a row on: the 90 x 90 plate's leaves),
own blocks of which 16, 32, 48 or 64 rows are live, update tiles first formed from
none, one and two children.

Both are backward stable solves of the same tangent, whose equilibrated condition
is below 1e7 at 90 x 90: the increments agree to 1e7 eps times a growth of a few,
1e-8."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu


def _increment(m, solver):
    dm = runtime.DeviceModel(m, solver=solver)
    dm.set_window(0.0, 1.0)
    dm.begin_step(0.0, 0.2)
    dm.assemble()
    assert dm.solve() == 0
    x = dm.increment()
    dm.close()
    return x


@pytest.mark.parametrize("nq", [3, 7, 10, 21, 33, 90])
def test_fronts_match_band(nq):
    m, _, _ = M.shell_plate(nq=nq, seed=nq)
    x = _increment(m, abi.GF_SOLVER_FRONTS)
    ref = _increment(m, abi.GF_SOLVER_BAND)
    assert np.abs(x - ref).max() <= 1e-8 * np.abs(ref).max()
