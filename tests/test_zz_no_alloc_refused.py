"""gf_btdsystem_noalloc refuses a solution in the right-hand side's place, and a refused
call writes neither the solution nor the flag."""
import numpy as np
import pytest

from giraffe_amd import abi, runtime
from test_zz_no_alloc import DevBuf, _hip, _system

pytestmark = pytest.mark.gpu


def test_solution_over_the_right_hand_side():
    m, nblk = 6, 40
    hip, L = _hip(), runtime.load()
    A, B, C, b = _system(m, nblk, 5)
    bufs = [DevBuf(hip, v) for v in (A, B, C, b, np.full(1, -1, np.int32))]
    d = [q.p for q in bufs]
    assert L.gf_btdsystem_noalloc(m, nblk, d[0], d[1], d[2], d[3], d[3], d[4], None) == abi.GF_E_ARG
    assert hip.hipDeviceSynchronize() == 0
    assert int(bufs[4].get()[0]) == -1 and np.array_equal(bufs[3].get(), b)
    for q in bufs:
        q.free()
