"""Fronts of more than 4 GB: a plate whose nodes are numbered at random and lie at one
coordinate of its largest extent (a beam far out makes that extent), so that bisection
finds no separator and the plan is a chain of supernodes whose update rows are most of
the plate.  42 x 42 quads: 25,920 rows in the largest front, whose parent gathers entries up to
5.2 GB from the first, 88 GB of fronts in all.

With the whole tangent Newton's increments square their relative size from one iteration to
the next (about 2e-3 after the first), so the fourth is far below 1e-9 of the first; a
solve that gathers other entries does not get there."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime
from renumber import renumber

pytestmark = pytest.mark.gpu


def scattered_plate(nq, seed=0):
    m, _, _ = M.shell_plate(nq=nq, imperf=0.0, p_max=2e2, ramp="linear")
    m.xyz = [[z, x, y] for x, y, z in m.xyz]  # the plate in the plane of one x
    m = renumber(m, np.random.default_rng(seed).permutation(m.n_nodes))
    i0 = m.add_nodes([[50.0, 0.0, 0.0], [50.5, 0.0, 0.0], [51.0, 0.0, 0.0]])
    m.add_beam(i0, i0 + 1, i0 + 2, M.cs_rows([0, 1, 0], [1, 0, 0]), 210e9, 0.3, 7850.0, *M.tube_section(0.02, 0.018))
    m.fix_dofs(i0, range(6))
    return m


@pytest.mark.parametrize("nq", [6, 20, 42])
def test_newton_contracts(nq, device_holds):
    m = scattered_plate(nq)
    device_holds(m, solver=abi.GF_SOLVER_FRONTS)
    if nq == 42:
        fr = runtime.front_plan(m)["front"].astype(np.int64)
        kp, mp = fr[:, 1], fr[:, 2]
        assert ((mp - kp) * mp * 8).max() > 2 ** 32
    dm = runtime.DeviceModel(m, solver=abi.GF_SOLVER_FRONTS)
    dm.set_window(0.0, 1.0)
    dm.begin_step(0.0, 1.0)
    inc = []
    for _ in range(4):
        dm.assemble()
        assert dm.solve() == 0
        inc.append(dm.update()[0])
    assert inc[0] > 0.0 and inc[3] <= 1e-9 * inc[0]
    dm.close()
