"""Shell element records by 16, 32 and 64 points a wavefront (up to 5,461 and 10,922
elements, and above), element matrices and pressure records with full and ragged last
workgroups (four and seven elements each), against the oracle: residual and Newton
increment of strips two cells wide, clamped along both edges.

The residual is a sum of at most 8 elements' forces, each below 60 times the
tangent's largest entry (bounded by the largest force a unit displacement gives,
E t, here below 2e9) times the displacements: 1e-13 of that.  The increment solves
a tangent of condition below 2e7 (4 to 61 elements, from the oracle's; the strip's own
length adds nothing, its edges are held): 2e7 eps and a growth of a few, 2e-8."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu


def _strip(ne):
    """ne elements: cells of 0.1 m, two a column, the last element of an odd ne left out."""
    m = M.Model("strip")
    nx, h = (ne + 3) // 4, 0.05
    ngx = 2 * nx + 1
    ii, jj = np.meshgrid(np.arange(ngx), np.arange(5), indexing="ij")
    m.add_nodes(np.stack([ii * h, jj * h, 0.0 * ii], axis=-1).reshape(-1, 3))

    def nid(i, j):
        return 5 * i + j

    conn = []
    for p in range(nx):
        for q in range(2):
            i, j = 2 * p, 2 * q
            conn.append([nid(i, j), nid(i + 2, j), nid(i + 2, j + 2), nid(i + 1, j), nid(i + 2, j + 1),
                         nid(i + 1, j + 1)])
            conn.append([nid(i, j), nid(i + 2, j + 2), nid(i, j + 2), nid(i + 1, j + 1), nid(i + 1, j + 2),
                         nid(i, j + 1)])
    for c in conn[:ne]:
        m.add_shell(c, 70e9, 0.33, 2700.0, 0.005)
    for i in range(ngx):
        for j in (0, 4):
            m.fix_dofs(nid(i, j), range(6))
    m.add_load(abi.GF_LOAD_SHELL_PRESSURE, range(ne), [0.0, 1.0],
               [[0.0] * 6, [1e4, 0, 0, 0, 0, 0]], flags=ne % 2)
    return m


@pytest.mark.parametrize("ne", [4, 7, 9, 5461, 5462, 10923])
def test_records_match_oracle(oracle_lib, ne):
    m = _strip(ne)
    d = np.random.default_rng(ne).normal(size=(m.n_nodes, 6)) * 1e-5
    res = []
    for x in (oracle_lib.OracleModel(m), runtime.DeviceModel(m, solver=abi.GF_SOLVER_FRONTS)):
        (x.begin_solution if hasattr(x, "begin_solution") else x.set_window)(0.0, 1.0)
        x.begin_step(0.4, 0.1)
        x.write_disp(d)
        x.assemble()
        r = x.residual()
        assert not x.solve()
        x.update()
        res.append((r, x.increment()))
    (ro, xo), (rg, xg) = res
    assert np.abs(rg - ro).max() <= 1e-13 * (60.0 * 2e9 * np.abs(d).max() + np.abs(ro).max())
    assert np.abs(xg - xo).max() <= 2e-8 * np.abs(xo).max()
