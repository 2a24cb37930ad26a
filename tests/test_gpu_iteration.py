"""The launches of a Newton iteration whose form depends on the size: the beam
assembly (two wavefronts a workgroup while a colour's workgroups of 7 elements
number at most 512) and the residual scan, whose last workgroup hands the scalar
block to the host.

Residuals are held to the oracle at 1e-11 of the largest entry, the bar of the
other assembly tests; norms to the residual's own maxima exactly; and the norms of
repeated assemblies and iterations to those of the first."""
import numpy as np
import pytest

from giraffe_amd import model as M, runtime

pytestmark = pytest.mark.gpu


# one element, a workgroup less one, full and one more; the last split colour, and
# the first that is not (7,168 elements in two colours)
@pytest.mark.parametrize("n", [1, 13, 14, 15, 7168, 7170])
def test_residual_matches_oracle(oracle_lib, n):
    m, p, _ = M.cantilever_rollup(n_elem=n, L=0.5 * n)
    d = np.random.default_rng(n).normal(scale=1e-4, size=(m.n_nodes, 6))
    d[0] = 0.0
    dm, om = runtime.DeviceModel(m), oracle_lib.OracleModel(m)
    dm.set_window(0.0, 1.0)
    om.begin_solution(0.0, 1.0)
    dm.begin_step(0.0, 0.1)
    om.begin_step(0.0, 0.1)
    dm.write_disp(d)
    om.write_disp(d)
    rg, ro = dm.assemble(), om.assemble()
    g, o = dm.residual(), om.residual()
    assert np.abs(g - o).max() <= 1e-11 * np.abs(o).max()
    assert rg[2] == 0.0 and ro[2] == 0.0
    assert rg[0] == np.abs(g[:, :3]).max() and rg[1] == np.abs(g[:, 3:]).max()
    if n <= 15:
        Kg, Ko = dm.tangent_dense(), om.tangent_dense()
        assert np.abs(Kg - Ko).max() <= 1e-11 * np.abs(Ko).max()


@pytest.mark.parametrize("n", [3, 40, 700])
def test_norms_do_not_depend_on_what_ran_before(n):
    """The step-by-step calls and whole solves leave the scalar block in either
    state; every order of them gives the same norms and the same solution."""
    m, p, _ = M.cantilever_rollup(n_elem=n, n_steps=3, turns=0.1)
    dm = runtime.DeviceModel(m)

    def pieces():
        dm.reset()
        dm.set_window(0.0, 1.0)
        dm.begin_step(0.0, 0.1)
        out = [dm.assemble()]
        out += [np.array([dm.solve()]), dm.update(), dm.assemble()]
        dm.rollback()
        return np.concatenate(out)

    def whole():
        dm.reset()
        rep, it = dm.static_solve(p)
        return np.concatenate([[rep.converged_steps, rep.total_solves], it, dm.nodes().ravel()])

    a, b = pieces(), whole()
    for _ in range(2):
        assert np.array_equal(whole(), b)
        assert np.array_equal(pieces(), a)
        assert np.array_equal(pieces(), a)
        assert np.array_equal(whole(), b)
