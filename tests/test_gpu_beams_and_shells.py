"""Models of beams and shells together: a plate with a line of beams on its mesh.
Their tangent is summed per colour (no rows are gathered), cleared along its
structure, and the nodal loads come with the residual scan.

Tangent and residual against the oracle with the bars of the plate's and the
chain's own tests (1e-12 of the largest tangent entry, 1e-11 of the largest
residual), node results of a static solve likewise (1e-8)."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu

TUBE = M.tube_section(0.02, 0.018)


def _stiffened(nq, line, seed=1, imperf=1e-4, p_max=2e5):
    """A clamped plate of nq x nq quads with beams along its mesh line `line`."""
    m, p, info = M.shell_plate(nq=nq, p_max=p_max, ramp="linear", n_steps=4, seed=seed, imperf=imperf)
    ng, j = info["ng"], 2 * line
    for i in range(0, ng - 2, 2):
        a = [j * ng + i, j * ng + i + 1, j * ng + i + 2]
        m.add_beam(*a, M.cs_rows([0, 1, 0], np.subtract(m.xyz[a[2]], m.xyz[a[0]])), 210e9, 0.3, 7850.0, *TUBE)
    return m, p, ng


@pytest.mark.parametrize("solver", [abi.GF_SOLVER_AUTO, abi.GF_SOLVER_BAND, abi.GF_SOLVER_FRONTS])
@pytest.mark.parametrize("nq,line,loaded", [(2, 1, 0), (4, 3, 5), (7, 2, 40)])
def test_assembly_matches_oracle(oracle_lib, nq, line, loaded, solver):
    m, _, ng = _stiffened(nq, line, seed=nq)
    m.gravity, m.gravity_on = (0.3, -0.5, -9.81), 1
    rng = np.random.default_rng(nq)
    if loaded:
        nodes = np.sort(rng.choice(m.n_nodes, loaded, replace=False))
        nodes[0] = 2 * line * ng + 1  # (a node of the beams and of shells)
        nodes = np.unique(nodes)
        for kind in (abi.GF_LOAD_NODAL, abi.GF_LOAD_NODAL_FOLLOWER):
            vals = np.zeros((len(nodes), 2, 6))
            vals[:, 1] = rng.normal(size=(len(nodes), 6)) * 50.0
            m.add_nodal_loads(kind, nodes, [0.0, 1.0], vals)
    om, dm = oracle_lib.OracleModel(m), runtime.DeviceModel(m, solver=solver)
    om.begin_solution(0.0, 1.0)
    dm.set_window(0.0, 1.0)
    for t_last, scale in ((0.3, 0.0), (0.6, 1e-4)):
        om.begin_step(t_last, 0.1)
        dm.begin_step(t_last, 0.1)
        d = rng.normal(size=(m.n_nodes, 6)) * scale
        om.write_disp(d)
        dm.write_disp(d)
        om.assemble()
        dm.assemble()
        norms = dm.assemble()  # (nothing of the first assembly is left)
        Ko, Kg, Ro, Rg = om.tangent_dense(), dm.tangent_dense(), om.residual(), dm.residual()
        assert np.abs(Kg - Ko).max() <= 1e-12 * np.abs(Ko).max()
        assert np.abs(Rg - Ro).max() <= 1e-11 * max(np.abs(Ro).max(), 1e-12 * np.abs(Ko).max())
        assert norms[0] == np.abs(Rg[:, :3]).max() and norms[1] == np.abs(Rg[:, 3:]).max()
    dm.close()


@pytest.mark.parametrize("solver", [abi.GF_SOLVER_BAND, abi.GF_SOLVER_FRONTS])
@pytest.mark.parametrize("precision", [abi.GF_PREC_FP64, abi.GF_PREC_MIXED])
def test_static_matches_oracle(oracle_lib, solver, precision):
    m, p, _ = _stiffened(5, 2)
    om = oracle_lib.OracleModel(m)
    ro, io = om.static_solve(p)
    dm = runtime.DeviceModel(m, precision=precision, solver=solver)
    rg, ig = dm.static_solve(p)
    assert rg.aborted == ro.aborted == 0
    assert len(ig) == len(io) and np.abs(ig - io).max() <= 1
    no, ng = om.nodes(), dm.nodes()
    moved = np.abs(no[:, :3] - m.freeze()["xyz"]).max()
    assert np.abs(ng[:, :3] - no[:, :3]).max() <= 1e-8 * moved
    assert np.abs(ng[:, 3:] - no[:, 3:]).max() <= 1e-8 * np.abs(no[:, 3:]).max()
    dm.close()


@pytest.mark.parametrize("nq", [24, 172])
def test_newton_contracts_in_the_last_rows(nq, device_holds):
    """172 x 172 quads: 618,684 free DOFs and 1.04 x 2^32 band entries, the beams in the
    last rows.  With the whole tangent Newton's increments square their relative size
    from one iteration to the next (the first is 2e-3 off at both sizes, so the fourth
    is far below 1e-9 of it); with the beams' terms at other entries they would fall by a
    constant factor."""
    m, _, _ = _stiffened(nq, nq - 1, imperf=0.0, p_max=2e2)
    device_holds(m)
    dm = runtime.DeviceModel(m)
    dm.set_window(0.0, 1.0)
    dm.begin_step(0.0, 1.0)
    inc = []
    for _ in range(4):
        dm.assemble()
        assert dm.solve() == 0
        inc.append(dm.update()[0])
    assert inc[3] <= 1e-9 * inc[0]
    if nq == 172:
        assert dm.info()["layout"] == 2 and dm.info()["factor_bytes"] > 2 ** 35
    dm.close()
