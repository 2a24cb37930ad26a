"""Nodal loads beside the first beam launch and added by the residual scan: residual,
tangent and norms of a chain under dead and follower loads with forces and moments,
two on some nodes, one on the clamped node, against the oracle; loaded nodes that fill
a workgroup (64 or 128 lanes) less one, exactly and one more, in every layout.

The bars of the other assembly tests: 1e-12 of the largest tangent entry, 1e-11 of
the largest residual."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", [abi.GF_SOLVER_AUTO, abi.GF_SOLVER_BAND, abi.GF_SOLVER_FRONTS])
@pytest.mark.parametrize("loaded", [1, 63, 64, 65, 128, 129])
def test_loads_match_oracle(oracle_lib, loaded, solver):
    n = 70
    m, _, _ = M.cantilever_rollup(n_elem=n)
    rng = np.random.default_rng(loaded)
    m.loads = []
    nodes = np.sort(rng.choice(m.n_nodes, loaded, replace=False))
    nodes[0] = 0
    for kind, some in ((abi.GF_LOAD_NODAL_FOLLOWER, nodes), (abi.GF_LOAD_NODAL, nodes[::2]), (abi.GF_LOAD_NODAL, nodes)):
        vals = np.zeros((len(some), 2, 6))
        vals[:, 1] = rng.normal(size=(len(some), 6)) * 1e4
        m.add_nodal_loads(kind, some, [0.0, 1.0], vals)
    om, dm = oracle_lib.OracleModel(m), runtime.DeviceModel(m, solver=solver)
    om.begin_solution(0.0, 1.0)
    dm.set_window(0.0, 1.0)
    for t_last, scale in ((0.3, 0.0), (0.6, 1e-3)):
        om.begin_step(t_last, 0.1)
        dm.begin_step(t_last, 0.1)
        d = rng.normal(size=(m.n_nodes, 6)) * scale
        om.write_disp(d)
        dm.write_disp(d)
        om.assemble()
        dm.assemble()
        norms = dm.assemble()  # (again: the loads come once)
        Ko, Kg, Ro, Rg = om.tangent_dense(), dm.tangent_dense(), om.residual(), dm.residual()
        assert np.abs(Kg - Ko).max() <= 1e-12 * np.abs(Ko).max()
        assert np.abs(Rg - Ro).max() <= 1e-11 * np.abs(Ro).max()
        assert norms[0] == np.abs(Rg[:, :3]).max() and norms[1] == np.abs(Rg[:, 3:]).max()
    dm.close()
