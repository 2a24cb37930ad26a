"""A shell model whose rows hold more entries than the assembly by rows takes (255):
its tangent is summed per colour.  A disc of triangles around one node, with rows
of 159 and 255 entries, which fit, and of more.  Bars as of the plate's own tests."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu


def _disc(k):
    """k triangles around node 0; rim clamped."""
    m = M.Model("disc")
    w = 2.0 * np.pi * np.arange(k) / k
    rim = np.stack([np.cos(w), np.sin(w), 0.0 * w], 1)
    rng = np.random.default_rng(k)
    hub = np.array([0.0, 0.0, 0.01])
    m.add_nodes(hub)
    m.add_nodes(rim)                                      # 1 .. k
    m.add_nodes(0.5 * (rim + hub))                        # k + 1 .. 2 k, spokes
    m.add_nodes(0.5 * (rim + np.roll(rim, -1, axis=0)))   # 2 k + 1 .. 3 k, rim mid-sides
    elems = []
    for i in range(k):
        j = (i + 1) % k
        m.add_shell([0, 1 + i, 1 + j, 1 + k + i, 1 + 2 * k + i, 1 + k + j], 70e9, 0.33, 2700.0, 0.005)
        elems.append(i)
    for i in range(k):
        if rng.uniform() < 0.3:
            m.fix_dofs(1 + i, [0, 1, 2])
    m.fix_dofs(1, [0, 1, 2])
    m.fix_dofs(2, [0, 1, 2])
    m.fix_dofs(1 + k // 2, [0, 1, 2])
    m.add_load(abi.GF_LOAD_SHELL_PRESSURE, elems, [0.0, 1.0], [[0.0] * 6, [1e3, 0, 0, 0, 0, 0]], flags=1)
    m.gravity, m.gravity_on = (0.0, 0.3, -9.81), 1
    return m


@pytest.mark.parametrize("k", [12, 18, 19, 24, 40])
def test_hub_matches_oracle(oracle_lib, k):
    m = _disc(k)
    om, dm = oracle_lib.OracleModel(m), runtime.DeviceModel(m, solver=abi.GF_SOLVER_FRONTS)
    om.begin_solution(0.0, 1.0)
    dm.set_window(0.0, 1.0)
    rng = np.random.default_rng(k)
    for t_last, scale in ((0.3, 0.0), (0.6, 1e-4)):
        om.begin_step(t_last, 0.1)
        dm.begin_step(t_last, 0.1)
        d = rng.normal(size=(m.n_nodes, 6)) * scale
        om.write_disp(d)
        dm.write_disp(d)
        om.assemble()
        dm.assemble()
        dm.assemble()  # (nothing of the first assembly is left)
        Ko, Kg, Ro, Rg = om.tangent_dense(), dm.tangent_dense(), om.residual(), dm.residual()
        assert np.abs(Kg - Ko).max() <= 1e-12 * np.abs(Ko).max()
        assert np.abs(Rg - Ro).max() <= 1e-11 * max(np.abs(Ro).max(), 1e-12 * np.abs(Ko).max())
    dm.close()
