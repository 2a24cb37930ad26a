"""Shell assembly by rows (shell_gather_kernel: multifrontal models of shells alone)
against the scatter per colour, which the band solver keeps: tangent and residual
of two states of plates with and without pressure, gravity and nodal loads (dead
and follower), blocks of which none to all rows are constrained, and nodes that
one to eight elements share (four are in flight at once).

Both add the same at most nine numbers an entry, the nodal loads last instead of
first: they differ by at most 8 roundings of a partial sum.  A tangent entry's
terms do not exceed a few times the largest entry: 8 * 8 * 2.2e-16 of it, 1e-13.
A residual entry's are 27 products of tangent entries and displacements, below 60
with the second order of the stretch, and the loads: 1e-13 * 60 of the largest
entry times the largest displacement, plus 1e-13 of the largest residual."""
import numpy as np
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu

CASES = [  # quads a side, pressure, gravity, nodal loads, supports
    (1, True, False, False, "clamped"), (2, False, True, False, "partial"), (2, True, True, True, "partial"),
    (3, True, False, True, "clamped"), (5, False, False, True, "free edge"), (9, True, True, True, "free edge"),
    (16, True, True, False, "fan")]


def _plate(nq, pressure, gravity, nodal, supports):
    m, _, info = M.shell_plate(nq=nq, p_max=2e5, ramp="linear", seed=nq)
    ng = info["ng"]
    if supports != "clamped":  # one edge clamped, the others free or held in single components
        for i in range(m.n_nodes):
            m.fix[i] = [int(i < ng)] * 6
            if supports == "partial" and i >= ng and i % 3 == 0:
                m.fix_dofs(i, [i % 5])
    if supports == "fan":  # alternating diagonals: corner nodes of four and of eight elements
        def nid(i, j):
            return j * ng + i
        for q in range(nq):
            for p in range(nq):
                if (p + q) % 2 == 0:
                    continue
                i, j = 2 * p, 2 * q
                c = nid(i + 1, j + 1)
                e = 2 * (q * nq + p)
                m.shell_conn[e] = [nid(i, j), nid(i + 2, j), nid(i, j + 2), nid(i + 1, j), c, nid(i, j + 1)]
                m.shell_conn[e + 1] = [nid(i + 2, j), nid(i + 2, j + 2), nid(i, j + 2), nid(i + 2, j + 1),
                                       nid(i + 1, j + 2), c]
                # the cell's middle on its new diagonal
                m.xyz[c][2] = 0.5 * (m.xyz[nid(i + 2, j)][2] + m.xyz[nid(i, j + 2)][2])
    if not pressure:
        m.loads = []
    if gravity:
        m.gravity, m.gravity_on = (0.3, -0.5, -9.81), 1
    if nodal:
        rng = np.random.default_rng(nq)
        nodes = rng.choice(m.n_nodes, min(m.n_nodes, 7), replace=False)
        for kind in (abi.GF_LOAD_NODAL, abi.GF_LOAD_NODAL_FOLLOWER):
            vals = np.zeros((len(nodes), 2, 6))
            vals[:, 1] = rng.normal(size=(len(nodes), 6)) * 50.0
            m.add_nodal_loads(kind, nodes, [0.0, 1.0], vals)
    m._frozen = None
    return m


def _states(m, solver):
    dm = runtime.DeviceModel(m, solver=solver)
    dm.set_window(0.0, 1.0)
    rng = np.random.default_rng(11)
    out = []
    for t_last, scale in ((0.3, 0.0), (0.5, 1e-4)):
        dm.begin_step(t_last, 0.1)
        d = rng.normal(size=(m.n_nodes, 6)) * scale
        dm.write_disp(d)
        dm.assemble()
        dm.assemble()  # (nothing of an earlier assembly is left)
        out.append((dm.tangent_dense(), dm.residual(), np.abs(d).max()))
    dm.close()
    return out


@pytest.mark.parametrize("nq,pressure,gravity,nodal,supports", CASES)
def test_rows_match_scatter(nq, pressure, gravity, nodal, supports):
    m = _plate(nq, pressure, gravity, nodal, supports)
    for (K, r, d), (Kb, rb, _) in zip(_states(m, abi.GF_SOLVER_FRONTS), _states(m, abi.GF_SOLVER_BAND)):
        top = np.abs(Kb).max()
        assert top > 0.0
        assert np.abs(K - Kb).max() <= 1e-13 * top
        assert np.abs(r - rb).max() <= 1e-13 * (60.0 * top * d + np.abs(rb).max())
