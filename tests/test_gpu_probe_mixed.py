"""Per-kernel event timing of a chain in mixed precision: the FP32 factorisations
count in the block-tridiagonal classes beside the FP64 solves (fallbacks, and direct
ones while the mode backs off)."""
import pytest

from giraffe_amd import abi, model as M, runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_elem", [20, 500])
def test_fp32_factorisations_are_counted(n_elem):
    m, p, _ = M.catenary(n_elem=n_elem)
    dm = runtime.DeviceModel(m, precision=abi.GF_PREC_MIXED)
    nblk = dm.info()["n_blocks"]
    dm.timing(True)
    dm.kernel_probe(dm.KERNEL_CLASSES)
    rep, _ = dm.static_solve(p)
    kp, st = dm.kernel_probe_read(reset=True), dm.stats()
    assert rep.aborted == 0 and st["fp32_factorizations"] > 0
    factorisations = st["fp32_factorizations"] + st["fallbacks"] + st["fp64_direct"]
    n, rows, levels = nblk, 0, 0
    while n > 16:
        rows += n // 2
        n //= 2
        levels += 1
    assert kp["btd_tail"][1] == factorisations and kp["btd_tail"][0] > 0
    if levels:
        assert kp["btd_level"][1:] == (levels * factorisations, rows * factorisations)
    dm.close()
