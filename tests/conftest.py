import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "oracle")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP path through the C ABI)")
    config.addinivalue_line("markers", "slow: longer CPU runs")


@pytest.fixture
def device_holds():
    """holds(model, solver): skips where the device's memory is below twice the model's footprint."""
    def holds(model, **kw):
        import ctypes as C
        from giraffe_amd import runtime
        need = runtime.footprint(model, **kw)  # (loads the library, and with it the HIP runtime)
        hip = C.CDLL("libamdhip64.so.7", mode=os.RTLD_NOLOAD | os.RTLD_GLOBAL)
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        if total.value < 2 * need:
            pytest.skip(f"{need / 1e9:.0f} GB model on a device of {total.value / 1e9:.0f} GB")
    return holds


@pytest.fixture(scope="session")
def oracle_lib():
    import oracle
    oracle.build()
    return oracle
