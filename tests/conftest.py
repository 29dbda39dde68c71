import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP device)")


def _gpu_available():
    try:
        import gpu_cdt_refine_amd as g
        return g.lib().gcdt_device_count() > 0
    except Exception:
        return False


@pytest.fixture(scope="session")
def gpu():
    if not _gpu_available():
        pytest.skip("no HIP device")
    import gpu_cdt_refine_amd as g
    g.lib()
    return g


@pytest.fixture(scope="session")
def oracle():
    from oracle import pyoracle
    if not os.path.exists(pyoracle.ORACLE_SO):
        pyoracle.build()
    if not os.path.exists(pyoracle.TRIREF_SO):
        # no reference tree to build Triangle from: tests that only need an
        # input CDT take it from the host builder, tests that compare with
        # Triangle itself skip
        pyoracle.triref = lambda: pytest.skip("the reference's Triangle is not built")
        pyoracle.triangle_cdt = _host_cdt
    return pyoracle


def _host_cdt(points, segments):
    import gpu_cdt_refine_amd as g
    P = np.ascontiguousarray(points, np.float64).reshape(-1, 2)
    return (P,) + g.build_cdt(P, segments)
