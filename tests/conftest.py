import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and the built HIP library")


@pytest.fixture(scope="session")
def oracle_lib():
    import oracle
    return oracle.lib()


@pytest.fixture(autouse=True)
def _default_lane_widths(request):
    """GPU tests start with the shipped columns per lane, whatever value a test
    before them left in ALTO_TUNE_NARROW_RANK."""
    if request.node.get_closest_marker("gpu"):
        import alto_amd
        alto_amd.check(alto_amd.lib().alto_tune_set(10, -1), "tune_set")
