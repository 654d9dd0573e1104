import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU and libpnjl_hip.so")


@pytest.fixture(scope="session")
def oracle():
    from oracle import oracle as O
    O.lib()
    return O


@pytest.fixture(scope="session")
def gpu_ctx():
    import julia_relaxtime_amd.pnjl as pnjl
    return pnjl.context(0)


@pytest.fixture(autouse=True)
def library_geometry(request):
    """Every GPU test starts at the launch geometry of a new context."""
    if "gpu_ctx" in request.fixturenames:
        request.getfixturevalue("gpu_ctx").set_launch_auto()


def golden_rows(name):
    import csv
    with open(os.path.join(GOLDEN, name)) as f:
        return list(csv.DictReader(f))
