import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on a machine that has one)")


@pytest.fixture(scope="session")
def oracle():
    import helpers
    return helpers.HostBackend()


@pytest.fixture(scope="session")
def rocm():
    import helpers
    backend = helpers.RocmBackend()
    yield backend
    backend.close()
