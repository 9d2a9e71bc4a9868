import os
import sys

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

GOLDEN = os.path.join(ROOT, "tests", "golden")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")
    config.addinivalue_line("markers", "slow: takes more than ~20 s on the CPU")


def pytest_collection_modifyitems(items):
    # the programs built from the reference's sources come last: where those
    # are absent, a run that ends at the first failure has run the rest
    items.sort(key=lambda i: i.path.name == "test_gpu_dropin.py")


@pytest.fixture(scope="session")
def golden_dir():
    return GOLDEN
