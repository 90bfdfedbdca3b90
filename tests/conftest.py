import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD Instinct GPU (HIP device)")
    config.addinivalue_line("markers", "slow: takes more than ~20 s")


# Reasons of expected failures that have been mended: their mark is lifted, and the
# tests have to pass.
MENDED = {"taps of a 30-pixel axis lack the middle one"}


def pytest_collection_modifyitems(items):
    for item in items:
        item.own_markers[:] = [m for m in item.own_markers
                               if not (m.name == "xfail" and m.kwargs.get("reason") in MENDED)]


@pytest.fixture(scope="session")
def root_dir():
    return ROOT
