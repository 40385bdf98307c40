import os
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
sys.path.insert(0, HERE)
sys.path.insert(0, os.path.join(ROOT, "multigrid-poisson_amd"))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library)")
    config.addinivalue_line("markers", "slow: long CPU test")


# the reference's sources the drop-in headers are compiled against: tests that
# read them run where they are there, and are skipped where the folder is absent
# or empty
REFERENCE_SOURCE = "/root/reference/src/problem_definition.cpp"


def pytest_collection_modifyitems(items):
    if os.path.isfile(REFERENCE_SOURCE):
        return
    for item in items:
        if item.name.startswith("test_reference_drivers_compile"):
            item.add_marker(pytest.mark.skip(reason="%s not present" % REFERENCE_SOURCE))
