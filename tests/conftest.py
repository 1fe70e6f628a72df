import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (ROOT, os.path.join(ROOT, "tests")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (HIP) device")


def pytest_collection_modifyitems(config, items):
    # the one drop-in test without a skip of its own for a tree in which the drop-in main is not built
    binary = os.path.join(ROOT, "hybird_amd", "host", "hybird_gpu")
    if os.path.exists(binary):
        return
    for item in items:
        if item.name == "test_dropin_drum_matches_reference":
            item.add_marker(pytest.mark.skip(reason="hybird_gpu not built (needs the reference's hybird.cpp)"))
