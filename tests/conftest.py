import gc
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for p in (os.path.join(ROOT, "scriptling-llm-lib_amd"), os.path.join(ROOT, "oracle"), ROOT):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")
    config.addinivalue_line("markers", "slow: larger shapes (seconds of oracle time)")


def has_gpu() -> bool:
    return os.path.exists("/dev/kfd")


def pytest_collection_modifyitems(config, items):
    if has_gpu():
        return
    skip = pytest.mark.skip(reason="no GPU (/dev/kfd absent)")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


def pytest_runtest_setup(item):
    # A graph (or weight) that an earlier test left in a reference cycle, as a caught
    # exception's traceback makes one, must not be collected while a later test captures
    # a graph: its destruction synchronizes the device, which aborts the process there.
    if "gpu" in item.keywords and any(k in item.nodeid for k in ("graph", "captur", "argmax", "decode")):
        gc.collect()
