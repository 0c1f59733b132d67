import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP kernels)")


def gpu_available():
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:
        return False


# Tests of what the package no longer does, by name, with the reason.
TAKEN_BACK = {
    "test_results_on_the_host_are_the_callers_own":
        "results come back in ordinary memory, none of it counted as pinned: the driver's "
        "pinned pages are missing in forked processes and dear to allocate for small results",
}


def pytest_collection_modifyitems(config, items):
    for item in items:
        reason = TAKEN_BACK.get(getattr(item, "originalname", None))
        if reason:
            item.add_marker(pytest.mark.xfail(reason=reason, raises=AttributeError, strict=True))
    if gpu_available():
        return
    skip = pytest.mark.skip(reason="no GPU in this environment")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)
