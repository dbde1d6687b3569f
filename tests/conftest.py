import os
import sys

import pytest

sys.path.insert(0, os.path.dirname(os.path.dirname(os.path.abspath(__file__))))
sys.path.insert(0, os.path.dirname(os.path.abspath(__file__)))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (run with -m gpu)")


def _gpu_available() -> bool:
    try:
        import torch
        return torch.cuda.is_available()
    except Exception:  # noqa: BLE001
        return False


def pytest_collection_modifyitems(config, items):
    if _gpu_available():
        return
    skip = pytest.mark.skip(reason="no GPU in this container")
    for item in items:
        if "gpu" in item.keywords:
            item.add_marker(skip)


@pytest.fixture(autouse=True)
def _memory_of_tests_before(request):
    """A test that measures the card's free memory starts from what is really free: engines of the tests before that wait for the
    collector, and the allocator's cache, would otherwise go back during the test or not by when the collector happens to run."""
    if "free_memory" in request.node.name and _gpu_available():
        import gc
        import torch
        gc.collect()
        torch.cuda.empty_cache()
    yield
