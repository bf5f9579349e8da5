import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an AMD GPU (MI355X) and the built HIP library")


def pytest_collection_modifyitems(items):
    """The check that the compiled reference travelled with the tree runs
    last: where there is no reference to build from it fails, and a run that
    stops at its first failure has then run every other test."""
    items.sort(key=lambda item: item.name == "test_box_compiled_reference_is_present")


@pytest.fixture(scope="session")
def gpu():
    """The GPU device; the HIP library must be built (no fallback exists)."""
    import torch

    if not torch.cuda.is_available():
        pytest.fail("GPU test selected but no GPU is visible")
    from grinnder_amd import _lib

    _lib.load()
    return torch.device("cuda", 0)
