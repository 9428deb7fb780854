import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

# every batch load in the tests times the SpMM shapes itself, unless a test
# names a tuning file of its own (the batch autotuner's persisted winners)
os.environ.setdefault("HECMW33_TUNE_CACHE", "off")


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs the HIP library)")


def pytest_collection_modifyitems(items):
    """Tests that run the library in a child process go first.  HIP gives the GPU's cooperative
    queue to one process: once this one has launched cooperatively, it refuses a child's
    cooperative launches (401), and the child's solves take the launches."""
    items.sort(key=lambda i: not (hasattr(i, "function") and "hip_shim" in i.function.__code__.co_names))


@pytest.fixture(scope="session")
def has_gpu():
    import frontistr_amd as fa
    return fa.lib().hecmw33_device_count() > 0
