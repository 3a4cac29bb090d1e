import gc
import os
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent
if str(ROOT) not in sys.path:
    sys.path.insert(0, str(ROOT))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (gfx950) GPU")


def gpu_available() -> bool:
    try:
        from cpmd_amd import _lib
        import ctypes
        n = ctypes.c_int(0)
        return _lib.lib().mc_device_count(ctypes.byref(n)) == 0 and n.value > 0
    except Exception:
        return False


@pytest.fixture(scope="session")
def gpu():
    if not gpu_available():
        pytest.fail("GPU test selected but no GPU / libmicpmd.so available")
    return True


@pytest.fixture(autouse=True)
def _no_leftovers(request):
    """A caught exception that a test keeps in a local holds the test's frame in a
    reference cycle, and with it the contexts and device arrays there.  They are
    freed before a GPU test begins, not when the collector happens to run: tests
    that read the device memory in use would see it fall."""
    if request.node.get_closest_marker("gpu"):
        gc.collect()
