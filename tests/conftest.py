"""Test configuration: the `gpu` marker and import paths.

`-m "not gpu"` runs the CPU suite (oracle vs golden vectors, host logic, the
C-ABI library loads and exports every declared symbol); `-m gpu` runs the
parity tests proper, which call the HIP library through its C ABI.
"""
import ctypes as C
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "the-rule-and-compass_amd")
for p in (ROOT, PKG, os.path.join(ROOT, "oracle")):
    if p not in sys.path:
        sys.path.insert(0, p)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP C ABI)")


@pytest.fixture
def free_memory():
    """Free bytes of the current device, from the HIP runtime that the library
    has loaded (a second one, such as torch brings, would be another process-wide
    state)."""
    from rcsr_hip import lib
    lib.load()
    hip = C.CDLL("libamdhip64.so.7")

    def read():
        free, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(free), C.byref(total)) == 0
        return free.value
    return read
