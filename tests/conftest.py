"""Shared test set-up: the `gpu` marker, the oracle import path, tolerances."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
sys.path.insert(0, os.path.join(ROOT, "oracle"))


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP library)")


def pytest_collection_modifyitems(items):
    """The GPU tests that run the reference's own kernels need their builds, which the oracle's
    makefile makes where the reference's sources are present."""
    ref = os.path.join(ROOT, "oracle", "_ref")
    if all(os.path.exists(os.path.join(ref, f)) for f in ("kernel19.co", "kernel27.co")):
        return
    skip = pytest.mark.skip(reason="the reference's kernels are not built (its sources are absent)")
    for item in items:
        if item.get_closest_marker("gpu") and "_reference_" in item.name:
            item.add_marker(skip)


def rel_l2(a, b):
    a = np.asarray(a, np.float64)
    b = np.asarray(b, np.float64)
    n = np.linalg.norm(b)
    return float(np.linalg.norm(a - b) / (n if n > 0 else 1.0))


def gpu_available():
    try:
        import ctypes
        hip = ctypes.CDLL("libamdhip64.so")
        n = ctypes.c_int(0)
        return hip.hipGetDeviceCount(ctypes.byref(n)) == 0 and n.value > 0
    except OSError:
        return False
