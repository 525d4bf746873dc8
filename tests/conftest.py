import contextlib
import ctypes
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a HIP device (MI355X); runs the engine through the C ABI")


@pytest.fixture(scope="session")
def oracle_lib():
    from oracle import oracle

    oracle.load()
    return oracle


def say(*a):
    """Progress line that names the case before a GPU step (flushed)."""
    print(*a, flush=True)


def _hip():
    """The HIP runtime that the engine library is linked to."""
    from opendust_amd import engine

    engine.load_library()
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(w.split()[-1] for w in f if "libamdhip64" in w))


def gpu_free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert _hip().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


@contextlib.contextmanager
def gpu_memory_left(left):
    """Holds all device memory but `left` bytes (allocated, never touched)."""
    hip = _hip()
    held = []
    try:
        while True:
            take = min(gpu_free_bytes() - left, 32 << 30)
            if take < 1 << 20:
                break
            p = ctypes.c_void_p()
            assert hip.hipMalloc(ctypes.byref(p), ctypes.c_size_t(take)) == 0
            held.append(p)
        say("  device memory left, GB:", round(gpu_free_bytes() / 1e9, 2))
        yield
    finally:
        for p in held:
            hip.hipFree(p)


def rel_err(a, b, floor=0.0):
    a = np.asarray(a, dtype=np.float64)
    b = np.asarray(b, dtype=np.float64)
    return np.abs(a - b) / np.maximum(np.abs(b), floor)


# error-model checkers shared with __graft_entry__.smoke() live with the oracle
from oracle.oracle import check_records, fp32c_position_bounds, fp32c_position_error_ok, orbit_sum_bound  # noqa: E402,F401
