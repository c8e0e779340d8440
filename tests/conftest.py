import ctypes
import os
import sys
import time

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs an MI355X (runs through the HIP C-ABI)")


@pytest.fixture(scope="session")
def H():
    import hw_amd
    return hw_amd


@pytest.fixture(scope="session")
def O():
    import oracle
    oracle.threads(min(8, os.cpu_count() or 1))
    return oracle


@pytest.fixture(scope="session")
def T():
    from hw_amd import types
    return types


@pytest.fixture(scope="session")
def gpu(H):
    if H.device_count() == 0:
        pytest.skip("no GPU")
    return True


def gen_traces(O, T, H, lanes, frames, chunks, seed=7, **kw):
    """Seeded synthetic traces from the oracle's generator: list of [lanes, frames, 64] int16."""
    p = H.tracegen_default(seed=seed, **kw)
    st = np.zeros(lanes, dtype=T.TRACEGEN_STATE)
    return [O.tracegen(p, lanes, frames, c * frames, st, c == 0) for c in range(chunks)]


def free_bytes(H):
    """Free device memory (the HIP runtime that the library is linked against).  The driver counts
    freed memory as free some milliseconds later, so the figure has to stand for 0.4 s."""
    H.sync()
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    seen = []
    while len(seen) < 40 and len(set(seen[-5:])) != 1 or len(seen) < 5:
        assert H.lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        seen.append(free.value)
        time.sleep(0.1)
    return seen[-1]
