"""Device memory that a diagnostics call takes."""
import ctypes

import numpy as np
import pytest

from lpmgpu import Context
from lpmgpu import _lib as L

pytestmark = pytest.mark.gpu


def _free_bytes():
    """Free device memory by the HIP runtime that the library is linked against."""
    L.lib()
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL(path).hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_diagnostics_take_no_active_list():
    """The diagnostics read the mask itself: a call holds its five arrays and the mask on
    the device and no list of active particles beside them."""
    n = 8 << 20
    u = np.ones(n)
    act = np.ones(n, np.int32)
    with Context(0) as c:
        c.diagnostics(u[:100], u[:100], u[:100], u[:100], u[:100], act[:100])
        before = _free_bytes()
        ke, en, circ = c.diagnostics(u, u, u, u, u, act)
        taken = before - _free_bytes()
    assert (ke, en, circ) == (1.5 * n, 0.5 * n, float(n))
    assert taken <= (5 * 8 + 4) * n + (16 << 20)  # the list would be 32 MiB more
