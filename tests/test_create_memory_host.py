"""Host memory that a projector's tables cannot have ends in an error code and a
message, not in an exception that leaves the C entry point (which would end the
process).  In a process of its own, with a bound on its address space."""
import subprocess
import sys

import pytest

CODE = """
import ctypes, resource, numpy as np
from sgd_amd import _lib
L = _lib.lib()
used = int(open("/proc/self/statm").read().split()[0]) * resource.getpagesize()
limit = used + (2 << 30)
resource.setrlimit(resource.RLIMIT_AS, (limit, limit))
a = np.zeros(4)
p = a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
nu = 200000000  # 6.4 GB of records a view
for f in (L.b0_init, L.b1_init):
    assert f(8, 8, 1, nu, 1.0, 1.0, 1.0, 1000.0, 500.0, p, None, None) is None
    assert "host allocation failed" in _lib.last_error(), _lib.last_error()
assert L.h0_init(8, 8, 1, nu, 1.0, 1.0, 1000.0, 500.0, p, None, None) is None
assert "host allocation failed" in _lib.last_error()
print("returned")
"""


def test_tables_without_memory_are_an_error():
    r = subprocess.run([sys.executable, "-c", CODE], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and "returned" in r.stdout, (r.returncode, r.stderr[-500:])
