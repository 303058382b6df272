"""The value check of host arrays, done in parts on several threads: the first bad value, wherever it lies."""
import subprocess
import sys

import numpy as np
import pytest

from conftest import ROOT


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


# below a part (2^20 values), at its edges, several parts, a ragged last one
@pytest.mark.parametrize("n", [8, 4095, 4096, 4097, 1 << 20, (1 << 21) + 8, 9 * (1 << 20) + 24])
def test_first_bad_value_is_reported(T, n):
    n -= n % 8
    v = np.random.default_rng(n).standard_normal(n).astype(np.float32)
    v[n // 2] = np.float32(9.999999e15)
    assert T.validate_queries(v, 8) == (T.OK, 0)
    for bad in (np.nan, np.inf, -np.inf, np.float32(1e16), np.float32(-1e16)):
        for at in {0, n - 1, n // 2, min(n - 1, 4096), min(n - 1, 1 << 20)}:
            w = v.copy()
            w[at] = bad
            w[n - 1] = np.nan
            assert T.validate_queries(w, 8) == (T.ERR_INVALID_QUERY_VALUE, at)


WRITER = '''
import ctypes as C, mmap, sys, threading
import numpy as np
sys.path.insert(0, sys.argv[1])
from turbovec_amd import _lib as T
T.lib()
libc = C.CDLL(None, use_errno=True)
page, n = mmap.PAGESIZE, 4096
pages = mmap.mmap(-1, n * 4 + page)
at = C.addressof(C.c_char.from_buffer(pages))
assert libc.mprotect(C.c_void_p(at + n * 4), C.c_size_t(page), 0) == 0       # nothing may be read behind the values
v = np.frombuffer(pages, np.float32, n)
stop = False
def flip():
    while not stop:
        v[n - 1] = np.nan
        v[n - 1] = 0.0
sys.setswitchinterval(1e-5)
t = threading.Thread(target=flip)
t.start()
try:
    for _ in range(4000):
        rc, bad = T.validate_queries(v, 8)
        assert (rc, bad) in ((T.OK, 0), (T.ERR_INVALID_QUERY_VALUE, n - 1)), (rc, bad)
finally:
    stop = True
    t.join()
'''


def test_values_that_change_during_the_check():
    """Another thread overwrites the one bad value, the last of the array, again and again: the check answers for
    what it read and reads nothing behind the array."""
    run = subprocess.run([sys.executable, "-c", WRITER, ROOT], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.returncode, run.stderr)
