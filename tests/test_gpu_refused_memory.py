"""A search whose staging memory the device cannot give: refused each time it is asked for, and nothing else changes."""
import ctypes as C

import numpy as np
import pytest

from helpers import bits_equal, unit_gaussian

pytestmark = pytest.mark.gpu


def test_refused_staging_memory_stays_refused():
    from turbovec_amd import _lib as T
    n, dim, many = 1 << 16, 8, 1 << 20
    ix = T.NativeIndex(dim, 4)
    ix.add(unit_gaussian(n, dim, seed=1))
    q = unit_gaussian(5, dim, seed=2)
    before = ix.search(q, 10)
    wide_q = np.zeros((many, dim), np.float32)
    wide_q[:, 0] = 1.0
    scores, slots, k_eff = np.zeros(1, np.float32), np.zeros(1, np.int64), C.c_size_t(0)
    for _ in range(2):      # 2^36 results, 0.8 TB: more than the device has, and nothing is written
        rc = T.lib().tv_search(ix.h, T.ptr(wide_q), many, n, None, 0, T.ptr(scores), T.ptr(slots), C.byref(k_eff))
        assert rc == T.ERR_HIP
        after = ix.search(q, 10)
        assert bits_equal(after[0], before[0]) and np.array_equal(after[1], before[1])
    ix.close()
