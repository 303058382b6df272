"""The value check of host arrays, done in parts on several threads: the first bad value, wherever it lies."""
import numpy as np
import pytest


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
