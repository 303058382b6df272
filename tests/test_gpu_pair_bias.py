"""The bias term of a TQ+ pair (an f64 sum of which the f32 rounding is used) against the oracle."""
import numpy as np
import pytest

from helpers import OracleIndex, bits_equal, to_native, unit_gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


# Large shifts: a thousand queries' sums, some of them near a rounding boundary; no shift: a sum of zeros, of either sign.
@pytest.mark.parametrize("dim,bits", [(8, 4), (1000, 3), (3032, 2)])
def test_bias_of_a_pair(T, oracle, dim, bits):
    rng = np.random.default_rng(dim)
    v = unit_gaussian(40, dim, seed=1)
    q = unit_gaussian(1024, dim, seed=2)
    for shift in (0.1, 1e6, 0.0):
        cal = ((rng.standard_normal(dim) * shift).astype(np.float32), np.linspace(0.5, 2.0, dim, dtype=np.float32))
        oidx = OracleIndex(oracle, dim, bits, v, calibration=cal)
        ix = to_native(T, oidx)
        s, i = ix.search(q, 3)
        os_, oi = oidx.search(q, 3)
        assert np.array_equal(i, oi) and bits_equal(s, os_)
        ix.close()
