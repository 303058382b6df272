"""u8-LUT batches on the sparse matrix-unit scan (k_scan_lut_mx): every instance, the edges of its
tiles, and its hand-over to the fallbacks, bit for bit against the oracle.  The scan serves more than
sixteen queries over 4096 or more (block, query tile) pairs with the u32 epilogue."""
import numpy as np
import pytest

from helpers import SAMPLED, OracleIndex, bits_equal, to_native, unit_gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


# One tile of queries (17, 32), two (33, 64), an odd number with a stand-in tile (65), several groups
# (200: four, 300: five); rows of 1, 2, 3 and 9 chunks, whole and ragged; 16-entry tables (2 and 4 bits)
# and 8-entry ones (3 bits); last blocks of 1, 31 and 32 rows.
@pytest.mark.parametrize("dim,bits,n,nq", [
    (64, 2, 131_073, 17), (128, 2, 131_103, 32), (136, 2, 70_000, 33), (200, 3, 65_536, 64), (64, 3, 131_075, 17),
    (72, 4, 131_072, 20), (384, 2, 50_001, 65), (1120, 2, 20_011, 200), (576, 3, 30_001, 300)])
def test_sparse_scan_matches_oracle(T, oracle, dim, bits, n, nq):
    oidx = OracleIndex(oracle, dim, bits, unit_gaussian(n, dim, seed=91))
    q = unit_gaussian(nq, dim, seed=92)
    ix = to_native(T, oidx, T.SCORE_L_U32)
    rng = np.random.default_rng(11)
    for m in (None, rng.random(n) < 0.5, rng.random(n) < 0.003, (np.arange(n) >= 9_000) & (np.arange(n) < 11_000)):
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 10, 100):
            os_, oi = oidx.search(q, k, mask_words=words, mode=oracle.MODE_L_U32)
            for path in (0, SAMPLED):               # every block's best score; candidates
                ix.set_path(path)
                s, i = ix.search(q, k, mask_words=words)
                assert np.array_equal(i, oi), (k, path)
                assert bits_equal(s, os_), (k, path)
                assert ix.queries_per_launch() == nq
    ix.close()


def test_equal_rows_overflow_to_the_exact_path(T, oracle):
    """All rows tie: every candidate segment overflows, and the lowest slots must come back."""
    dim, bits, n, nq = 32, 2, 131_080, 40
    oidx = OracleIndex(oracle, dim, bits, np.tile(unit_gaussian(1, dim, seed=3), (n, 1)))
    ix = to_native(T, oidx)
    ix.set_path(SAMPLED)
    q = unit_gaussian(nq, dim, seed=4)
    for k in (10, 40):
        s, i = ix.search(q, k)
        os_, oi = oidx.search(q, k)
        assert np.array_equal(i, np.tile(np.arange(k), (nq, 1)))
        assert np.array_equal(i, oi) and bits_equal(s, os_)
    assert ix.overflow_redos() > 0
    ix.close()


@pytest.mark.parametrize("dim,nq", [(1536, 6), (3072, 3)])
def test_few_queries_on_long_rows(T, oracle, dim, nq):
    """Fewer queries than a sixteen-query pass, more than whole tables of such rows fit the LDS for."""
    n = 5_001
    oidx = OracleIndex(oracle, dim, 3, unit_gaussian(n, dim, seed=93))
    ix = to_native(T, oidx)
    q = unit_gaussian(nq, dim, seed=94)
    s, i = ix.search(q, 10)
    os_, oi = oidx.search(q, 10)
    assert np.array_equal(i, oi) and bits_equal(s, os_)
    ix.close()
