"""The all-queries permute-dot scan at odd chunk counts (3, 5 and 7 chunks of 64 dimensions, the last one partly
filled too), where its weights come in a slice whose pieces do not divide among the waves: against the oracle."""
import numpy as np
import pytest

from helpers import SAMPLED, OracleIndex, bits_equal, to_native, unit_gaussian

pytestmark = pytest.mark.gpu


# one block, a ragged last block, more blocks than a round of the grid holds (256 workgroups of 8 waves with 4, 3 or 2
# blocks each: 8192, 6144 and 4096); 129 queries are the fewest that take this kernel, 1024 the most of one launch
@pytest.mark.parametrize("dim,n,nq", [(136, 33, 129), (176, 5_001, 1024), (192, 270_000, 161), (264, 6_007, 129), (320, 200_033, 300),
                                      (392, 4_001, 1024), (432, 140_000, 130), (448, 2_015, 1030)])
def test_odd_chunk_counts_match_oracle(oracle, dim, n, nq):
    from turbovec_amd import _lib as T
    oidx = OracleIndex(oracle, dim, 4, unit_gaussian(n, dim, seed=dim + n))
    q = unit_gaussian(nq, dim, seed=79)
    ix = to_native(T, oidx)
    ix.set_path(SAMPLED)
    rng = np.random.default_rng(3)
    for m in (None, rng.random(n) < 0.5, (np.arange(n) >= n // 2) & (np.arange(n) < n // 2 + 70)):
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 30):
            s, i = ix.search(q[:300], k, mask_words=words)
            os_, oi = oidx.search(q[:300], k, mask_words=words)
            assert ix.queries_per_launch() == min(nq, 300)
            assert np.array_equal(i, oi) and bits_equal(s, os_), k
    s, i = ix.search(q, 10)
    assert ix.queries_per_launch() == min(nq, 1024)
    ix.set_path(1)
    s2, i2 = ix.search(q, 10)
    assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()
