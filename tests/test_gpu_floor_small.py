"""Floors from a sample's best words on indexes of any size: as long as the sample holds k blocks with a row that may be
returned the answer comes from one sampled pass, below that from the ladder of rows, and it is the exact path's either way."""
import numpy as np
import pytest

from helpers import bits_equal, unit_gaussian

pytestmark = pytest.mark.gpu
EXACT, MASKED = 1, 32


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


# The smallest sample is every fourth block: k of them from 4 k blocks on.  The tile-group kernel, the all-queries one, tables in LDS, the
# sparse table scan, and the largest k of a search without sampling.
@pytest.mark.parametrize("dim,bits,nq,k", [(1536, 4, 64, 100), (512, 4, 200, 100), (1536, 2, 12, 100), (2048, 2, 150, 61), (640, 4, 64, 128)])
def test_small_samples(T, dim, bits, nq, k):
    ix = T.NativeIndex(dim, bits)
    q = unit_gaussian(nq, dim, seed=2)
    rng = np.random.default_rng(3)
    rows = unit_gaussian(32 * (4 * k + 40), dim, seed=1)
    n = 0
    for add, one_level in ((32 * (4 * k - 1), False), (1, True), (31, True), (37, None), (32 * 39 - 5, None)):
        ix.add(rows[n:n + add])
        n += add
        strides = ix.sampling_plan(nq, k)[0]
        if one_level is not None and bits == 4:     # (tables: few (block, tile) pairs take another scan)
            assert (strides[0] == 4 and len(strides) == 2) == one_level, strides
        for m in (None, rng.random(n) < 0.5, (np.arange(n) >= 999) & (np.arange(n) < 999 + n // 3), rng.random(n) < 0.02):
            words = None if m is None else T.pack_mask(m)[0]
            out = []
            for path in (0, MASKED, EXACT):
                ix.set_path(path)
                out.append(ix.search(q, k, mask_words=words))
            ix.set_path(0)
            for s, i in out[:2]:
                assert np.array_equal(i, out[2][1]) and bits_equal(s, out[2][0])
    ix.close()


# 256 words are ranked as they are, more are thinned out first; and of few rows that may be returned
@pytest.mark.parametrize("bits,nq", [(4, 64), (2, 12)])
@pytest.mark.parametrize("words", [255, 256, 257])
def test_words_ranked_as_they_are(T, words, bits, nq):
    dim, k, n = 1536, 100, words * 4 * 32
    ix = T.NativeIndex(dim, bits)
    ix.add(unit_gaussian(n, dim, seed=words))
    q = unit_gaussian(nq, dim, seed=7)
    assert list(ix.sampling_plan(nq, k)[0]) == [4, 1]
    for m in (None, np.arange(n) % 128 < 3):      # (blocks of the sample alone)
        mask = None if m is None else T.pack_mask(m)[0]
        out = []
        for path in (0, MASKED, EXACT):
            ix.set_path(path)
            out.append(ix.search(q, k, mask_words=mask))
        for s, i in out[:2]:
            assert np.array_equal(i, out[2][1]) and bits_equal(s, out[2][0])
    assert ix.overflow_redos() == 0
    ix.close()


# 820 blocks and five tiles of queries are the fewest pairs the sparse table scan takes: a sample of 205 blocks
@pytest.mark.parametrize("dim,bits,nq,k,n", [(1536, 2, 150, 61, 820 * 32), (1536, 2, 150, 64, 820 * 32 - 31), (1536, 3, 129, 62, 1500 * 32 + 1)])
def test_small_samples_of_the_sparse_scan(T, dim, bits, nq, k, n):
    ix = T.NativeIndex(dim, bits)
    ix.add(unit_gaussian(n, dim, seed=5))
    q = unit_gaussian(nq, dim, seed=6)
    strides = ix.sampling_plan(nq, k)[0]
    assert len(strides) == 2, strides
    s, i = ix.search(q, k)
    assert ix.queries_per_launch() == nq and ix.overflow_redos() == 0
    ix.set_path(EXACT)
    s2, i2 = ix.search(q, k)
    assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()


def test_a_range_of_rows_leaves_no_floor_open(T):
    """Of 600,000 rows a sample of best words reads one block in eighteen: a range of 5 % has 52 such blocks, fewer than k.
    The search knows, and no query is repeated."""
    dim, n, nq, k = 1536, 600_000, 64, 60
    torch = pytest.importorskip("torch")
    gen = torch.Generator(device="cuda:0").manual_seed(4)
    ix = T.NativeIndex(dim, 4)
    for _ in range(6):
        x = torch.randn(n // 6, dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(x.data_ptr(), len(x))
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    m = (np.arange(n) >= 200_000) & (np.arange(n) < 230_000)
    words = T.pack_mask(m)[0]
    s, i = ix.search(q, k, mask_words=words)
    assert ix.overflow_redos() == 0
    ix.set_path(EXACT)
    s2, i2 = ix.search(q, k, mask_words=words)
    assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()
