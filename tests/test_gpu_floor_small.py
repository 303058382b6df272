"""Floors from a sample's best words: as long as the sample holds k blocks with a row that may be returned the answer comes from
one sampled pass, below that from the ladder of rows, and it is the exact path's either way."""
import numpy as np
import pytest

from helpers import bits_equal, unit_gaussian

pytestmark = pytest.mark.gpu
EXACT = 1


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


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
