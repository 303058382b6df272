"""Short rows, many queries: on both sides of the number of blocks from where a floor from a sample goes before the scan, with and
without a filter, results are those of the exact path."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim,n,nq", [
    (256, 328_000, 1000), (256, 328_001, 1000), (192, 491_985, 1024), (192, 492_065, 1024), (640, 665_000, 150), (640, 770_000, 140), (696, 560_000, 300), (128, 600_000, 700)])
def test_both_sides(dim, n, nq):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, 4)
    for at in range(0, n, 100_000):
        v = torch.randn(min(100_000, n - at), dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), len(v))
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    words = T.pack_mask(np.random.default_rng(n).random(n) < 0.8)[0]
    some = np.linspace(0, nq - 1, 6).astype(int)
    for k, m in ((1, None), (20, None), (10, words)):
        ix.set_path(0)
        s, i = ix.search(q, k, mask_words=m)
        ix.set_path(16)      # (a sample goes first on either side)
        s2, i2 = ix.search(q, k, mask_words=m)
        assert np.array_equal(i, i2) and bits_equal(s, s2), k
        ix.set_path(1)
        s1, i1 = ix.search(q[some], k, mask_words=m)
        assert np.array_equal(i[some], i1) and bits_equal(s[some], s1), k
    ix.close()


@pytest.mark.parametrize("dim,n,nq", [(256, 418_176, 1000), (256, 418_177, 1000), (192, 469_376, 1024), (192, 469_377, 1024), (640, 667_872, 150), (640, 667_873, 150)])
def test_both_sides_of_decoding_blocks_again(dim, n, nq):
    test_both_sides(dim, n, nq)
