"""Searches without sampling whose tiles of queries go three to a workgroup: full and part tiles, rows of one chunk to twelve, filters;
bit for bit against the exact path."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim,n,nqs", [(64, 66_001, (65, 96)), (128, 40_011, (129, 161)), (192, 25_000, (257, 288)), (256, 70_003, (70, 150)),
                                       (448, 66_017, (96, 192)), (512, 35_001, (130, 280)), (640, 66_600, (66,)), (768, 66_001, (65, 96))])
def test_three_tiles(dim, n, nqs):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, 4)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    words = T.pack_mask(np.random.default_rng(n).random(n) < 0.7)[0]
    for nq in nqs:
        q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
        some = np.unique(np.concatenate([np.arange(0, nq, 32), np.arange(31, nq, 32), [nq - 1]]))
        for k, m in ((1, None), (10, None), (10, words)):
            ix.set_path(1)
            s1, i1 = ix.search(q[some], k, mask_words=m)
            for path in (0, 32):
                ix.set_path(path)
                s, i = ix.search(q, k, mask_words=m)
                assert np.array_equal(i[some], i1) and bits_equal(s[some], s1), (nq, k, path)
    ix.close()
