"""The second scoring of a search without sampling where a block's chunks go to several waves: results fewer than waves, rows whose
chunks the parts do not divide, shares of blocks among workgroups, filters; bit for bit against the exact path."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim,bits,n,nq,ks", [
    (3072, 4, 40_001, 1, (1, 2, 3, 5, 9, 12, 17)), (1000, 3, 20_015, 3, (1, 4, 7, 33)), (1416, 2, 20_001, 1, (1, 3, 10, 24)), (128, 4, 50_001, 40, (1, 2)),
    (64, 2, 30_031, 1, (1,)), (776, 4, 9_001, 100, (1, 2, 5)), (2760, 2, 9_017, 256, (1, 2)), (1536, 4, 70_003, 257, (1,)), (3032, 3, 12_001, 1, (4, 54, 100))])
def test_few_results(dim, bits, n, nq, ks):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, bits)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    words = T.pack_mask(np.random.default_rng(n).random(n) < 0.6)[0]
    for k in ks:
        for m in (None, words):
            ix.set_path(1)
            s1, i1 = ix.search(q, k, mask_words=m)
            for path in (0, 32):            # (32: masks are read as the scan runs)
                ix.set_path(path)
                s, i = ix.search(q, k, mask_words=m)
                assert np.array_equal(i, i1) and bits_equal(s, s1), (k, path)
    ix.close()
