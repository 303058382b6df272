"""The scan of few blocks, where a block's chunks go to several waves: chunks the parts do not divide, a last workgroup with fewer
blocks than the others, blocks without an allowed row, every form of its results; bit for bit against the exact path."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.mark.parametrize("dim,bits,ns,nqs", [
    (512, 4, (1, 33, 20_011), (1, 33)), (584, 4, (40, 8_200, 32_801), (2, 64)), (1536, 4, (65, 4_097, 20_000, 65_537), (1, 40)), (2056, 4, (300, 9_001), (1, 100)),
    (3072, 4, (2_000, 30_000), (1, 8)), (128, 2, (31, 3_333), (1, 2)), (200, 3, (64, 9_999), (1, 4, 5)), (384, 2, (500, 60_001), (1, 3, 8)),
    (1000, 3, (33, 12_345), (1, 2, 4, 8)), (1400, 2, (1_000, 50_001), (1, 2, 6)), (3072, 3, (97, 16_411), (1, 2, 3)), (3072, 2, (8_000, 24_033), (1, 4)),
    (384, 3, (1_000, 16_001), (9, 16, 47)), (1536, 2, (310, 5_001), (5, 7, 18)), (2432, 3, (4_700,), (9, 16)), (128, 2, (300, 20_001), (9, 44))])
def test_parts_of_blocks(dim, bits, ns, nqs):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + bits)
    rng = np.random.default_rng(dim)
    for n in ns:
        ix = T.NativeIndex(dim, bits)
        v = torch.randn(n, dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), n)
        allowed = rng.random(n) < 0.7
        allowed[(np.arange(n) // 32) % 3 == 1] = False      # (whole blocks)
        allowed[0] = True
        words = T.pack_mask(allowed)[0]
        for nq in nqs:
            q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
            for k in (1, 10, 100):
                for m in (None, words):
                    ix.set_path(1)
                    s1, i1 = ix.search(q, k, mask_words=m)
                    for path in (0, 32):        # (32: masks are read as the scan runs)
                        ix.set_path(path)
                        s, i = ix.search(q, k, mask_words=m)
                        assert np.array_equal(i, i1) and bits_equal(s, s1), (n, nq, k, path)
        ix.close()
