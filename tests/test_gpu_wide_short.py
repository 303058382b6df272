"""The all-queries permute-dot scan on rows of 2 to 8 chunks, whose workgroups meet once for several query tiles: over several
rounds of the grid (256 workgroups of 8 waves with 6, 4, 3 or 2 blocks each) and counts of tiles that the meetings do not divide, so that a
round ends between two of them: against the exact path."""
import numpy as np
import pytest

from helpers import SAMPLED, bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


# 129 queries are five tiles, the fewest; two rounds and a few blocks (waves without one among them), three, one
@pytest.mark.parametrize("dim,n,nq", [(128, 800_003, 129), (128, 393_217, 1024), (192, 530_001, 200), (256, 530_001, 225), (256, 262_145, 993),
                                      (320, 400_001, 150), (384, 400_003, 330), (384, 196_609, 1024), (448, 270_001, 129), (448, 131_073, 1024),
                                      (512, 270_033, 260), (512, 131_072, 1024)])
def test_rounds_that_end_between_hand_overs(dim, n, nq):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, 4)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    rng = np.random.default_rng(n)
    for m in (None, rng.random(n) < 0.7, np.arange(n) >= n - 70_000):
        words = None if m is None else T.pack_mask(m)[0]
        ix.set_path(1)
        s1, i1 = ix.search(q, 10, mask_words=words)
        redos = ix.overflow_redos()
        for path in (0, SAMPLED):      # (SAMPLED also has masks read during the scan, not their rows gathered)
            ix.set_path(path)
            for _ in range(2):
                s, i = ix.search(q, 10, mask_words=words)
                assert np.array_equal(i, i1) and bits_equal(s, s1), path
                assert ix.overflow_redos() == redos, path      # (a candidate that got lost would show here, and not in the repeated answer)
    ix.close()
