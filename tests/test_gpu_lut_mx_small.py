"""u8-LUT batches over few blocks on the sparse matrix-unit scan, which takes batches of more than 48 queries there where the rows are
short or of 3-bit codes, or the queries more than 384, or from 1400 (block, query tile) pairs on: against the exact path and against
passes of eight queries."""
import numpy as np
import pytest

from helpers import SAMPLED, bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

NO_LUT16 = 8      # set_path: at most eight queries a pass


# each clause of the rule and its other side: 48 and 49 queries, 6 and 7 chunks, 384 and 385 queries, 1350 and 1450 pairs; a block of one
# row, of 31, and a second one of one row; a call whose last chunk is on the other side
@pytest.mark.parametrize("dim,bits,n,nq", [
    (128, 2, 1, 49), (128, 2, 31, 65), (768, 2, 33, 130), (64, 3, 700, 49), (64, 3, 700, 48), (768, 2, 6_001, 100), (776, 2, 3_001, 100),
    (1536, 3, 701, 65), (1536, 3, 3_001, 300), (384, 4, 2_001, 49), (1536, 2, 701, 384), (1536, 2, 701, 385), (3072, 2, 3_001, 400),
    (1536, 2, 21_600, 64), (1536, 2, 23_200, 64), (3072, 2, 1_003, 1070), (512, 3, 5_001, 1040)])
def test_few_blocks(dim, bits, n, nq):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, bits)
    ix.set_score_mode(T.SCORE_L_U32)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    for m in (None, np.random.default_rng(n).random(n) < 0.5):
        if m is not None and not m.any():
            m[0] = True
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 30, 100):
            ix.set_path(1)
            s1, i1 = ix.search(q, k, mask_words=words)
            for path in (0, SAMPLED, NO_LUT16):
                ix.set_path(path)
                redos = ix.overflow_redos()
                s, i = ix.search(q, k, mask_words=words)
                assert np.array_equal(i, i1) and bits_equal(s, s1), (k, path)
                assert ix.overflow_redos() == redos, (k, path)      # (a candidate that got lost would show here, and not in the repeated answer)
    ix.close()
