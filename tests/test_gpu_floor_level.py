"""Searches that take their floors from a sample of the blocks' best scores (indexes of more than 16384 blocks, on every
kernel without a floorless mode of its own): against the exact path, bit for bit."""
import numpy as np
import pytest

from helpers import SAMPLED, bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


# the tile-group kernel (weights in either order: 64 and 2560 dimensions), the all-queries kernel on short rows, u8 tables
# for a few queries (whole in LDS), up to sixteen (streamed) and more (matrix unit); a last block of one row
@pytest.mark.parametrize("dim,bits,n,nq", [(64, 4, 524_321, 40), (128, 4, 600_001, 100), (768, 4, 524_321, 64), (2560, 4, 524_321, 70),
                                           (136, 4, 540_000, 140), (448, 4, 524_321, 300), (64, 2, 700_000, 2), (256, 3, 524_321, 8),
                                           (200, 2, 600_000, 13), (128, 2, 600_000, 33), (64, 3, 524_321, 160)])
def test_floors_from_best_scores(T, dim, bits, n, nq):
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, bits)
    for at in range(0, n, 131_072):
        v = torch.randn(min(131_072, n - at), dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), len(v))
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    rng = np.random.default_rng(5)
    few = np.zeros(n, bool)
    few[rng.integers(0, n, 40)] = True                    # the sample sees hardly any of these
    for m, k in ((None, 1), (None, 10), (None, 100), (rng.random(n) < 0.5, 10), (few, 20)):
        words = None if m is None else T.pack_mask(m)[0]
        ix.set_path(SAMPLED)
        if m is None and (k < 100 or nq < 33 or bits == 4):
            assert len(ix.sampling_plan(nq, k)[0]) == 2
        s, i = ix.search(q, k, mask_words=words)
        ix.set_path(1)
        s2, i2 = ix.search(q, k, mask_words=words)
        assert np.array_equal(i, i2) and bits_equal(s, s2), k
    ix.close()


def test_equal_rows_and_rows_sorted_by_score(T):
    """Every score ties at the floor; and rows in rising order of score, where the sample is as good as any other."""
    dim, n, nq = 64, 530_000, 64
    one = torch.randn(1, dim, device="cuda:0", generator=torch.Generator(device="cuda:0").manual_seed(1))
    v = one.repeat(n, 1).contiguous()
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, 4)
    ix.add_dev(v.data_ptr(), n)
    ix.set_path(SAMPLED)
    s, i = ix.search(v[:nq].cpu().numpy(), 10)
    assert np.array_equal(i, np.tile(np.arange(10), (nq, 1)))
    ix.close()
    w = torch.randn(n, dim, device="cuda:0", generator=torch.Generator(device="cuda:0").manual_seed(2))
    w = w[torch.argsort(w @ one[0])].contiguous()
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, 4)
    ix.add_dev(w.data_ptr(), n)
    q = (one + 0.1 * torch.randn(nq, dim, device="cuda:0")).cpu().numpy()
    ix.set_path(SAMPLED)
    s, i = ix.search(q, 10)
    ix.set_path(1)
    s2, i2 = ix.search(q, 10)
    assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()
