"""The selection over a sampled search's candidates where they lie unevenly in their segments: of the queries' neighbours, so many sit in
the blocks of one workgroup that its segment holds sixteen, a multiple of that, all 64 or one more than fit; or all of them sit side
by side.  Few results take a threshold from groups' best keys, more are counted out.  Against the exact path."""
import numpy as np
import pytest

from helpers import SAMPLED, bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")


def near(v, at, q, gen):
    """Rows `at` become neighbours of the queries, each query's in turn."""
    which = torch.arange(len(at), device="cuda:0") % len(q)
    v[torch.from_numpy(at).to("cuda:0")] = q[which] + 0.2 * torch.randn(len(at), q.shape[1], device="cuda:0", generator=gen)


@pytest.mark.parametrize("dim,bits,nq", [(64, 4, 1), (128, 2, 1), (1536, 2, 1), (1024, 3, 1), (64, 4, 9), (64, 3, 20), (128, 4, 70), (64, 4, 150)])
@pytest.mark.parametrize("together", [1, 15, 16, 17, 33, 48, 64, 65, 400])
def test_candidates_in_few_segments(dim, bits, nq, together):
    from turbovec_amd import _lib as T
    n = 300_001 if dim <= 128 else 100_001      # (long rows: 256 segments at the most, which four threads each read for one query of many results)
    gen = torch.Generator(device="cuda:0").manual_seed(together + dim)
    v, q = torch.randn(n, dim, device="cuda:0", generator=gen), torch.randn(nq, dim, device="cuda:0", generator=gen)
    slots = np.arange(n)
    for at in (slots[slots // 32 % 256 == 3], slots[n // 3:]):
        near(v, at[:together * nq], q, gen)
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, bits)
    ix.add_dev(v.data_ptr(), n)
    queries = q.cpu().numpy()
    for k in (1, 16, 17, 100, 129, 256, 400):
        ix.set_path(1)
        s1, i1 = ix.search(queries, k)
        ix.set_path(SAMPLED)
        s, i = ix.search(queries, k)
        assert np.array_equal(i, i1) and bits_equal(s, s1), k
    ix.close()
