"""Filtered searches that run on a copy of their allowed rows: the same bits as with the mask read during the scan."""
import numpy as np
import pytest

from helpers import bits_equal

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")

MASKED, GATHERED = 32, 64     # set_path


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


def filled(T, dim, bits, n, seed=1):
    gen = torch.Generator(device="cuda:0").manual_seed(seed)
    ix = T.NativeIndex(dim, bits)
    for at in range(0, n, 131_072):
        v = torch.randn(min(131_072, n - at), dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), len(v))
    return ix, gen


def masks(n, rng):
    """One row, the first and the last; a block less one row, a block, and one row more; words' and workgroups' edges; scattered
    rows from few to all but one; a range."""
    for slots in ([0], [n - 1], [0, n - 1], range(31), range(32), range(n - 33, n), range(0, n, 64), range(63, n, 64), range(65_535, min(n, 65_537))):
        if len(slots):
            m = np.zeros(n, bool)
            m[list(slots)] = True
            yield m
    for share in (0.001, 0.03, 0.5, 0.9):
        m = rng.random(n) < share
        m[n // 2] = True
        yield m
    m = np.ones(n, bool)
    m[n // 3] = False
    yield m
    yield (np.arange(n) >= n // 3) & (np.arange(n) < n // 3 + 1000)


# rows of 1 to 96 chunks (runs of eight, less and more), 2, 3 and 4 bits, every kind of batch; one row past a word, a block and a workgroup's share of the mask
@pytest.mark.parametrize("dim,bits,n,nq", [(64, 4, 65_537, 3), (8, 4, 65_536, 70), (576, 4, 10_001, 40), (1536, 4, 5_000, 300), (6144, 4, 1_003, 5),
                                           (128, 2, 131_073, 1), (1536, 2, 9_001, 12), (256, 2, 66_000, 100), (1000, 3, 6_400, 37), (72, 3, 70_001, 9)])
def test_gathered_rows_give_the_masked_scan_s_bits(T, dim, bits, n, nq):
    ix, gen = filled(T, dim, bits, n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    rng = np.random.default_rng(dim + n)
    for m in masks(n, rng):
        words, allowed = T.pack_mask(m)
        words = words.copy()
        if n % 64:
            words[-1] |= np.uint64(0xFFFFFFFFFFFFFFFF) << np.uint64(n % 64)      # bits past the rows say nothing
        for k in (1, 10, 600) if allowed < 5000 else (10,):
            ix.set_path(MASKED)
            s, i = ix.search(q, k, mask_words=words)
            before = ix.gathered_searches()[0]
            ix.set_path(GATHERED)
            s2, i2 = ix.search(q, k, mask_words=words)
            assert ix.gathered_searches()[0] == before + 1
            assert np.array_equal(i, i2) and bits_equal(s, s2), (allowed, k)
    ix.close()


def test_equal_rows_and_scores_that_are_no_numbers(T):
    """Ties go to the lower slot; queries that were not validated leave the same places empty."""
    dim, n = 64, 40_000
    one = torch.randn(1, dim, device="cuda:0", generator=torch.Generator(device="cuda:0").manual_seed(1))
    v = one.repeat(n, 1).contiguous()
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, 4)
    ix.add_dev(v.data_ptr(), n)
    m = np.random.default_rng(3).random(n) < 0.1
    words, allowed = T.pack_mask(m)
    q = v[:5].cpu().numpy()
    q[1] = np.inf
    q[2, 3] = np.nan
    q[3] = -1e30
    out = []
    for path in (MASKED, GATHERED):
        ix.set_path(path)
        out.append(ix.search(q, 20, mask_words=words))
    assert np.array_equal(out[0][1], out[1][1])
    assert np.array_equal(out[0][0], out[1][0], equal_nan=True)
    assert np.array_equal(out[1][1][0], np.flatnonzero(m)[:20])
    ix.close()


@pytest.mark.parametrize("stated", [-7, 9])
def test_a_count_that_is_not_the_mask_s(T, stated):
    """Device callers state how many rows their mask allows: a wrong statement changes nothing."""
    dim, n, nq, k = 128, 70_000, 40, 10
    ix, gen = filled(T, dim, 4, n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen)
    words, allowed = T.pack_mask(np.random.default_rng(4).random(n) < 0.02)
    mask = torch.from_numpy(words.view(np.int64)).cuda()
    out = []
    for path in (MASKED, GATHERED):
        s, i = torch.zeros(nq, k, device="cuda:0"), torch.zeros(nq, k, dtype=torch.int64, device="cuda:0")
        torch.cuda.synchronize()
        ix.set_path(path)
        ix.search_dev(q.data_ptr(), nq, k, s.data_ptr(), i.data_ptr(), mask.data_ptr(), allowed + stated)
        out.append((s.cpu().numpy(), i.cpu().numpy()))
    assert ix.gathered_searches()[0] == 0
    assert np.array_equal(out[0][1], out[1][1]) and bits_equal(out[0][0], out[1][0])
    ix.close()


def test_where_the_rows_are_gathered(T):
    """Scattered rows of a large batch; not a range of rows, whose blocks are whole, and not a call that is short anyway."""
    dim, n = 1536, 200_000
    ix, gen = filled(T, dim, 4, n)
    q = torch.randn(1024, dim, device="cuda:0", generator=gen).cpu().numpy()
    few = np.random.default_rng(5).random(n) < 0.01
    for m, nq, yes in ((few, 1024, True), (np.arange(n) < 40_000, 1024, False), (few, 1, False), (np.ones(n, bool), 1024, False)):
        words, _ = T.pack_mask(m)
        before = ix.gathered_searches()[0]
        ix.set_path(0)
        s, i = ix.search(q[:nq], 10, mask_words=words)
        assert ix.gathered_searches()[0] == before + yes
        ix.set_path(MASKED)
        s2, i2 = ix.search(q[:nq], 10, mask_words=words)
        assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()


def wide_masks(n, rng):
    m = rng.random(n) < 0.5
    yield m
    m = rng.random(n) < 0.9
    m[[0, n - 1]] = True
    yield m
    yield (np.arange(n) % 64 < 32) | (np.arange(n) > n - 100)


# every instance that reads rows from a list; k large enough for the sampled search, a last block of a few rows
@pytest.mark.parametrize("dim,nq,k", [(768, 300, 60), (768, 1024, 64), (1024, 150, 45), (1536, 130, 30), (1536, 1500, 26), (2048, 140, 20), (3072, 257, 13)])
def test_rows_read_in_place(T, dim, nq, k):
    n = 60_001
    ix, gen = filled(T, dim, 4, n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    for m in wide_masks(n, np.random.default_rng(dim)):
        words, _ = T.pack_mask(m)
        ix.set_path(MASKED)
        s, i = ix.search(q, k, mask_words=words)
        before = ix.gathered_searches()
        ix.set_path(GATHERED)
        s2, i2 = ix.search(q, k, mask_words=words)
        after = ix.gathered_searches()
        assert (after[0] - before[0], after[1] - before[1]) == (1, 1)
        assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()


def test_rows_in_place_whose_candidates_do_not_fit(T):
    """Every row ties, so every candidate passes: the search is done again on a copy, and on the exact path."""
    dim, n, nq, k = 768, 60_001, 140, 60
    one = torch.randn(1, dim, device="cuda:0", generator=torch.Generator(device="cuda:0").manual_seed(1))
    v = one.repeat(n, 1).contiguous()
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, 4)
    ix.add_dev(v.data_ptr(), n)
    m = np.random.default_rng(3).random(n) < 0.5
    words, _ = T.pack_mask(m)
    ix.set_path(GATHERED)
    s, i = ix.search(v[:nq].cpu().numpy(), k, mask_words=words)
    assert ix.gathered_searches() == (1, 0) and ix.exact_redos() > 0
    assert np.array_equal(i, np.tile(np.flatnonzero(m)[:k], (nq, 1)))
    ix.close()


def test_rows_in_place_of_more_than_4_gib(T):
    """Rows of one block 4 GiB of codes apart are copied instead; scattered over such an index they are read in place."""
    dim, n, nq, k = 3072, 2_900_000, 140, 13
    ix, gen = filled(T, dim, 4, n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    ends = np.zeros(n, bool)
    ends[:20_016] = True
    ends[-16:] = True                   # the last block: sixteen rows of either end
    for m, in_place in ((np.random.default_rng(1).random(n) < 0.5, 1), (ends, 0)):
        words, _ = T.pack_mask(m)
        ix.set_path(MASKED)
        s, i = ix.search(q, k, mask_words=words)
        before = ix.gathered_searches()
        ix.set_path(GATHERED)
        s2, i2 = ix.search(q, k, mask_words=words)
        after = ix.gathered_searches()
        assert (after[0] - before[0], after[1] - before[1]) == (1, in_place)
        assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()


# the wide kernel's forms of two waves per SIMD and of one; two groups of queries, one in each (and a third without) to repeat
@pytest.mark.parametrize("dim,nq,k,rows", [(768, 300, 60, [7, 150]), (3072, 140, 13, [139]), (768, 3 * 8192, 60, [5, 8192 + 9])])
def test_only_the_queries_that_do_not_fit_are_repeated(T, dim, nq, k, rows):
    """A few queries find their row stored many times over, in blocks that one workgroup of 256 reads: those queries are
    repeated, once, and the others' results stand."""
    n = 60_001
    gen = torch.Generator(device="cuda:0").manual_seed(7)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen)
    others = torch.ones(nq, dtype=torch.bool, device="cuda:0")
    others[rows] = False
    basis = torch.linalg.qr(q[rows].T.cpu())[0].cuda()
    q[others] -= q[others] @ basis @ basis.T                # at right angles to those rows
    for j, row in enumerate(rows):
        for at in range(1000 + 5000 * j, n - 800, 2 * 256 * 32):      # (every second row is allowed)
            v[at:at + 800] = q[row]
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, 4)
    ix.add_dev(v.data_ptr(), n)
    words, allowed = T.pack_mask(np.random.default_rng(5).random(n) < 0.5)
    mask = torch.from_numpy(words.view(np.int64)).cuda()
    out = []
    for path in (GATHERED, MASKED):
        s, i = torch.zeros(nq, k, device="cuda:0"), torch.zeros(nq, k, dtype=torch.int64, device="cuda:0")
        torch.cuda.synchronize()
        ix.set_path(path)
        ix.search_dev(q.data_ptr(), nq, k, s.data_ptr(), i.data_ptr(), mask.data_ptr(), allowed)
        out.append((s.cpu().numpy(), i.cpu().numpy()))
        if path == GATHERED:
            assert ix.gathered_searches() == (1, 0) and ix.overflow_redos() == len(rows)
    assert np.array_equal(out[0][1], out[1][1]) and bits_equal(out[0][0], out[1][0])
    ix.close()


# the counting workgroups take one piece of 8192 rows to a wave up to 8388608 rows, several beyond
@pytest.mark.parametrize("n", [8_388_608, 8_388_609, 17_000_003])
def test_rows_counted_in_several_turns(T, n):
    ix, gen = filled(T, 8, 4, n)
    q = torch.randn(2, 8, device="cuda:0", generator=gen)
    for m in (np.arange(n) % 97 == 5, np.arange(n) >= n - 70_000):
        words, allowed = T.pack_mask(m)
        mask = torch.from_numpy(words.view(np.int64)).cuda()
        out = []
        for path in (MASKED, GATHERED):
            s, i = torch.zeros(2, 10, device="cuda:0"), torch.zeros(2, 10, dtype=torch.int64, device="cuda:0")
            torch.cuda.synchronize()
            ix.set_path(path)
            before = ix.gathered_searches()[0]
            ix.search_dev(q.data_ptr(), 2, 10, s.data_ptr(), i.data_ptr(), mask.data_ptr(), allowed)
            assert ix.gathered_searches()[0] - before == (path == GATHERED)
            out.append((s.cpu().numpy(), i.cpu().numpy()))
        assert np.array_equal(out[0][1], out[1][1]) and bits_equal(out[0][0], out[1][0])
        ix.set_path(GATHERED)
        ix.search_dev(q.data_ptr(), 2, 10, s.data_ptr(), i.data_ptr(), mask.data_ptr(), allowed - 1)      # not the mask's count
        assert ix.gathered_searches()[0] == before + 1
    ix.close()


# beyond the k of the all-queries scan's floorless level, over more blocks than are searched without sampling
def test_rows_in_place_for_many_results(T):
    n, dim, nq, k = 1_100_000, 768, 140, 100
    ix, gen = filled(T, dim, 4, n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen)
    words, allowed = T.pack_mask(np.random.default_rng(8).random(n) < 0.5)
    mask = torch.from_numpy(words.view(np.int64)).cuda()
    out = []
    for path in (0, MASKED):
        s, i = torch.zeros(nq, k, device="cuda:0"), torch.zeros(nq, k, dtype=torch.int64, device="cuda:0")
        torch.cuda.synchronize()
        ix.set_path(path)
        ix.search_dev(q.data_ptr(), nq, k, s.data_ptr(), i.data_ptr(), mask.data_ptr(), allowed)
        out.append((s.cpu().numpy(), i.cpu().numpy()))
        assert ix.gathered_searches() == (1, 1)
    assert np.array_equal(out[0][1], out[1][1]) and bits_equal(out[0][0], out[1][0])
    ix.close()
