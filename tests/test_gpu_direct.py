"""Searches of small indexes, which score every block and go without sampling: against the oracle, bit for bit."""
import numpy as np
import pytest

from helpers import SAMPLED, OracleIndex, bits_equal, to_native, unit_gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


def unsampled(ix, nq, k, mask=None):
    """Whether the library searches without sampling here: it has no ladder then."""
    return len(ix.sampling_plan(nq, k if mask is None else min(k, int(mask.sum())))[0]) == 0


# One and several tiles of queries, rows of 1 to 72 chunks (odd counts too), indexes of less than a block to
# several rounds of the grid; 768 and 1536 dimensions with 140 queries: the all-queries kernel from 513 blocks on.
@pytest.mark.parametrize("dim,n,nq", [
    (64, 1, 3), (64, 31, 1), (128, 33, 70), (8, 500, 1), (136, 5_001, 9), (200, 20_011, 40), (64, 60_003, 1), (128, 49_000, 300),
    (448, 9_001, 33), (576, 16_500, 257), (768, 17_000, 140), (768, 700, 1025), (1536, 17_001, 129), (1536, 2_001, 65),
    (1536, 40_000, 2), (3072, 1_201, 97), (4608, 333, 2), (4608, 1_003, 130)])
def test_unsampled_search_matches_oracle(T, oracle, dim, n, nq):
    oidx = OracleIndex(oracle, dim, 4, unit_gaussian(n, dim, seed=dim + n))
    q = unit_gaussian(nq, dim, seed=78)
    ix = to_native(T, oidx)
    rng = np.random.default_rng(5)
    redos = 0       # (k = 100 on long rows and several tiles of queries is sampled, and may repeat queries)
    for m in (None, rng.random(n) < 0.5, rng.random(n) < 0.01, (np.arange(n) >= n // 3) & (np.arange(n) < n // 3 + 40)):
        if m is not None and not m.any():
            m[0] = True
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 10 if dim <= 3840 else 8, 100):      # (k times the chunks of a row is bounded)
            assert k == 100 or unsampled(ix, nq, k, m)
            s, i = ix.search(q, k, mask_words=words)
            os_, oi = oidx.search(q, k, mask_words=words)
            assert np.array_equal(i, oi) and bits_equal(s, os_), k
            assert not unsampled(ix, nq, k, m) or ix.overflow_redos() == redos
        redos = ix.overflow_redos()
    ix.close()


@pytest.mark.parametrize("dim,nq", [(128, 1), (128, 300), (768, 140)])
def test_ties_and_wild_row_scales(T, oracle, dim, nq):
    """Equal rows: every block and every row of the chosen blocks ties, the lowest slots come back.  Row scales of
    zero, of either sign and far from the encoder's: the same answer as the exact path's."""
    n = 30_000
    oidx = OracleIndex(oracle, dim, 4, np.tile(unit_gaussian(1, dim, seed=3), (n, 1)))
    q = unit_gaussian(nq, dim, seed=4)
    ix = to_native(T, oidx)
    for k in (10, 40):
        assert unsampled(ix, nq, k)
        s, i = ix.search(q, k)
        os_, oi = oidx.search(q, k)
        assert ix.overflow_redos() == 0
        assert np.array_equal(i, np.tile(np.arange(k), (nq, 1)))
        assert np.array_equal(i, oi) and bits_equal(s, os_)
    ix.close()
    oidx = OracleIndex(oracle, dim, 4, unit_gaussian(n, dim, seed=5))
    rng = np.random.default_rng(6)
    oidx.scales = (oidx.scales * rng.choice(np.array([0.0, 1e-38, -1.0, 1.0, 1e6], np.float32), size=n)).astype(np.float32)
    ix = to_native(T, oidx)
    for k in (10, 40):
        assert unsampled(ix, nq, k)
        s, i = ix.search(q, k)
        ix.set_path(1)
        s2, i2 = ix.search(q, k)
        ix.set_path(0)
        assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()


@pytest.mark.parametrize("nq", [2, 300])
def test_best_blocks_in_any_place(T, oracle, nq):
    """More blocks that tie than are ranked as they are, and allowed rows in blocks a thousand apart only, which one thread of the
    selection holds: no more are taken for the best than are."""
    n, dim = 70_000, 64
    v = unit_gaussian(n, dim, seed=21)
    v[:40_000] = v[0]
    oidx = OracleIndex(oracle, dim, 4, v)
    q = np.concatenate([v[:1] + np.float32(0.01) * unit_gaussian(1, dim, seed=22), unit_gaussian(nq - 1, dim, seed=23)])
    ix = to_native(T, oidx)
    block = np.arange(n) // 32
    for m in (None, block % 1024 == 3, (block % 256 == 5) & (np.arange(n) % 32 == 7)):
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 16, 17, 100):
            assert unsampled(ix, nq, k, m)
            s, i = ix.search(q, k, mask_words=words)
            os_, oi = oidx.search(q, k, mask_words=words)
            assert np.array_equal(i, oi) and bits_equal(s, os_), k
    assert ix.overflow_redos() == 0
    ix.close()


@pytest.mark.parametrize("dim,nq", [(64, 3), (64, 257), (768, 33), (1536, 300)])
@pytest.mark.parametrize("n", [1, 33, 1025, 4096, 4097])
def test_few_rows(T, oracle, n, dim, nq):
    """Up to 4096 rows every row's score is kept: on either side of that, of a filter's rows too, and with rows that tie."""
    v = unit_gaussian(n, dim, seed=n + dim)
    v[n // 2:n // 2 + 1500] = v[0]
    oidx = OracleIndex(oracle, dim, 4, v)
    q = unit_gaussian(nq, dim, seed=31)
    q[0] = v[0]
    ix = to_native(T, oidx)
    for m in (None, np.random.default_rng(3).random(n) < 0.3, np.arange(n) % 32 == 31):
        if m is not None and not m.any():
            m[0] = True
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 16, 17, 100):
            # (rows of which the search has room for a score are never sampled; a query that came up short would be repeated)
            kept, redos = min(k, n if m is None else int(m.sum())), ix.overflow_redos()
            if n <= 4096 and (nq <= 256 or n <= 75 * kept * dim // 64):
                assert unsampled(ix, nq, k, m), k
            s, i = ix.search(q, k, mask_words=words)
            os_, oi = oidx.search(q, k, mask_words=words)
            assert np.array_equal(i, oi) and bits_equal(s, os_), k
            assert not unsampled(ix, nq, k, m) or ix.overflow_redos() == redos
    ix.close()


# Long rows and few queries: the chosen blocks are dealt out to several workgroups (24 to 48 chunks times k; of tables three times that),
# all of whose rows tie -- every one's share is full, and up to 3200 rows are left to rank -- or all but a few of which score -infinity.
@pytest.mark.parametrize("dim,bits,n,nq", [(1536, 4, 30_000, 1), (1536, 4, 10_001, 33), (3072, 4, 5_001, 2), (1536, 2, 30_000, 1), (1024, 3, 9_999, 7)])
def test_shared_blocks_that_tie(T, oracle, dim, bits, n, nq):
    oidx = OracleIndex(oracle, dim, bits, np.tile(unit_gaussian(1, dim, seed=3), (n, 1)))
    q = unit_gaussian(nq, dim, seed=4)
    ix = to_native(T, oidx)
    third = (np.arange(n) % 96 < 32) & (np.arange(n) % 3 == 0)      # (of every third block)
    ran = 0
    for m in (None, third):
        words = None if m is None else T.pack_mask(m)[0]
        first = np.arange(n) if m is None else np.flatnonzero(m)
        for k in (9, 30, 63, 100):
            ran += unsampled(ix, nq, k, m)
            redos = ix.overflow_redos()
            s, i = ix.search(q, k, mask_words=words)
            os_, oi = oidx.search(q, k, mask_words=words)
            assert np.array_equal(i, np.tile(first[:k], (nq, 1)))
            assert np.array_equal(i, oi) and bits_equal(s, os_), k
            assert not unsampled(ix, nq, k, m) or ix.overflow_redos() == redos, k
    assert ran >= (8 if nq == 1 else 2)
    ix.close()


@pytest.mark.parametrize("k", [9, 20, 60])
def test_shared_blocks_of_minus_infinity(T, oracle, k):
    dim, n = 1536, 4_200
    oidx = OracleIndex(oracle, dim, 4, unit_gaussian(n, dim, seed=1))
    q = unit_gaussian(1, dim, seed=2) * np.float32(1e6)
    ix = to_native(T, oidx)
    raw = ix.debug_scan(q)[1][0]
    ix.close()
    oidx.scales = (np.float32(3e38) * -np.sign(raw)).astype(np.float32)
    finite = [40, 41, 1050, 1060, 2000, 3000, 3500, 3600, 3700, 4000, 4100, 4199]
    oidx.scales[finite] = 1.0
    ix = to_native(T, oidx)
    assert unsampled(ix, 1, k)
    s, i = ix.search(q, k)
    os_, oi = oidx.search(q, k)
    assert np.isneginf(os_[0, len(finite):]).all() and np.isfinite(os_[0, :len(finite)]).all()
    assert np.array_equal(i, oi) and bits_equal(s, os_)
    assert ix.overflow_redos() == (1 if k > len(finite) else 0)      # (-infinity does not count: such a query goes to the exact path)
    ix.close()


@pytest.mark.parametrize("k", [3, 10, 60])
def test_rows_that_score_minus_infinity(T, oracle, k):
    """Row scales that take most rows' scores beyond the float range: the blocks of the few finite rows hold -infinity
    too, and rows of other blocks with lower slots tie with it."""
    dim, n = 64, 96
    oidx = OracleIndex(oracle, dim, 4, unit_gaussian(n, dim, seed=1))
    q = unit_gaussian(1, dim, seed=2) * np.float32(1e6)
    ix = to_native(T, oidx)
    raw = ix.debug_scan(q)[1][0]
    ix.close()
    oidx.scales = (np.float32(3e38) * -np.sign(raw)).astype(np.float32)
    oidx.scales[[40, 41, 50, 60]] = 1.0
    ix = to_native(T, oidx)
    assert unsampled(ix, 1, k)
    s, i = ix.search(q, k)
    os_, oi = oidx.search(q, k)
    assert np.isneginf(os_[0, 4:]).all() and np.isfinite(os_[0, :4]).all()
    assert np.array_equal(i, oi) and bits_equal(s, os_)
    ix.close()


def test_scan_time_leaves_out_the_preparation(T):
    """A TQ+ pair makes preparing a query take 40 us longer (a chain of f64 additions) and the scan no longer.  1024
    queries of 4608 dimensions are two rounds of the chip's workgroups in preparation, one block in the scan."""
    torch = pytest.importorskip("torch")
    dim, nq, k = 4608, 1024, 5
    q = torch.from_numpy(unit_gaussian(nq, dim, seed=9)).to("cuda:0")
    s = torch.zeros(nq, k, device="cuda:0")
    i = torch.zeros(nq, k, dtype=torch.int64, device="cuda:0")
    torch.cuda.synchronize()
    least = []
    for calibrated in (False, True):
        ix = T.NativeIndex(dim, 4)
        if calibrated:
            ix.calibrate(unit_gaussian(64, dim, seed=7))
        ix.add(unit_gaussian(32, dim, seed=8))
        ms = []
        for _ in range(10):
            ix.search_dev(q.data_ptr(), nq, k, s.data_ptr(), i.data_ptr())
            ms.append(ix.last_scan_ms())
        assert unsampled(ix, nq, k)
        assert all(launches == 1 for _, launches in ms)
        least.append(min(ms)[0])
        ix.close()
    assert least[1] < least[0] + 0.020, least


@pytest.mark.parametrize("mode,nq,launches", [("L_CLASSIC", 1024, 64), ("L_CLASSIC", 80, 5), ("L_SCALAR", 40, 40), ("L_U32", 1024, 1)])
def test_every_launch_of_the_timed_scan_counts(T, mode, nq, launches):
    ix = T.NativeIndex(64, 2)
    ix.set_score_mode(getattr(T, "SCORE_" + mode))
    ix.set_path(SAMPLED)
    ix.add(unit_gaussian(70_000, 64, seed=5))
    ix.search(unit_gaussian(nq, 64, seed=6), 10)
    assert len(ix.sampling_plan(nq, 10)[0]) == 2      # a level before the full scan: timed between stamps
    assert ix.last_scan_ms()[1] == launches
    ix.close()


# The number of blocks a thread of the last launch keeps changes behind 16384, and 32768 are its most; 1048577 rows
# are sampled.  Batches of a few queries, of several tiles and of more than a launch's worth.
@pytest.mark.parametrize("dim,n,nq", [(64, 524_288, 9), (64, 524_289, 70), (128, 1_048_576, 1), (128, 1_048_577, 1), (64, 1_048_545, 200),
                                      (128, 60_001, 1030), (768, 100_003, 5), (768, 600_000, 130), (1024, 540_000, 64)])
def test_unsampled_search_agrees_with_the_sampled_one(T, dim, n, nq):
    torch = pytest.importorskip("torch")
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, 4)
    for at in range(0, n, 262_144):
        v = torch.randn(min(262_144, n - at), dim, device="cuda:0", generator=gen)
        if at == 0:
            v[1000:1100] = v[:100]       # equal rows
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), len(v))
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    rng = np.random.default_rng(5)
    for m, k in ((None, 1), (None, 10), (rng.random(n) < 0.02, 12)):
        words = None if m is None else T.pack_mask(m)[0]
        assert unsampled(ix, nq, k, m) == (n <= 1_048_576)
        res = []
        for path in (0, 16):
            ix.set_path(path)
            res.append(ix.search(q, k, mask_words=words))
        ix.set_path(0)
        assert np.array_equal(res[0][1], res[1][1]) and bits_equal(res[0][0], res[1][0]), k
    ix.close()
