"""u8-LUT batches in two steps -- an int8 scan that tells which rows may reach the floor (k_scan_p4_wide on 2- and 3-bit codes),
then those rows from the tables (k_near_rescore) -- bit for bit against the exact path and the oracle."""
import numpy as np
import pytest

from helpers import OracleIndex, bits_equal, to_native, unit_gaussian

pytestmark = pytest.mark.gpu
torch = pytest.importorskip("torch")
TWO_STEP = 128      # set_path: wherever there is an instance


def check(ix, q, ks=(1, 10, 100), always=True):
    for k in ks:
        ix.set_path(1)
        s1, i1 = ix.search(q, k)
        ix.set_path(TWO_STEP)
        for _ in range(2):
            s, i = ix.search(q, k)
            assert ix.last_scan_ms()[1] >= 2 or not always       # (launches: both steps')
            assert np.array_equal(i, i1) and bits_equal(s, s1), k


# Every instance (chunks of 64 dimensions: 2 to 24 and 28 to 48), rows that fill it and rows a chunk short of it or ragged; over a
# round of the grid and part of another; last groups of one block and of seven, last blocks of 1, 31 and 32 rows; query
# tiles of 1 and 31 queries, query groups of the second step cut short.
@pytest.mark.parametrize("dim,bits,n,nq", [
    (64, 2, 600_001, 33), (256, 2, 410_031, 65), (384, 2, 310_000, 95), (504, 2, 210_001, 161), (640, 2, 210_223, 67), (768, 2, 105_001, 130),
    (896, 2, 105_015, 33), (1024, 2, 105_001, 97), (1152, 2, 105_017, 34), (1280, 2, 105_250, 129), (1400, 2, 105_001, 70), (1536, 2, 105_239, 1024),
    (1664, 2, 55_001, 65), (1920, 2, 55_001, 40), (2048, 2, 55_000, 65), (2176, 2, 55_003, 33), (2560, 2, 55_031, 66), (2816, 2, 55_001, 35),
    (3072, 2, 55_017, 100),
    (64, 3, 600_031, 40), (192, 3, 410_001, 66), (256, 3, 410_001, 33), (384, 3, 310_001, 129), (512, 3, 210_015, 35), (640, 3, 210_001, 65),
    (704, 3, 105_001, 33), (896, 3, 105_031, 99), (1000, 3, 105_001, 65), (1152, 3, 105_001, 34), (1216, 3, 105_003, 65), (1408, 3, 105_001, 36),
    (1536, 3, 105_033, 70)])
def test_instances_match_exact_path(dim, bits, n, nq):
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + n)
    ix = T.NativeIndex(dim, bits)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    check(ix, torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy())
    ix.close()


@pytest.mark.parametrize("dim,bits,n,nq,calibrated", [(256, 2, 450_015, 40, False), (200, 3, 320_003, 33, True), (768, 2, 110_001, 65, True)])
def test_matches_oracle(oracle, dim, bits, n, nq, calibrated):
    from turbovec_amd import _lib as T
    rng = np.random.default_rng(5)
    pair = (rng.normal(0, 0.02, dim).astype(np.float32), rng.uniform(0.8, 1.25, dim).astype(np.float32)) if calibrated else None
    oidx = OracleIndex(oracle, dim, bits, unit_gaussian(n, dim, seed=21), pair)
    ix = to_native(T, oidx, T.SCORE_L_U32)
    ix.set_path(TWO_STEP)
    q = unit_gaussian(nq, dim, seed=22)
    for k in (3, 64):
        os_, oi = oidx.search(q, k, mode=oracle.MODE_L_U32)
        s, i = ix.search(q, k)
        assert ix.last_scan_ms()[1] >= 2
        assert np.array_equal(i, oi) and bits_equal(s, os_)
    ix.close()


@pytest.mark.parametrize("dim,bits,n,nq", [(128, 2, 700_017, 70), (1000, 3, 150_003, 33), (1536, 2, 150_031, 97)])
def test_filters(dim, bits, n, nq):
    """Masks read as the rows are, and searches of the allowed rows' copies."""
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim)
    ix = T.NativeIndex(dim, bits)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    rng = np.random.default_rng(n)
    for m in (rng.random(n) < 0.9, rng.random(n) < 0.3, np.arange(n) >= n // 2, np.arange(n) % 64 < 32):
        words = T.pack_mask(m)[0]
        for k in (1, 40):
            ix.set_path(1)
            s1, i1 = ix.search(q, k, mask_words=words)
            for path in (TWO_STEP, TWO_STEP + 64):
                ix.set_path(path)
                s, i = ix.search(q, k, mask_words=words)
                assert ix.last_scan_ms()[1] >= 2, path
                assert np.array_equal(i, i1) and bits_equal(s, s1), path
    few = T.pack_mask(rng.random(n) < 0.0005)[0]            # too few for a sample's floor: the other scans
    ix.set_path(1)
    s1, i1 = ix.search(q, 10, mask_words=few)
    ix.set_path(TWO_STEP)
    s, i = ix.search(q, 10, mask_words=few)
    assert np.array_equal(i, i1) and bits_equal(s, s1)
    ix.close()


def test_row_scales_without_a_bound(oracle):
    """Scales that are zero, negative, subnormal, huge, infinite or no number, and rows that tie."""
    from turbovec_amd import _lib as T
    dim, n = 128, 700_031
    v = unit_gaussian(n, dim, seed=31)
    v[70_000:70_300] = v[:300]
    oidx = OracleIndex(oracle, dim, 2, v)
    odd = np.array([0.0, -0.0, -1.0, 1e-38, 1e-42, -np.inf, np.nan, 3.0], np.float32)
    at = np.random.default_rng(1).choice(n, 4000, replace=False)
    oidx.scales[at] = odd[np.arange(4000) % len(odd)]
    ix = to_native(T, oidx, T.SCORE_L_U32)
    q = np.concatenate([unit_gaussian(40, dim, seed=32), v[:8], -v[:8]])
    check(ix, q, (1, 10, 100), always=False)            # (rows at -inf times a negative sum come first: floors are open)
    ix.close()
    oidx.scales[at] = np.where(np.isinf(oidx.scales[at]), np.float32(1e31), oidx.scales[at])
    ix = to_native(T, oidx, T.SCORE_L_U32)
    check(ix, q, (10,), always=False)                   # (floors beyond what the bound is made for)
    ix.close()
    oidx.scales[at] = np.where(oidx.scales[at] > 1e30, np.float32(0.0), oidx.scales[at])
    ix = to_native(T, oidx, T.SCORE_L_U32)
    check(ix, q)
    ix.close()
    oidx.scales[:] = -np.abs(oidx.scales)
    ix = to_native(T, oidx, T.SCORE_L_U32)
    check(ix, q, (10,), always=False)                   # (no row has a bound)
    ix.close()


def test_neighbours_that_lie_together():
    """A query's neighbours are one run of rows, seven blocks full of them."""
    from turbovec_amd import _lib as T
    dim, n, nq, k = 64, 820_000, 96, 100
    gen = torch.Generator(device="cuda:0").manual_seed(8)
    centres = torch.randn(n // 200, dim, device="cuda:0", generator=gen)
    v = centres.repeat_interleave(200, 0) + 0.15 * torch.randn(n, dim, device="cuda:0", generator=gen)
    ix = T.NativeIndex(dim, 2)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    check(ix, centres[:: len(centres) // nq][:nq].cpu().numpy(), (k, 33))
    ix.close()


def test_neighbours_of_the_first_stage():
    """All of a query's best rows are among the first rows looked at (groups x * mul % total of a golden-section order, eight
    blocks each): the floor guessed from them is too high, and the query is repeated."""
    from turbovec_amd import _lib as T
    dim, n, nq, k = 64, 2_000_000, 200, 100
    total = -(-(-(-n // 32)) // 8)
    mul = int(total * 0.6180339887498949)
    while np.gcd(mul, total) != 1:
        mul += 1
    blocks = [x * mul % total + w * total for x in range(64) for w in range(8)]
    slots = (np.array([b for b in blocks if b < n // 32])[:, None] * 32 + np.arange(32)).ravel()
    gen = torch.Generator(device="cuda:0").manual_seed(8)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    near = np.random.default_rng(4).permutation(slots)[: 40 * 120]
    v[torch.from_numpy(near).cuda()] = q[:40].repeat_interleave(120, 0) + 0.3 * torch.randn(4800, dim, device="cuda:0", generator=gen)
    ix = T.NativeIndex(dim, 2)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    ix.set_path(1)
    s1, i1 = ix.search(q.cpu().numpy(), k)
    ix.set_path(TWO_STEP)
    redos = []
    for _ in range(3):
        before = ix.overflow_redos()
        s, i = ix.search(q.cpu().numpy(), k)
        assert ix.last_scan_ms()[1] >= 2
        assert np.array_equal(i, i1) and bits_equal(s, s1)
        redos.append(ix.overflow_redos() - before)
    assert redos[0] >= 40 and max(redos[1:]) < 10           # (an eighth and more: the next searches take floors that are sure)
    ix.close()


def test_equal_rows(oracle):
    """All rows tie: every row is in, workgroups give up, and the lowest slots must come back."""
    from turbovec_amd import _lib as T
    dim, n = 64, 131_080
    oidx = OracleIndex(oracle, dim, 2, np.tile(unit_gaussian(1, dim, seed=3), (n, 1)))
    ix = to_native(T, oidx, T.SCORE_L_U32)
    ix.set_path(TWO_STEP)
    q = unit_gaussian(40, dim, seed=4)
    for k in (10, 40):
        s, i = ix.search(q, k)
        os_, oi = oidx.search(q, k, mode=oracle.MODE_L_U32)
        assert np.array_equal(i, oi) and bits_equal(s, os_)
    assert ix.overflow_redos() > 0
    ix.close()


def test_queries_that_are_not_finite():
    """Host arrays passed unchecked: rows of infinities and NaN leave the other queries' results alone."""
    from turbovec_amd import _lib as T
    dim, n = 128, 700_000
    gen = torch.Generator(device="cuda:0").manual_seed(9)
    ix = T.NativeIndex(dim, 2)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    q = torch.randn(70, dim, device="cuda:0", generator=gen).cpu().numpy()
    ix.set_path(1)
    s1, i1 = ix.search(q, 10)
    bad = q.copy()
    bad[5] = np.nan
    bad[17, 3] = np.inf
    bad[40] = 0.0
    bad[41] *= np.float32(1e-30)
    ix.set_path(TWO_STEP)
    s, i = ix.search(bad, 10)
    good = [r for r in range(70) if r not in (5, 17, 40, 41)]
    assert np.array_equal(i[good], i1[good]) and bits_equal(s[good], s1[good])
    ix.close()


@pytest.mark.parametrize("bits,nq", [(2, 400), (3, 65)])
def test_fewer_blocks_than_a_sample(bits, nq):
    """The hook asks for two steps where there is no sample to take a floor from: the other scans."""
    from turbovec_amd import _lib as T
    dim = 64
    gen = torch.Generator(device="cuda:0").manual_seed(bits)
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    for n in (1, 31, 96, 97, 129):
        ix = T.NativeIndex(dim, bits)
        v = torch.randn(n, dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), n)
        check(ix, q, (1, 10), always=False)
        ix.close()


@pytest.mark.parametrize("dim,bits,n", [(128, 2, 700_000), (128, 3, 700_001), (1536, 2, 105_239), (3072, 2, 55_017)])
def test_queries_of_zero_and_of_extreme_size(dim, bits, n):
    """Valid queries that no bound can be had for (zero, and so small or large that a unit of their tables is out of range), among others."""
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(dim + bits)
    ix = T.NativeIndex(dim, bits)
    v = torch.randn(n, dim, device="cuda:0", generator=gen)
    torch.cuda.synchronize()
    ix.add_dev(v.data_ptr(), n)
    q = torch.randn(70, dim, device="cuda:0", generator=gen).cpu().numpy()
    q[40] = 0.0
    for row, size in ((41, 1e-30), (3, 1e-19), (12, 1e-25), (32, 1e-36), (50, 1e-44), (63, 1e15), (64, 1e25), (69, 1e33)):
        q[row] *= np.float32(size)
    q[20] = 0.0
    q[20, 1] = 1.0
    assert np.isfinite(q).all()
    ix.set_path(1)
    s1, i1 = ix.search(q, 10)
    ix.set_path(TWO_STEP)
    s, i = ix.search(q, 10)
    assert ix.last_scan_ms()[1] >= 2
    assert np.array_equal(i, i1) and bits_equal(s, s1)
    check(ix, q, always=False)      # (so many queries repeated, with those that share their workgroups, have the searches after it go other ways)
    ix.close()


@pytest.mark.parametrize("dim,bits,n,nq,two_step", [
    (768, 2, 342_848, 200, False), (768, 2, 342_849, 200, True), (64, 2, 3_400_001, 64, False), (64, 2, 3_400_001, 65, True),
    (256, 3, 738_432, 400, False), (256, 3, 738_433, 400, True)])
def test_where_it_starts(dim, bits, n, nq, two_step):
    """What users get, with and without a filter, on both sides of the least blocks and queries."""
    from turbovec_amd import _lib as T
    gen = torch.Generator(device="cuda:0").manual_seed(n)
    ix = T.NativeIndex(dim, bits)
    for at in range(0, n, 400_000):
        v = torch.randn(min(400_000, n - at), dim, device="cuda:0", generator=gen)
        torch.cuda.synchronize()
        ix.add_dev(v.data_ptr(), len(v))
    q = torch.randn(nq, dim, device="cuda:0", generator=gen).cpu().numpy()
    words = T.pack_mask(np.random.default_rng(n).random(n) < 0.95)[0]
    some = np.unique(np.linspace(0, nq - 1, 40).astype(int))
    for m in (None, words):
        ix.set_path(1)
        s1, i1 = ix.search(q[some], 3, mask_words=m)
        ix.set_path(0)
        for _ in range(2):
            s, i = ix.search(q, 3, mask_words=m)
            if m is None:       # (launches: both steps')
                assert (ix.last_scan_ms()[1] >= 2) == two_step
            assert np.array_equal(i[some], i1) and bits_equal(s[some], s1)
    ix.close()
