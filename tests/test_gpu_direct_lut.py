"""u8-LUT searches (u32 epilogue) without sampling: every scan kernel's best-of-block form and the second scoring, against
the oracle and against the sampled search."""
import numpy as np
import pytest

from helpers import SAMPLED, OracleIndex, bits_equal, to_native, unit_gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


# One query (byte tables whole and in part), a few (whole tables: 1, 2, 4 or 8 of them in LDS), up to sixteen (streamed), several
# such tiles side by side with a last one of one query, and the matrix-unit scan (4096 pairs of a block and a tile on);
# rows of 1 to 48 chunks, odd counts, 4-bit tables; last blocks of 1, 31 and 32 rows.
@pytest.mark.parametrize("dim,bits,n,nq", [
    (128, 2, 270_001, 1), (1536, 2, 22_031, 1), (1024, 3, 17_000, 1), (3072, 3, 6_001, 1),
    (128, 2, 33, 2), (128, 2, 5_001, 8), (64, 3, 9_985, 5), (768, 2, 9_000, 7), (1536, 3, 3_001, 3), (3072, 3, 1_201, 2),
    (128, 2, 31, 9), (200, 2, 30_000, 16), (1536, 3, 3_001, 10), (1120, 2, 1, 16), (576, 3, 9_001, 33), (3072, 2, 2_001, 49), (512, 4, 5_000, 17),
    (128, 2, 131_103, 32), (136, 2, 70_000, 65), (1120, 2, 20_011, 200), (576, 3, 30_001, 300), (96, 4, 131_072, 20)])
def test_unsampled_lut_search_matches_oracle(T, oracle, dim, bits, n, nq):
    oidx = OracleIndex(oracle, dim, bits, unit_gaussian(n, dim, seed=dim + n))
    q = unit_gaussian(nq, dim, seed=81)
    ix = to_native(T, oidx, T.SCORE_L_U32)
    rng = np.random.default_rng(5)
    for m in (None, rng.random(n) < 0.5, rng.random(n) < 0.01, (np.arange(n) >= n // 3) & (np.arange(n) < n // 3 + 40)):
        if m is not None and not m.any():
            m[0] = True
        words = None if m is None else T.pack_mask(m)[0]
        for k in (1, 8, 30):
            kk = k if m is None else min(k, int(m.sum()))
            if k <= 8:
                assert len(ix.sampling_plan(nq, kk)[0]) == 0
            s, i = ix.search(q, k, mask_words=words)
            os_, oi = oidx.search(q, k, mask_words=words, mode=oracle.MODE_L_U32)
            assert np.array_equal(i, oi) and bits_equal(s, os_), k
    assert ix.overflow_redos() == 0
    ix.set_path(SAMPLED)
    s2, i2 = ix.search(q, 30, mask_words=words)
    assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()


@pytest.mark.parametrize("nq", [3, 12, 40])
def test_calibrated_ties_and_wild_row_scales(T, oracle, nq):
    """Equal rows: the lowest slots; row scales of zero, of either sign and far from the encoder's: as the exact path."""
    dim, n = 256, 70_000
    cal = (unit_gaussian(1, dim, seed=6)[0] * np.float32(0.1), np.linspace(0.5, 2.0, dim, dtype=np.float32))
    oidx = OracleIndex(oracle, dim, 2, np.tile(unit_gaussian(1, dim, seed=3), (n, 1)), calibration=cal)
    q = unit_gaussian(nq, dim, seed=4)
    ix = to_native(T, oidx)
    s, i = ix.search(q, 20)
    os_, oi = oidx.search(q, 20)
    assert len(ix.sampling_plan(nq, 20)[0]) == 0 and ix.overflow_redos() == 0
    assert np.array_equal(i, np.tile(np.arange(20), (nq, 1))) and np.array_equal(i, oi) and bits_equal(s, os_)
    ix.close()
    oidx = OracleIndex(oracle, dim, 2, unit_gaussian(n, dim, seed=5), calibration=cal)
    rng = np.random.default_rng(6)
    oidx.scales = (oidx.scales * rng.choice(np.array([0.0, 1e-38, -1.0, 1.0, 1e6, np.inf], np.float32), size=n)).astype(np.float32)
    ix = to_native(T, oidx)
    s, i = ix.search(q, 20)
    ix.set_path(1)
    s2, i2 = ix.search(q, 20)
    assert np.array_equal(i, i2) and bits_equal(s, s2)
    ix.close()
