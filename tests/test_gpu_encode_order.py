"""Where the encoder's shortcuts apply and where they do not, against the oracle byte for byte: a boundary found through
its cell or by comparing with all of them, and the row scale's f64 sum taken in any order or in the reference's."""
import numpy as np
import pytest

from helpers import bits_equal, unit_gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


def encoded(T, O, v, bits, calibration=None, centroids=None):
    n, dim = v.shape
    ix = T.NativeIndex(dim, bits)
    if centroids is not None:
        ix.set_tables(centroids=centroids)
    if calibration is not None:
        ix.set_calibration(*calibration)
    ix.add(v)
    seq, scales = ix.download_seq()
    ix.close()
    if centroids is None:
        packed, want = O.encode(O.Rotation(dim), v, bits, calibration)
    else:
        b = (centroids[:-1] + centroids[1:]) * np.float32(0.5)
        packed, want = np.zeros((n, bits * dim // 8), np.uint8), np.zeros(n, np.float32)
        rot = O.Rotation(dim)
        O.lib().tvo_encode(rot.h, O._p(v), n, dim, bits, O._p(b), O._p(centroids), None, None, O._p(packed), O._p(want))
    return seq, scales, O.repack_seq(packed, n, bits, dim), want


# rows of 8 to 64 lanes, of one to eight groups of elements per lane; a last workgroup that is not full
@pytest.mark.parametrize("dim,bits", [(8, 4), (24, 2), (136, 3), (512, 4), (520, 4), (1000, 2), (1536, 3), (2048, 4), (2056, 4), (3072, 2), (4096, 4)])
def test_every_row_width(T, oracle, dim, bits):
    v = unit_gaussian(1203, dim, seed=dim) * np.float32(2.5)
    for cal in (None, (unit_gaussian(1, dim, seed=3)[0] * np.float32(0.2), np.linspace(0.5, 2.0, dim, dtype=np.float32))):
        seq, scales, want_seq, want = encoded(T, oracle, v, bits, calibration=cal)
        assert np.array_equal(seq, want_seq) and bits_equal(scales, want)


# every number of butterfly stages: within a lane, between lanes of a row of sixteen, between rows of sixteen, between a lane's
# groups; rows that leave lanes and groups idle; a single row, and one more or less than workgroups hold
@pytest.mark.parametrize("dim", [16, 32, 64, 128, 192, 256, 640, 768, 1024, 1040, 1792, 2560, 3464, 3584, 4096])
def test_every_block_size(T, oracle, dim):
    for n, bits in ((1, 4), (63, 3), (65, 2)):
        v = unit_gaussian(n, dim, seed=dim + n) * np.float32(0.7)
        v[0, 0] = 0.0
        for cal in (None, (unit_gaussian(1, dim, seed=4)[0] * np.float32(0.1), np.linspace(2.0, 0.5, dim, dtype=np.float32))):
            seq, scales, want_seq, want = encoded(T, oracle, v, bits, calibration=cal)
            assert np.array_equal(seq, want_seq) and bits_equal(scales, want)


# A pair with a large shift: the terms are some dim^(1/2) times larger than their sum, and about one row in 7000 (2048
# dimensions) or 2500 (4096) lies closer to a rounding boundary than the two orders of addition can differ.
@pytest.mark.parametrize("dim,n,shift", [(1536, 30_000, 1e8), (2048, 20_000, 1e8), (4096, 8_000, 1e8), (256, 4_000, 1e14)])
def test_sums_near_a_rounding_boundary(T, oracle, dim, n, shift):
    v = unit_gaussian(n, dim, seed=dim + 1)
    rng = np.random.default_rng(dim)
    cal = ((rng.standard_normal(dim) * shift).astype(np.float32), np.ones(dim, np.float32))
    seq, scales, want_seq, want = encoded(T, oracle, v, 4, calibration=cal)
    assert np.array_equal(seq, want_seq) and bits_equal(scales, want)
    assert (want > 0).any()


# sixteen levels in equal steps (a cell each), two of them close together (two boundaries in a cell: compared one by
# one), all of them far beyond the values, all equal
@pytest.mark.parametrize("levels", [np.linspace(-0.09, 0.09, 16), np.r_[np.linspace(-0.09, 0.0, 8), 1e-4, np.linspace(0.01, 0.09, 7)],
                                    np.linspace(-50, 50, 16), np.full(16, 0.02), np.linspace(-1e-30, 1e-30, 16)])
def test_handed_over_levels(T, oracle, levels):
    v = unit_gaussian(777, 768, seed=11)
    v[3] = 0.0
    seq, scales, want_seq, want = encoded(T, oracle, v, 4, centroids=np.ascontiguousarray(levels, np.float32))
    assert np.array_equal(seq, want_seq) and bits_equal(scales, want)


def test_rows_with_values_that_are_no_numbers(T, oracle):
    """Rows on the device are not checked; a row with NaN or infinity in it gets what the reference's operations give."""
    torch = pytest.importorskip("torch")
    dim, n = 256, 70
    v = unit_gaussian(n, dim, seed=12)
    v[1, 5], v[2, 7], v[3, 9], v[4] = np.nan, np.inf, -np.inf, 1e30
    d = torch.from_numpy(v).cuda()
    torch.cuda.synchronize()
    ix = T.NativeIndex(dim, 4)
    ix.add_dev(d.data_ptr(), n)
    seq, scales = ix.download_seq()
    ix.close()
    packed, want = oracle.encode(oracle.Rotation(dim), v, 4)
    assert np.array_equal(seq, oracle.repack_seq(packed, n, 4, dim))
    assert np.array_equal(np.isnan(scales), np.isnan(want)) and bits_equal(scales[~np.isnan(want)], want[~np.isnan(want)])


class _Bytes:
    """Device memory as torch takes it."""

    def __init__(self, ptr, count):
        self.__cuda_array_interface__ = dict(shape=(count,), typestr="|u1", data=(ptr, False), version=2)


@pytest.mark.parametrize("dim,bits,pieces", [(1000, 4, (20_000, 33, 40_000, 1)), (1536, 2, (40_000, 31, 64, 9_000)), (4104, 4, (3_000, 100, 4_000))])
def test_grown_indexes_hold_nothing_else(T, dim, bits, pieces):
    """Rows added in pieces to an index that grows into memory another one gave up: padding, lanes without a row and scales
    are those of an index uploaded whole, and rows appended later land in cleared blocks."""
    torch = pytest.importorskip("torch")
    n = sum(pieces)
    x = torch.randn(2 * n, dim, device="cuda")
    torch.cuda.synchronize()
    dirty = T.NativeIndex(dim, bits)
    dirty.add_dev(x.data_ptr(), 2 * n)
    dirty.close()
    ix, at = T.NativeIndex(dim, bits), 0
    for rows in pieces:
        ix.add_dev(x[at:].data_ptr(), rows)
        at += rows
    seq, scales = ix.download_seq()
    whole = T.NativeIndex(dim, bits)
    whole.upload_seq(seq, n, scales)

    def contents(index):
        codes, row_scales, code_bytes = index.device_ptrs()
        return [torch.as_tensor(_Bytes(p, b), device="cuda").cpu().numpy() for p, b in ((codes, code_bytes), (row_scales, (len(index) + 31) // 32 * 128))]

    for index in (ix, whole):
        index.append_rows(np.full((1, index.n_byte_groups), 0x55, np.uint8), np.ones(1, np.float32))
    for got, want in zip(contents(ix), contents(whole)):
        assert np.array_equal(got, want)
    ix.close()
    whole.close()
