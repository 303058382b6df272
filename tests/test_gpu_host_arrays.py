"""Host arrays through pinned memory: queries read and results written in place, copied first, or (too large for a block)
unstaged; rows added in pieces; images fetched in pieces; values refused on the way."""
import threading

import numpy as np
import pytest

from helpers import bits_equal, unit_gaussian

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def T():
    from turbovec_amd import _lib
    _lib.lib()
    return _lib


def filled(T, dim, bits, n, seed=1):
    ix = T.NativeIndex(dim, bits)
    ix.add(unit_gaussian(n, dim, seed))
    return ix


# in place up to 1 MiB of queries (2048 x 128), copied to the device beyond, unstaged behind 32 MiB in all (70000 x 128)
@pytest.mark.parametrize("nq", [1, 2048, 2049, 70_000])
def test_every_way_of_the_queries(T, nq):
    torch = pytest.importorskip("torch")
    dim, n, k = 128, 5_003, 3
    ix = filled(T, dim, 4, n)
    q = unit_gaussian(nq, dim, seed=2)
    d = torch.from_numpy(q).cuda()
    s, i = torch.empty(nq, k, device="cuda"), torch.empty(nq, k, dtype=torch.int64, device="cuda")
    torch.cuda.synchronize()
    ix.search_dev(d.data_ptr(), nq, k, s.data_ptr(), i.data_ptr())
    words = T.pack_mask(np.random.default_rng(0).random(n) < 0.3)[0]
    for checked in (False, True):
        hs, hi = ix.search(q, k, checked=checked)
        assert bits_equal(hs, s.cpu().numpy()) and np.array_equal(hi, i.cpu().numpy())
        ms, mi = ix.search(q, k, mask_words=words, checked=checked)
        some = ix.search(q[-5:], k, mask_words=words)
        assert bits_equal(ms[-5:], some[0]) and np.array_equal(mi[-5:], some[1])
    q[nq // 2, 7] = np.nan
    with pytest.raises(T.TurbovecHipError) as e:
        ix.search(q, k, checked=True)
    assert e.value.status == T.ERR_INVALID_QUERY_VALUE and e.value.bad_index == nq // 2 * dim + 7
    ix.close()


def test_more_callers_than_blocks(T):
    """Twenty threads, each with its own queries: blocks are lent to some, the others do without."""
    dim, n = 64, 9_001
    ix = filled(T, dim, 4, n)
    qs = [unit_gaussian(1 + t, dim, seed=50 + t) for t in range(20)]
    want = [ix.search(q, 5) for q in qs]
    wrong = []

    def caller(t):
        for _ in range(30):
            s, i = ix.search(qs[t], 5, checked=t % 2 == 0)
            if not (bits_equal(s, want[t][0]) and np.array_equal(i, want[t][1])):
                wrong.append(t)
    threads = [threading.Thread(target=caller, args=(t,)) for t in range(len(qs))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    ix.close()


# rows of one piece, of several (4 MiB each), of more than one slice (256 MiB), the bad value in the last of them; rows in front
# that share a block with the refused ones, or none
@pytest.mark.parametrize("before,n,dim", [(0, 5, 8), (37, 700, 2048), (37, 34_000, 2048), (64, 34_000, 2048)])
def test_refused_rows_leave_the_index_as_it_was(T, before, n, dim):
    rows = np.tile(unit_gaussian(500, dim, seed=5), (n // 500 + 1, 1))[:n]
    first = unit_gaussian(max(before, 1), dim, seed=6)[:before]
    ix = T.NativeIndex(dim, 4)
    if before:
        ix.add(first)
    image = ix.to_bytes()
    bad = rows.copy()
    bad[n - 1, dim - 3] = np.inf
    with pytest.raises(T.TurbovecHipError) as e:
        ix.add(bad)
    assert e.value.status == T.ERR_INVALID_QUERY_VALUE and f"vector {n - 1} " in str(e.value)
    assert len(ix) == before and ix.to_bytes() == image
    ix.add(rows)
    ix.add(first)
    other = T.NativeIndex(dim, 4)
    for at in range(0, before, 7):
        other.add(first[at:at + 7])
    for at in range(0, n, 999):
        other.add(rows[at:at + 999])
    other.add(first) if before else None
    assert ix.to_bytes() == other.to_bytes()
    ix.close()
    other.close()
