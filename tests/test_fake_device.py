"""The library's host side on a HIP runtime without a device (fake_hip.c): device memory that runs out, waits that take
as long as the test says.  Each test runs in a process of its own, which loads that runtime in front of the library."""
import os
import subprocess
import sys

import pytest

from conftest import ROOT

HERE = os.path.dirname(os.path.abspath(__file__))
HEAD = '''
import ctypes as C, sys, threading, time
import numpy as np
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from turbovec_amd import _lib as T
def var(name, kind=C.c_int):
    return kind.in_dll(fake, "fake_" + name)
limit, used = var("limit", C.c_size_t), var("used", C.c_size_t)
fake.fake_lds.restype = C.c_size_t
def launched(part):
    return fake.fake_launched(part.encode())
def index(rows, dim=64):
    ix = T.NativeIndex(dim, 4)
    if rows:
        ix.append_rows(np.zeros((rows, dim // 2), np.uint8), np.zeros(rows, np.float32))
    return ix
'''


@pytest.fixture(scope="session")
def fake(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("fake") / "libfake_hip.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-pthread", "-o", out, os.path.join(HERE, "fake_hip.c")], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", HEAD + body, out, ROOT], capture_output=True, text=True, timeout=100)
        assert r.returncode == 0, r.stdout + r.stderr
    return run


def test_an_index_is_made_from_memory_the_library_holds(fake):
    """Blocks a grown index gave up are kept for later ones; memory that a new index needs is not refused for them."""
    fake('''
a = index(100_000)
a.append_rows(np.zeros((200_000, 32), np.uint8), np.zeros(200_000, np.float32))
before = used.value
limit.value = before                     # nothing is left but what the library keeps
b = index(0)
assert used.value < before
b.close(); a.close()
assert used.value == 0
''')


def test_a_wait_for_the_device_holds_up_no_other_index(fake):
    """An index that gives its blocks up waits for the device's work first; another one is made meanwhile."""
    fake('''
a = index(100_000)
b = index(0)
busy, waits = var("device_busy"), var("device_waits")
busy.value = 1
closing = threading.Thread(target=a.close)
closing.start()
while waits.value == 0:
    time.sleep(0.001)
made = []
making = threading.Thread(target=lambda: made.append(index(0)))
making.start()
making.join(10)
held_up = making.is_alive()
busy.value = 0
making.join(); closing.join()
assert not held_up
made[0].close(); b.close()
assert used.value == 0
''')


def test_no_pause_for_callers_that_cannot_be_merged(fake):
    """A caller that waited for another's search gives callers a moment to register, but not where the two could not
    have shared a launch (another k).  (The moment would be seen by the clock: it is read in a loop.)"""
    fake('''
ix = index(64)
clock, wait = var("clock_reads", C.c_long), var("stream_wait_us")
wait.value = 2000                        # the other caller is always there before a search ends
turns = 20
q = np.ones((1, 64), np.float32)
def caller(k):
    for _ in range(turns):
        ix.search(q, k)
before = clock.value
callers = [threading.Thread(target=caller, args=(k,)) for k in (1, 2)]
for t in callers: t.start()
for t in callers: t.join()
per_search = (clock.value - before) / (2 * turns)
assert per_search <= 2, per_search
''')


@pytest.mark.parametrize("cus", [256, 64])
def test_the_encoder_fills_the_device_it_runs_on(fake, cus):
    """Rows beyond what is resident at once are turns of the same workgroups: three of these to a CU (128 dimensions, LDS)."""
    fake(f'''
var("cus").value = {cus}
ix = index(0, 128)
ix.add(np.ones((100_000, 128), np.float32))
assert var("largest_grid").value == 3 * {cus}, var("largest_grid").value
''')


# 32 MiB in all is the most that is staged in pinned memory: beyond it the snapshot is the call's own
@pytest.mark.parametrize("rows", [1000, 140_000])
def test_the_values_that_were_checked_are_the_ones_searched(fake, rows):
    """A caller's array changes while its call waits for another search to end: what then goes to the device is what was checked."""
    fake(f'''
ix = index(64)
fake_marker = var("marker", C.c_uint32)
fake_marker.value = 0x7fc0dead           # a NaN
other = threading.Thread(target=lambda: ix.search(np.ones((1, 64), np.float32), 2))
var("stream_wait_us").value = 1_000_000
other.start()
time.sleep(0.2)                          # it holds the index
q = np.ones(({rows}, 64), np.float32)
said = []
def caller():
    try:
        ix.search(q, 1, checked=True)
        said.append("searched")
    except T.TurbovecHipError as e:
        said.append(e.status)
waiting = threading.Thread(target=caller)
waiting.start()
time.sleep(0.4)                          # checked, and waiting for the index
assert other.is_alive() and waiting.is_alive()
q.view(np.uint32)[{rows} // 2, 5] = 0x7fc0dead
other.join()
var("stream_wait_us").value = 0
waiting.join()
assert said == ["searched"], said
assert var("marker_copies").value == 0
''')


def test_small_indexes_are_searched_without_sampling(fake):
    """Batches of a few queries on the shortest rows, one query and many on short rows of u8 tables; few blocks of long ones are not."""
    fake('''
for dim, bits, rows, nq, k, unsampled in ((64, 4, 60_000, 2, 10, True), (8, 4, 1_000_000, 8, 100, True), (128, 2, 100_000, 1, 10, True), (1536, 2, 20_000, 1, 10, True),
                                          (64, 2, 131_073, 40, 10, True), (32, 3, 131_072, 400, 10, True), (512, 2, 1000, 1, 10, True), (3072, 2, 1000, 1, 10, False),
                                          (1024, 3, 2048, 1, 10, False), (1024, 3, 2049, 1, 10, True)):
    ix = T.NativeIndex(dim, bits)
    ix.append_rows(np.zeros((rows, ix.n_byte_groups), np.uint8), np.zeros(rows, np.float32))
    assert (len(ix.sampling_plan(nq, k)[0]) == 0) == unsampled, (dim, bits, rows, nq, k)
    ix.close()
''')


def test_segments_are_read_by_four_threads_where_they_are_long(fake):
    """One query's first level, where it fills its segments, and its other levels from eight candidates a segment on average on: not
    with fewer, nor for two queries, nor for blocks' best rows, dealt out evenly, up to sixteen a segment."""
    fake('''
parted = var("parted")
# the levels' strides, and the launches of them: 64 dimensions, 18 and 1 from best rows of blocks, 625, 73, 8 and 1 with more segments than
# 256 behind the first; 1536 dimensions 2-bit, 256 segments at the most: 31, 5 (2480 candidates, and its conditional repeat) and 1 (2000)
for dim, bits, rows, nq, k, launches in ((64, 4, 300_000, 1, 64, 0), (64, 4, 2_000_000, 1, 400, 1), (64, 4, 2_000_000, 2, 400, 0),
                                         (1536, 2, 100_000, 1, 10, 0), (1536, 2, 1_200_000, 1, 128, 0), (1536, 2, 100_000, 1, 100, 1), (1536, 2, 100_000, 1, 400, 3)):
    ix = T.NativeIndex(dim, bits)
    ix.append_rows(np.zeros((rows, ix.n_byte_groups), np.uint8), np.zeros(rows, np.float32))
    ix.set_path(16)
    before = parted.value
    ix.search(np.ones((nq, dim), np.float32), k)
    assert parted.value - before == launches, (dim, nq, k, ix.sampling_plan(nq, k), parted.value - before)
    ix.close()
''')


FILTERED = '''
def filtered(ix, path, nq=4):
    """A sampled search (16) of half the rows; path 64 gathers them, 32 reads the mask."""
    words = T.pack_mask(np.arange(len(ix)) % 2 == 1)[0]
    ix.set_path(path | 16)
    before = ix.gathered_searches()[0]
    ix.search(np.ones((nq, 64), np.float32), 3, mask_words=words)
    return ix.gathered_searches()[0] - before
'''


def test_rows_kept_of_a_filtered_search_give_way(fake):
    """Rows that fitted beside an index are not refused for the copy its filtered search left behind."""
    fake(FILTERED + '''
a, b = index(400_000), index(0)
assert filtered(a, 32) == 0
plain, before = a.workspace_bytes()[0], used.value
assert filtered(a, 64) == 1
kept = used.value - before
assert kept >= 6_400_000                 # 200000 rows of 32 bytes
# b wants 31 MB: 8 are free, the pool holds the 17 of a's first workspace, and the copy its 10
limit.value = used.value + 8_000_000
b.append_rows(np.zeros((400_000, 32), np.uint8), np.zeros(400_000, np.float32))
limit.value = used.value
assert filtered(a, 64) == 0 and filtered(a, 32) == 0           # the mask is read, as there is no memory for a copy
assert a.workspace_bytes()[0] < plain + kept
limit.value = 1 << 34
assert filtered(a, 64) == 1 and a.workspace_bytes()[0] == plain + kept
a.close(); b.close()
assert used.value == 0
''')


def test_rows_that_have_room_wait_for_their_own_work_only(fake):
    """Rows for which there is room: one wait for their codes, one for their scales, none for an index that did not grow."""
    fake('''
ix, waits = index(64), var("stream_waits")
before = waits.value
ix.append_rows(np.zeros((1, 32), np.uint8), np.zeros(1, np.float32))
assert waits.value - before == 2, waits.value - before
before = waits.value
ix.add(np.ones((1, 64), np.float32))
assert waits.value - before == 2, waits.value - before      # the row's way to the device, and the encoder
ix.close()
''')


def test_an_add_that_fails_shows_none_of_its_rows(fake):
    """The encoder has run and the outgrown memory cannot be given back: the call says so, and its rows are not the index's."""
    fake('''
ix = index(64)
v = np.ones((10_000, 64), np.float32)
var("frees_refused").value = 1
try:
    ix.add_dev(v.ctypes.data, len(v))
    said = None
except T.TurbovecHipError as e:
    said = e.status
assert said == T.ERR_HIP and len(ix) == 64, (said, len(ix))
ix.add_dev(v.ctypes.data, len(v))
assert len(ix) == 10_064
ix.close()
assert used.value == 0
''')


def test_room_to_grow_is_not_taken_from_others(fake):
    """Rows that fit as they are: the library gives nothing up, neither pooled blocks nor a filtered search's copy, for the room beyond them."""
    fake(FILTERED + '''
a, b, c = index(400_000), index(100_000), index(50_000)
assert filtered(a, 64) == 1
c.close()                                # 1.6 MB of codes are in the pool
held, before = a.workspace_bytes()[0], used.value
# needed: 3.96 MB; by half: 5.4; twice: 7.2
limit.value = before + 4_200_000
b.append_rows(np.zeros((10_000, 32), np.uint8), np.zeros(10_000, np.float32))
assert len(b) == 110_000 and a.workspace_bytes()[0] == held
assert used.value > before + 3_000_000   # (100000 rows' codes went to the pool, their scales back to the device)
a.close(); b.close()
assert used.value == 0
''')


def test_indexes_that_grow_ahead_hold_no_more_than_a_bound(fake):
    """Many indexes that have grown once: what they hold beyond growing by half is 256 MiB in all, and is there again once they are gone."""
    fake('''
n, row = 1_000_000, 36                   # dim 64: 32 bytes and a scale; a multiple of a block's rows
def grown():
    ix = index(n)
    before = used.value
    ix.append_rows(np.zeros((1, 32), np.uint8), np.zeros(1, np.float32))
    return ix, (used.value - before) / (n * row)      # (the old blocks are in the pool)
made = [grown() for _ in range(20)]
growth = [g for _, g in made]
assert abs(growth[0] - 2.0) < 0.01 and abs(growth[-1] - 1.5) < 0.01, growth
ahead = sum(growth) - 1.5 * len(growth)
assert ahead * n * row <= 256 << 20, growth
for ix, _ in made: ix.close()
assert used.value == 0
ix, g = grown()
assert abs(g - 2.0) < 0.01
ix.close()
''')


def test_a_copy_of_rows_gives_way_to_the_search_it_is_made_for(fake):
    """Memory for the copy or for the workspace, not for both: the mask is read, as where there is none for the copy."""
    fake(FILTERED + '''
a = index(400_000)
filtered(a, 32)
grown, before = a.workspace_bytes()[0] - 16_777_216, used.value
filtered(a, 64)
kept = used.value - before
a.close()
b = index(400_000)
assert b.workspace_bytes()[0] == 16_777_216 and 2_000_000 < grown < kept
limit.value = used.value + kept + 1_000_000
filtered(b, 64)
assert used.value <= limit.value
b.close()
assert used.value == 0
''')


def test_pinned_memory_is_shared_by_the_devices_indexes(fake):
    """A new index's first calls on host arrays find what another one's calls had allocated; it all goes with the last index."""
    fake('''
blocks, pinned = var("pinned_blocks"), var("pinned", C.c_size_t)
a = index(64)
for nq in (1, 1000):
    a.search(np.ones((nq, 64), np.float32), 3)
before = blocks.value
assert before == 2
b = index(64)
a.close()
for nq in (1000, 1):
    b.search(np.ones((nq, 64), np.float32), 3)
assert blocks.value == before
b.close()
assert pinned.value == 0
''')


def test_pinned_memory_has_a_limit(fake):
    """256 MiB on a device, whatever its indexes' calls want at once; what is idle makes room, and a call that gets none does without."""
    fake('''
pinned, peak = var("pinned", C.c_size_t), var("pinned_peak", C.c_size_t)
made = [index(64) for _ in range(9)]
rows = 1
while rows <= 32768:                     # blocks of 64 KiB to 16 MiB, idle
    made[0].search(np.ones((rows, 64), np.float32), 1)
    rows *= 2
idle = pinned.value
assert idle >= 16 << 20
q = np.ones((100_000, 64), np.float32)   # 32 MiB each
var("stream_wait_us").value = 100_000
started = threading.Barrier(len(made))
def call(ix):
    started.wait()
    ix.search(q, 1, checked=True)
calls = [threading.Thread(target=call, args=(ix,)) for ix in made]
for t in calls: t.start()
for t in calls: t.join()
var("stream_wait_us").value = 0
assert 128 << 20 < peak.value <= 256 << 20, peak.value
for ix in made: ix.close()
assert pinned.value == 0 and used.value == 0
''')


@pytest.mark.parametrize("bad", [True, False])
def test_rows_count_once_all_of_them_have_passed(fake, bad):
    """An add of several slices shows none of its rows before the last one is there, and none at all if it refuses one."""
    fake(f'''
ix = index(64)
v = np.ones((1_050_000, 64), np.float32)           # a slice is 256 MiB: 1048576 rows
if {bad}: v[-1, 3] = np.nan
var("stream_wait_us").value = 1000
said = []
def add():
    try:
        ix.add(v)
        said.append("added")
    except T.TurbovecHipError as e:
        said.append(e.status)
adding = threading.Thread(target=add)
adding.start()
seen = set()
while adding.is_alive():
    seen.add(len(ix))
    time.sleep(1e-4)
var("stream_wait_us").value = 0
assert said == ([T.ERR_INVALID_QUERY_VALUE] if {bad} else ["added"]), said
end = 64 if {bad} else 64 + len(v)
assert 64 in seen and seen <= {{64, end}}, seen
assert len(ix) == end
ix.close()
''')


def test_a_mask_of_another_length_is_refused_unread(fake):
    """The words a call says there are beyond the index's rows are not looked at."""
    fake('''
import mmap
ix = index(64)
page = mmap.mmap(-1, 2 * mmap.PAGESIZE)
at = C.addressof(C.c_char.from_buffer(page))
assert C.CDLL(None).mprotect(C.c_void_p(at + mmap.PAGESIZE), C.c_size_t(mmap.PAGESIZE), 0) == 0
q, s, i = np.ones((2, 64), np.float32), np.zeros(2, np.float32), np.zeros(2, np.int64)
mask = at + mmap.PAGESIZE - 8            # one word before memory nobody may read
ke, bad = C.c_size_t(0), C.c_size_t(0)
for words in (2, 300_000, 1 << 62):
    assert T.lib().tv_search(ix.h, T.ptr(q), 2, 1, mask, words, T.ptr(s), T.ptr(i), C.byref(ke)) == T.ERR_MASK_LENGTH_MISMATCH
    assert T.lib().tv_search_checked(ix.h, T.ptr(q), 2, 1, mask, words, T.ptr(s), T.ptr(i), C.byref(ke), C.byref(bad)) == T.ERR_MASK_LENGTH_MISMATCH
''')


def test_a_mask_that_changed_is_another_mask(fake):
    """A call waits with what its mask array held; one made after the array changed is searched with what it holds then."""
    fake('''
ix = index(64 * 64)
words = np.full(64, 1, np.uint64)
q, bad = np.ones((2, 64), np.float32), []
def search(mask):
    ke, s, i = C.c_size_t(0), np.zeros(2, np.float32), np.zeros(2, np.int64)
    bad.append(T.lib().tv_search(ix.h, T.ptr(q), 2, 1, mask, 64, T.ptr(s), T.ptr(i), C.byref(ke)))
calls = [threading.Thread(target=search, args=(m,)) for m in (None, T.ptr(words), T.ptr(words))]
var("stream_wait_us").value = 300_000
calls[0].start()
time.sleep(0.1)                          # it holds the index
calls[1].start()
time.sleep(0.1)                          # waits
marker = var("marker", C.c_uint32)
marker.value = 0x7fc0dead
words.view(np.uint32)[7] = marker.value
calls[2].start()
for t in calls: t.join()
assert bad == [T.OK] * 3, bad
assert ix.merged_calls() == 0 and var("marker_copies").value == 1
''')


def test_masks_of_host_arrays_are_counted_on_the_host(fake):
    """Whether a mask's rows lie scattered is counted on the device, and waited for, only where the mask lies there."""
    fake('''
ix, n, counts = index(100_000, 1536), 100_000, var("counts")
q, s, i = np.ones((1024, 1536), np.float32), np.zeros((1024, 10), np.float32), np.zeros((1024, 10), np.int64)
for rows, gathers in ((np.arange(n) // 2 % 10 == 0, True), ((np.arange(n) > 30_000) & (np.arange(n) < 50_000), False)):
    words, allowed = T.pack_mask(rows)
    before = ix.gathered_searches()[0]
    ix.search(q, 10, mask_words=words)
    assert ix.gathered_searches()[0] == before + gathers and counts.value == 0
    ix.search_dev(q.ctypes.data, 1024, 10, s.ctypes.data, i.ctypes.data, words.ctypes.data, allowed)
    assert ix.gathered_searches()[0] == before + 2 * gathers and counts.value == 1
    counts.value = 0
''')


# (a 2-bit batch takes the matrix-unit scan over so few blocks from 385 queries on, a 3-bit one from 49)
@pytest.mark.parametrize("bits,nq", [(2, 400), (3, 65)])
def test_the_two_step_scan_of_a_few_rows(fake, bits, nq):
    """Asked for by the test hook over fewer blocks than a sample takes one of: the other scans."""
    fake(f'''
for rows in (1, 31, 96, 97, 128, 129):
    ix = T.NativeIndex(64, {bits})
    ix.append_rows(np.zeros((rows, ix.n_byte_groups), np.uint8), np.zeros(rows, np.float32))
    ix.set_path(128)
    ix.sampling_plan({nq}, 3)
    ix.search(np.ones(({nq}, 64), np.float32), 3)
    assert ix.last_scan_ms()[1] == 1
    ix.close()
ix = T.NativeIndex(64, {bits})           # a filter's few rows, gathered
ix.append_rows(np.zeros((40_000, ix.n_byte_groups), np.uint8), np.zeros(40_000, np.float32))
ix.set_path(128 + 64)
ix.search(np.ones(({nq}, 64), np.float32), 3, mask_words=T.pack_mask(np.arange(40_000) % 1000 == 7)[0])
assert ix.gathered_searches()[0] == 1
ix.close()
''')


@pytest.mark.parametrize("dim,bits,nq", [(1536, 2, 372), (1024, 2, 416), (640, 2, 424)])
def test_fixed_scratch_is_not_charged_for_the_two_step_scan(fake, dim, bits, nq):
    """Batches on lent scratch, which never go in two steps: the largest that fit on the matrix-unit scan are all served in one launch."""
    fake(f'''
ix = T.NativeIndex({dim}, {bits})
ix.append_rows(np.zeros((20_000, ix.n_byte_groups), np.uint8), np.zeros(20_000, np.float32))
def served(nq):
    q, s, i = np.ones((nq, {dim}), np.float32), np.zeros((nq, 10), np.float32), np.zeros((nq, 10), np.int64)
    ix.search_dev_noalloc(q.ctypes.data, nq, 10, s.ctypes.data, i.ctypes.data)
    return ix.queries_per_launch()
assert served({nq}) == {nq}
try:
    served({nq + 1})
    raise SystemExit("one more was searched")
except T.TurbovecHipError as e:
    assert e.status == T.ERR_BAD_ARGUMENT
ix.set_path(128)                         # the hook does not change what fits
assert served({nq}) == {nq}
ix.close()
''')


STAGES = '''
def batch_index(rows):
    """An index whose batches of 1024 queries go in two steps, with a stage of about 20 KB for every 256 rows."""
    ix = T.NativeIndex(8, 2)
    ix.append_rows(np.zeros((rows, 2), np.uint8), np.zeros(rows, np.float32))
    return ix
queries = np.ones((1024, 8), np.float32)
def together(indexes):
    """All at once; whether each went in two steps."""
    var("stream_wait_us").value = 500_000
    calls = [threading.Thread(target=ix.search, args=(queries, 10)) for ix in indexes]
    for t in calls: t.start()
    for t in calls: t.join()
    var("stream_wait_us").value = 0
    return [ix.last_scan_ms()[1] > 1 for ix in indexes]
def rooms(indexes):
    """What the searches' stages hold, of an amount of memory that was read before any search."""
    return used.value - start - sum(ix.workspace_bytes()[0] for ix in indexes)
'''


def test_room_for_stages_that_nobody_uses_makes_way(fake):
    """Three searches at once, which leave almost all that stages may hold; a later one that wants more than any of the three had."""
    fake(STAGES + '''
small, large = [batch_index(6_600_000) for _ in range(3)], batch_index(20_000_000)
start = used.value
assert together(small) == [True] * 3
held = rooms(small)
assert 1.8 * 2**30 < held < 2**31, held
assert together([large]) == [True]
assert held / 3 * 1.5 < rooms(small + [large]) <= 2**31, rooms(small + [large])
assert together(small[:1]) == [True]
for ix in small + [large]: ix.close()
assert used.value == 0
''')


def test_room_for_stages_has_a_limit(fake):
    """Searches that start together count what the others are still allocating: 2 GiB for all, and the rest go without.  A block
    that the library holds already, larger than asked for, counts whole."""
    fake(STAGES + '''
made = [batch_index(20_000_000) for _ in range(4)]
start = used.value
var("large_alloc_us").value = 200_000
took = together(made)
var("large_alloc_us").value = 0
assert sum(took) == 2 and rooms(made) <= 2**31, (took, rooms(made))
for ix in made: ix.close()
assert used.value == 0
made = [batch_index(20_000_000) for _ in range(2)]
start = used.value
gone = batch_index(37_000_000)           # 1.10 GiB of codes, which go to the pool when their index does
gone.close()
took = together(made)
assert sum(took) == 1 and rooms(made) < 1.5 * 2**30, (took, rooms(made))      # (with what else is in the pool)
for ix in made: ix.close()
assert used.value == 0
''')


def test_an_index_is_made_when_its_tables_are_there(fake):
    """The call that makes an index waits for its tables, and an error on their way is that call's."""
    fake('''
waits, refused = var("stream_waits"), var("stream_waits_refused")
before = waits.value
a = index(0)
assert waits.value > before
refused.value = 1
try:
    index(0)
    said = None
except T.TurbovecHipError as e:
    said = e.status
assert said == T.ERR_HIP, said
a.close()
assert used.value == 0
''')


def test_the_line_between_unsampled_and_sampled_of_short_rows(fake):
    """Short 4-bit rows and many queries: unsampled as far as decoding a block once more for every further four tiles, and scoring the
    results' blocks again, cost less than a sample's floors and the empty places of the other kernel's last round."""
    fake('''
for dim, rows, nq, k, unsampled in ((256, 350_000, 1024, 10, True), (256, 650_000, 160, 10, True), (256, 418_176, 1000, 10, True), (256, 418_177, 1000, 10, False),
                                    (192, 469_376, 1024, 10, True), (192, 469_377, 1024, 10, False), (192, 524_289, 1024, 10, True), (640, 667_872, 150, 10, True),
                                    (640, 667_873, 150, 10, False), (384, 700_000, 1000, 10, False), (640, 850_000, 300, 10, False), (512, 850_000, 512, 10, False),
                                    (136, 729_140, 397, 59, False), (368, 388_650, 928, 75, False), (168, 318_674, 387, 100, True), (256, 350_000, 1024, 100, False),
                                    (640, 4_096, 1024, 100, True), (640, 4_200, 1024, 60, True), (128, 1_000_000, 1024, 100, True), (640, 1_000_000, 128, 60, True)):
    ix = index(0, dim)
    ix.append_rows(np.zeros((rows, dim // 2), np.uint8), np.zeros(rows, np.float32))
    assert (len(ix.sampling_plan(nq, k)[0]) == 0) == unsampled, (dim, rows, nq, k)
    ix.close()
''')


def test_rows_scored_again_whole_have_no_room_for_parts(fake):
    """The second scoring of a search without sampling: only where a block's chunks go to several waves is there LDS for their sums."""
    fake('''
for dim, bits, rows, nq, k, chunks, table in ((1536, 2, 3_000, 800, 14, 12, 1024), (64, 4, 10_000, 900, 82, 1, 64), (320, 3, 5_000, 700, 96, 5, 1024)):
    ix = T.NativeIndex(dim, bits)
    ix.append_rows(np.zeros((rows, ix.n_byte_groups), np.uint8), np.zeros(rows, np.float32))
    ix.search(np.ones((nq, dim), np.float32), k)
    assert fake.fake_lds(b"k_pickI") == k * 256 + chunks * table, (dim, fake.fake_lds(b"k_pickI"))
    ix.close()
''')


def test_parts_of_blocks_are_as_many_as_save_time(fake):
    """The second scoring in parts: where few results leave waves idle, not in so many turns of short parts that they cost more, and not where
    several queries share a CU."""
    fake('''
def scored(dim, bits, rows, nq, k):
    ix = T.NativeIndex(dim, bits)
    ix.append_rows(np.zeros((rows, ix.n_byte_groups), np.uint8), np.zeros(rows, np.float32))
    # (blocks a thread keeps: 16; tables; several workgroups a query; parts)
    before = [launched(f"k_pickILj1024ELj16ELb{lut}ELb{shared}ELb1EE") for lut in (0, 1) for shared in (0, 1)]
    ix.search(np.ones((nq, dim), np.float32), k)
    after = [launched(f"k_pickILj1024ELj16ELb{lut}ELb{shared}ELb1EE") for lut in (0, 1) for shared in (0, 1)]
    ix.close()
    return sum(after) - sum(before)
for shape in ((3072, 4, 40_001, 1, 1), (3072, 4, 40_001, 1, 12), (1000, 3, 20_015, 3, 4), (1416, 2, 20_001, 1, 3), (776, 4, 9_001, 100, 2)):
    assert scored(*shape) == 1, shape
for shape in ((1152, 4, 9_638, 168, 23), (720, 4, 153_761, 200, 34), (1536, 3, 4_000, 300, 1), (768, 4, 6_722, 257, 1), (64, 2, 30_031, 1, 1), (768, 4, 50_000, 8, 16)):
    assert scored(*shape) == 0, shape
''')


def test_filtered_batches_of_tables_gather_where_that_is_less(fake):
    """Half of the rows at random: whether the two-step scan could take the index with its mask goes by the rows allowed, and what it
    takes counts its stages' launches."""
    fake('''
for dim, bits, rows, nq, k in ((384, 3, 225_592, 929, 40), (2048, 2, 398_963, 780, 26), (512, 3, 352_922, 810, 54), (256, 3, 400_795, 916, 80), (320, 2, 322_259, 705, 2)):
    ix = T.NativeIndex(dim, bits)
    ix.append_rows(np.zeros((rows, ix.n_byte_groups), np.uint8), np.zeros(rows, np.float32))
    words = T.pack_mask(np.random.default_rng(7).random(rows) < 0.5)[0]
    ix.search(np.ones((nq, dim), np.float32), k, mask_words=words)
    assert ix.gathered_searches()[0] == 1, (dim, bits)
    ix.close()
''')


CHOSEN = '''
def launches(part, dim, bits, n, nq, k=10, allowed=1.0):
    """Launches of kernels with `part` in their name in one search."""
    ix = T.NativeIndex(dim, bits)
    ix.append_rows(np.zeros((n, ix.n_byte_groups), np.uint8), np.zeros(n, np.float32))
    before = launched(part)
    ix.search(np.ones((nq, dim), np.float32), k, mask_words=T.pack_mask(np.random.default_rng(n).random(n) < allowed)[0] if allowed < 1 else None)
    ix.close()
    return launched(part) - before
'''


def test_where_the_two_step_scan_starts(fake):
    """Batches of tables, on both sides of the least blocks and queries; under a filter too."""
    fake(CHOSEN + '''
for dim, bits, n, nq, k, takes in ((768, 2, 342_848, 200, 10, False), (768, 2, 342_849, 200, 10, True), (64, 2, 3_400_001, 64, 3, False), (64, 2, 3_400_001, 65, 3, True),
                                   (256, 3, 738_432, 400, 10, False), (256, 3, 738_433, 400, 10, True)):
    assert (launches("k_near_rescore", dim, bits, n, nq, k) > 0) == takes, (dim, bits, n, nq)
for dim, bits, n, nq, k in ((64, 2, 3_400_001, 65, 3), (768, 2, 1_000_001, 200, 10), (256, 3, 800_001, 400, 10)):
    assert launches("k_near_rescore", dim, bits, n, nq, k, 0.95) > 0, (dim, bits, n, nq)
''')


def test_blocks_in_parts_are_scanned_so(fake):
    """Few blocks: the scans whose waves take parts of one -- and not where blocks are many or rows of one chunk."""
    fake(CHOSEN + '''
for dim, n, nq, parts in ((512, 1, 1, 1), (512, 33, 33, 1), (584, 8_200, 64, 1), (1536, 4_097, 40, 1), (1536, 20_000, 40, 0), (1536, 65_537, 1, 0), (2056, 9_001, 1, 1),
                          (2056, 9_001, 100, 0), (3072, 30_000, 8, 1), (128, 3_000, 1, 0)):
    assert launches("k_scan_p4_partsI", dim, 4, n, nq) == parts, (dim, n, nq)
for dim, bits, n, nq, parts in ((200, 3, 64, 5, 1), (384, 2, 60_001, 8, 1), (1000, 3, 12_345, 8, 1), (1400, 2, 50_001, 2, 1), (1400, 2, 50_001, 6, 0), (3072, 3, 16_411, 3, 1),
                                (3072, 2, 24_033, 4, 1), (384, 3, 16_001, 16, 1), (384, 3, 16_001, 47, 0), (1536, 2, 5_001, 18, 1), (2432, 3, 4_700, 16, 1), (128, 2, 3_333, 2, 0)):
    assert launches("k_scan_lut_partsI", dim, bits, n, nq) == parts, (dim, bits, n, nq)
''')


def test_three_tiles_to_a_workgroup(fake):
    """As many tiles of queries as make no more workgroups so than with four each."""
    fake(CHOSEN + '''
for dim, n, nq, three in ((64, 66_001, 65, 1), (128, 40_011, 161, 1), (192, 25_000, 288, 1), (256, 70_003, 150, 1), (448, 66_017, 192, 1), (768, 66_001, 96, 1),
                          (256, 70_003, 64, 0), (256, 70_003, 128, 0), (256, 70_003, 256, 0), (1536, 70_003, 96, 0), (256, 2_000, 96, 0)):
    assert launches("k_scan_p4_bestILi3E", dim, 4, n, nq) == three, (dim, n, nq)
''')


def test_values_are_refused_wherever_they_are(fake):
    """Searches of host arrays look at every value of what they copy: first and last, next to the ends of the runs that are looked
    at together; the largest that is accepted is."""
    fake('''
ix = index(1000, 8)
largest = np.nextafter(np.float32(1e16), np.float32(0))
for nq in (1, 3, 512, 513, 2049):
    q = np.full((nq, 8), 0.5, np.float32)
    q[::2] *= -1
    places = sorted({p for p in (0, 1, 7, 4095, 4096, 4097, nq * 8 // 2, nq * 8 - 9, nq * 8 - 1) if 0 <= p < nq * 8})
    for p in places:
        for value in (np.nan, -np.nan, np.inf, -np.inf, 1e16, -1e16, np.float32(3e38), largest, -largest, np.float32(1e-45), -0.0):
            held = q.flat[p]
            q.flat[p] = value
            try:
                ix.search(q, 3, checked=True)
                refused = False
            except T.TurbovecHipError as e:
                assert e.status == T.ERR_INVALID_QUERY_VALUE
                refused = True
            assert refused == (not abs(np.float32(value)) < np.float32(1e16)), (nq, p, value)
            q.flat[p] = held
ix.close()
''')


def test_selections_that_check_guessed_floors(fake):
    """Only the two-step table scan's selections are the instances that know of guessed floors."""
    fake(CHOSEN + '''
def guessed(*shape):
    # (threads, threads a segment, guessed floors)
    return sum(launches(f"k_finalILj{t}ELj1ELb1EE", *shape) for t in (256, 512, 1024)) > 0
assert guessed(64, 2, 3_400_001, 65, 3)
for shape in ((64, 2, 3_400_001, 64, 3), (128, 4, 1_472_940, 7, 66), (64, 4, 1_200_000, 1024, 10), (768, 4, 200_000, 2, 200)):
    assert launches("k_finalI", *shape) > 0 and not guessed(*shape), shape
''')
