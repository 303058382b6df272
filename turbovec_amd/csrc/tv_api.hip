// C ABI of the search path (see include/turbovec_hip.h).
#include "../../include/turbovec_hip.h"

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <cstdlib>
#include <exception>
#include <memory>
#include <new>
#include <string>
#include <thread>
#include <utility>
#include <vector>

#include "tv_internal.h"
#include "tv_snapshot.h"

namespace {

thread_local std::string g_last_error;

int fail_hip(hipError_t e, const char *what) {
    char buf[256];
    snprintf(buf, sizeof buf, "%s: %s", what, hipGetErrorString(e));
    g_last_error = buf;
    return TV_ERR_HIP;
}

#define TV_HIP(call)                                        \
    do {                                                    \
        hipError_t e__ = (call);                            \
        if (e__ != hipSuccess) return fail_hip(e__, #call); \
    } while (0)

size_t round_up(size_t v, size_t m) { return (v + m - 1) / m * m; }

// Bump allocator over the index's cached workspace.
struct Arena {
    uint8_t *base = nullptr;
    size_t used = 0;
    template <typename T>
    T *take(size_t count) {
        T *p = reinterpret_cast<T *>(base + used);
        used += round_up(count * sizeof(T), 256);
        return p;
    }
};

// ---- the scratch buffer of tv_search_dev_noalloc ---------------------------------------------
// One array per GPU, in the library's device image: every device the library runs on holds
// kScratchBytes of it from the moment the image is loaded there until the process ends.  In host
// code the array's name is only a handle for hipGetSymbolAddress; each device's copy has an
// address of its own, looked up once per device and kept in g_scratch.
constexpr size_t kScratchBytes = size_t(64) << 20;
static __device__ __align__(256) uint8_t scratch[kScratchBytes];

constexpr int kMaxDevices = 64;
struct DeviceScratch {
    void *ptr = nullptr;     // device address of `scratch` on this device
    std::mutex in_use;       // calls on one device share the array: one at a time within the process
};
DeviceScratch g_scratch[kMaxDevices];
std::mutex g_scratch_setup;

// Device `device` must be current.
int scratch_address(int device, void **out) {
    if (device < 0 || device >= kMaxDevices) { g_last_error = "device ordinal beyond the scratch table"; return TV_ERR_NO_DEVICE; }
    std::lock_guard<std::mutex> lock(g_scratch_setup);
    if (!g_scratch[device].ptr) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return fail_hip(e, "hipGetSymbolAddress(scratch)");
        g_scratch[device].ptr = p;
    }
    *out = g_scratch[device].ptr;
    return TV_OK;
}

// f(lo, hi) over [0, n) in parts of at least min_part on up to eight threads, the calling one among them.
// (What cannot start a thread runs on this one.)
constexpr size_t kMaxParts = 8;
template <typename F>
void in_parts(size_t n, size_t min_part, const F &f) {
    const size_t parts = std::min<size_t>({kMaxParts, std::max<size_t>(1, std::thread::hardware_concurrency()), std::max<size_t>(1, n / min_part)});
    const size_t per = (n + parts - 1) / parts;
    std::thread started[kMaxParts];
    for (size_t i = 1; i < parts; ++i) {
        const size_t lo = std::min(i * per, n), hi = std::min(lo + per, n);
        try {
            started[i] = std::thread([&f, lo, hi] { f(lo, hi); });
        } catch (const std::exception &) {     // no thread, or no memory for one
            f(lo, hi);
        }
    }
    f(0, std::min(per, n));
    for (std::thread &t : started) if (t.joinable()) t.join();
}
// Faults in fresh host memory about to be overwritten, several threads at once: a copy into 77 MB that
// nothing has touched yet takes 18 ms, into touched memory 4.4.
void touch_pages(uint8_t *p, size_t n) {
    in_parts(n, size_t(4) << 20, [p](size_t lo, size_t hi) {
        for (size_t i = lo; i < hi; i += 4096) *static_cast<volatile uint8_t *>(p + i) = 0;
    });
}
constexpr uint32_t kTooLargeBits = 0x5a0e1bcau;      // 1e16f

// ---- device memory of indexes ----------------------------------------------------------------
// Large blocks that an index gives up (it grew, or went) are kept for the next one, per device: up to
// kPoolBytes, handed on only to requests they exceed by a quarter at most, and given back when the last
// index of the device goes or an allocation fails -- any of an index's, so all of them come through
// device_alloc.  What filtered searches keep of their allowed rows (tv_spare) goes the same way when the pool was not
// enough.  An index built by four equal adds allocates 1.75 times its size on the way (by half each time, 2.6 times);
// fresh memory costs 28 us per MB once the driver has to clear what was freed before (400K x
// 1536 rows in four adds that grew by half: 4 ms a build while cleared memory lasts, 22.8 ms after).
constexpr size_t kPoolBytes = size_t(2) << 30, kPoolMinBytes = size_t(1) << 20;
// What the indexes of a device may hold beyond growing by half (ensure_capacity): nothing takes it back but their end, so it is
// a thousandth of the device's memory and not a share of its indexes.
constexpr size_t kAheadBytes = size_t(256) << 20;
struct DevicePool {
    std::mutex mu;         // held for the bookkeeping only: allocations, frees and waits are long
    std::mutex giving;     // held while an allocation that failed empties the pool and tries again
    std::vector<std::pair<size_t, void *>> blocks;
    size_t held = 0, indexes = 0;
    size_t ahead = 0;                // at most kAheadBytes, the sum of the indexes'
    tv_index *newest = nullptr;      // of the device's indexes
    static constexpr int kPinned = 64;
    tv_pinned pinned[kPinned];       // host memory: pinned_take
    static constexpr int kStaged = 4;
    tv_spare staged[kStaged];        // staged_take
    bool takes(size_t bytes) const { return bytes >= kPoolMinBytes && held + bytes <= kPoolBytes && indexes != 0; }   // mu held
    std::vector<std::pair<size_t, void *>> empty() {      // mu held
        held = 0;
        return std::exchange(blocks, {});
    }
};
DevicePool g_pool[kMaxDevices];

void free_blocks(const std::vector<std::pair<size_t, void *>> &blocks) {
    for (auto &b : blocks) (void)hipFree(b.second);
}

// A block some index of the device keeps for its filtered searches and is not using, or one of the table scans' stages, or null.  pool.mu held.
void *take_spare(DevicePool &pool) {
    for (tv_index *ix = pool.newest; ix != nullptr; ix = ix->older)
        for (tv_spare *s : {&ix->gathered, &ix->slots})
            if (!s->in_use && s->p != nullptr) { s->bytes = 0; return std::exchange(s->p, nullptr); }
    for (tv_spare &s : pool.staged)
        if (!s.in_use && s.p != nullptr) { s.bytes = 0; return std::exchange(s.p, nullptr); }
    return nullptr;
}

// The smallest block of the pool that holds so much, a quarter more or `most` at most, or null.  pool.mu held.
void *take_pooled(DevicePool &pool, size_t bytes, size_t *got, size_t most = ~size_t(0)) {
    most = std::min(most, bytes + bytes / 4);
    size_t best = pool.blocks.size();
    for (size_t i = 0; i < pool.blocks.size(); ++i) {
        const size_t have = pool.blocks[i].first;
        if (have >= bytes && have <= most && (best == pool.blocks.size() || have < pool.blocks[best].first)) best = i;
    }
    if (best == pool.blocks.size()) return nullptr;
    void *p = pool.blocks[best].second;
    *got = pool.blocks[best].first;
    pool.held -= *got;
    pool.blocks[best] = pool.blocks.back();
    pool.blocks.pop_back();
    return p;
}

thread_local bool g_refused;      // an allocation of this thread's call was refused for good
// `device` is current.  *got: what the block holds, 0 on failure.  insist: nothing is refused for what the library only keeps;
// without, nothing is given up for a block that the caller can do without.
hipError_t device_alloc(int device, size_t bytes, void **out, size_t *got, bool insist = true) {
    DevicePool &pool = g_pool[device];
    {
        std::lock_guard<std::mutex> lock(pool.mu);
        if (void *p = take_pooled(pool, bytes, got)) { *out = p; return hipSuccess; }
    }
    hipError_t e = hipMalloc(out, bytes);
    if (e != hipSuccess && insist) {
        (void)hipGetLastError();
        std::lock_guard<std::mutex> giving(pool.giving);      // (another thread's blocks may be on their way back)
        std::unique_lock<std::mutex> lock(pool.mu);
        const auto blocks = pool.empty();
        lock.unlock();
        free_blocks(blocks);
        e = hipMalloc(out, bytes);
        while (e != hipSuccess) {
            (void)hipGetLastError();
            lock.lock();
            void *spare = take_spare(pool);
            lock.unlock();
            if (spare == nullptr) break;
            (void)hipFree(spare);
            e = hipMalloc(out, bytes);
        }
        g_refused |= e != hipSuccess;
    }
    *got = e == hipSuccess ? bytes : 0;     // (callers keep it: a size without a block would pass for one)
    if (e != hipSuccess) (void)hipGetLastError();     // reported by this call, not by a later launch
    return e;
}
// Waits for the whole device first, as hipFree does: an index's memory is visible outside it
// (tv_index_device_ptrs), and work of other streams may still be reading.
hipError_t device_free(int device, void *p, size_t bytes) {
    if (p == nullptr) return hipSuccess;
    DevicePool &pool = g_pool[device];
    std::unique_lock<std::mutex> lock(pool.mu);
    const bool room = pool.takes(bytes);
    lock.unlock();
    if (room && hipDeviceSynchronize() == hipSuccess) {
        lock.lock();
        if (pool.takes(bytes)) {
            pool.blocks.emplace_back(bytes, p);
            pool.held += bytes;
            return hipSuccess;
        }
        lock.unlock();
    }
    const hipError_t e = hipFree(p);
    if (e != hipSuccess) (void)hipGetLastError();     // reported by this call, not by a later launch
    return e;
}

// Room for the stages of one search's two-step table scan (NearPlan): lent to one search of the device at a time, whichever
// index it is of, so that a device holds as many as it has such searches at once, kStagedBytes in all between them, and they do
// not take the place of blocks that indexes give up and take again (in the pool a 1 GiB block did: building the next index of 10M x 1536 2-bit
// rows 85 and 249 ms).  What idle places hold makes way where it stands between a search and that limit.  Null where there is no
// memory for one, or the searches that run hold too much: nothing else is given up for it.
constexpr size_t kStagedBytes = size_t(2) << 30;
tv_spare *staged_take(int device, size_t bytes) {
    DevicePool &pool = g_pool[device];
    tv_spare *s = nullptr;
    void *old[DevicePool::kStaged] = {};
    {
        std::lock_guard<std::mutex> lock(pool.mu);
        size_t held = 0, lent = 0;
        for (tv_spare &b : pool.staged) held += b.bytes, lent += b.in_use ? b.bytes : 0;
        for (tv_spare &b : pool.staged)      // the smallest that is large enough, otherwise the largest there is, or a free place
            if (!b.in_use && (s == nullptr || (b.bytes >= bytes ? s->bytes < bytes || b.bytes < s->bytes : s->bytes < bytes && b.bytes > s->bytes))) s = &b;
        if (s == nullptr || (s->bytes < bytes && lent + bytes > kStagedBytes)) return nullptr;
        s->in_use = true;
        if (s->bytes >= bytes) return s;
        held -= s->bytes;
        old[0] = std::exchange(s->p, nullptr);
        s->bytes = bytes;      // (counted while it is being allocated)
        s->p = take_pooled(pool, bytes, &s->bytes, kStagedBytes - lent);
        for (int i = 0, n = 1; i < DevicePool::kStaged; ++i) {
            tv_spare &b = pool.staged[i];
            if (b.in_use || held + s->bytes <= kStagedBytes) continue;
            held -= b.bytes;
            old[n++] = std::exchange(b.p, nullptr);
            b.bytes = 0;
        }
    }
    for (void *p : old) if (p != nullptr) (void)hipFree(p);
    if (s->p != nullptr) return s;      // (lent: nobody else changes it)
    void *p = nullptr;
    const hipError_t e = hipMalloc(&p, bytes);
    if (e != hipSuccess) (void)hipGetLastError();
    std::lock_guard<std::mutex> lock(pool.mu);
    s->p = e == hipSuccess ? p : nullptr;
    if (e != hipSuccess) s->bytes = 0;
    s->in_use = e == hipSuccess;
    return e == hipSuccess ? s : nullptr;
}
void staged_give(int device, tv_spare *s) {
    std::lock_guard<std::mutex> lock(g_pool[device].mu);
    s->in_use = false;
}

int ensure_workspace(tv_index *ix, size_t bytes) {
    if (bytes <= ix->ws_bytes) return TV_OK;
    if (ix->ws_fixed) {   // the caller lent a buffer of fixed size: never replaced
        g_last_error = "search needs " + std::to_string(bytes) + " bytes of scratch, the fixed buffer holds " +
                       std::to_string(ix->ws_bytes);
        return TV_ERR_BAD_ARGUMENT;
    }
    if (ix->ws) { TV_HIP(device_free(ix->device, ix->ws, ix->ws_bytes)); ix->ws = nullptr; ix->ws_bytes = 0; }
    bytes = round_up(bytes + bytes / 4, size_t(1) << 20);
    TV_HIP(device_alloc(ix->device, bytes, &ix->ws, &ix->ws_bytes));
    return TV_OK;
}

// An allocation of the index that grows on demand: what it held is gone then.
int ensure_block(tv_index *ix, void *&p, size_t &have, size_t bytes) {
    if (bytes <= have) return TV_OK;
    if (p) { TV_HIP(device_free(ix->device, p, have)); p = nullptr; have = 0; }
    bytes = round_up(bytes + bytes / 4, size_t(1) << 16);
    TV_HIP(device_alloc(ix->device, bytes, &p, &have));
    return TV_OK;
}
int ensure_io(tv_index *ix, size_t bytes) { return ensure_block(ix, ix->io, ix->io_bytes, bytes); }

// ---- host arrays ---------------------------------------------------------------------------------
// A copy from or to pageable memory is staged by the runtime, on one thread and with a wait of its own: 500 KB 30 us, 614 MB
// 20 to 39 ms.  Here calls on host arrays pass through pinned blocks that the device's indexes share: queries are copied in
// on the calling thread -- the snapshot of them that the search then reads -- and read by the device where they lie,
// results are written there by the last kernel; rows to add go through in pieces, several threads filling.  Through the Python
// surface, before and now: one query over 100K x 128 73 us and 37, 1000 queries 138 and 101, 1024 of 3072 dimensions 2.41 ms and 1.22; 100K
// x 1536 rows to an image 37.9 ms and 22.9.
constexpr size_t kPinnedBytes = size_t(256) << 20, kPinnedLargest = size_t(32) << 20;
constexpr size_t kReadInPlace = size_t(1) << 20;      // larger sets of queries are copied to the device first, by the copy engine

// A block of at least `bytes`, or null: none to spare, or none to be had (the caller then does without).  They are allocated on
// first use, at most kPinnedBytes of them, and freed with the device's last index; `device` is current.  (Pinning is slow: a
// new index's first search of 1000 queries of 128 dimensions 141 us with blocks of its own and 115 with another index's, of one query 70 and 44;
// with no other index it is 170, and 142 without pinned blocks.)
tv_pinned *pinned_take(int device, size_t bytes) {
    if (bytes > kPinnedLargest) return nullptr;
    size_t want = size_t(64) << 10;
    while (want < bytes) want *= 2;
    DevicePool &pool = g_pool[device];
    std::unique_lock<std::mutex> lock(pool.mu);
    size_t lent = 0, idle = 0;
    tv_pinned *fits = nullptr, *place = nullptr;
    for (tv_pinned &b : pool.pinned) {
        (b.lent ? lent : idle) += b.bytes;
        if (b.lent) continue;
        if (b.bytes >= want && (!fits || b.bytes < fits->bytes)) fits = &b;
        if (b.bytes == 0 && !place) place = &b;
    }
    if (fits) { fits->lent = true; return fits; }
    if (lent + want > kPinnedBytes) return nullptr;
    uint8_t *given_up[DevicePool::kPinned];      // of the idle blocks, all smaller, the largest first
    int n_given_up = 0;
    while (!place || lent + idle + want > kPinnedBytes) {
        tv_pinned *largest = nullptr;
        for (tv_pinned &b : pool.pinned)
            if (!b.lent && b.bytes != 0 && (!largest || b.bytes > largest->bytes)) largest = &b;
        if (!largest) return nullptr;     // (every block is lent)
        idle -= largest->bytes;
        given_up[n_given_up++] = largest->host;
        *largest = tv_pinned{};
        place = largest;
    }
    place->bytes = want;      // (counted, and nobody else's, while it is allocated)
    place->lent = true;
    lock.unlock();
    for (int i = 0; i < n_given_up; ++i) (void)hipHostFree(given_up[i]);
    void *host = nullptr, *dev = nullptr;
    bool got = hipHostMalloc(&host, want, hipHostMallocMapped) == hipSuccess;
    if (got && hipHostGetDevicePointer(&dev, host, 0) != hipSuccess) { (void)hipHostFree(host); got = false; }
    if (!got) (void)hipGetLastError();
    lock.lock();
    *place = got ? tv_pinned{static_cast<uint8_t *>(host), static_cast<uint8_t *>(dev), want, true} : tv_pinned{};
    return got ? place : nullptr;
}
struct PinnedLoan {      // given back when it goes out of scope; whoever reads or writes the block has finished by then
    int device;
    tv_pinned *b;
    PinnedLoan(int device_, size_t bytes) : device(device_), b(pinned_take(device_, bytes)) {}
    PinnedLoan(const PinnedLoan &) = delete;
    ~PinnedLoan() {
        if (!b) return;
        std::lock_guard<std::mutex> lock(g_pool[device].mu);
        b->lent = false;
    }
};
// Whether any of these values is not finite or 1e16 or larger.  A function of its own at the start of a cache line: inlined, the loop
// worked its end out anew at each turn and lay wherever the code around it put it, one line or two (1000 queries of 128
// dimensions 95.9 or 100.8 us a call from one build to the next, with the same kernels).
__attribute__((noinline, aligned(64))) bool any_refused(const uint32_t *v, size_t m) {
    uint32_t any = 0;
    for (size_t i = 0; i < m; ++i) any |= (kTooLargeBits - 1u) - (v[i] & 0x7fffffffu);      // (the sign, where the value is larger)
    return any >> 31;
}
// Copies values and says whether any of the copied ones is refused (tv_validate_queries).
bool copy_checked(float *to, const float *from, size_t n) {
    constexpr size_t kRun = 4096;      // copied, then looked at while in the first-level cache
    bool any = false;
    for (size_t r = 0; r < n; r += kRun) {
        const size_t m = std::min(kRun, n - r);
        std::memcpy(to + r, from + r, m * sizeof(float));
        any |= any_refused(reinterpret_cast<const uint32_t *>(to + r), m);
    }
    return any;
}

// The allocations of an index that has grown, which the copy out of them may still be reading: given up once the
// index's stream has been waited for.
struct Outgrown {
    tv_index *ix;
    uint8_t *codes = nullptr;
    float *scales = nullptr;
    size_t codes_bytes = 0, scales_bytes = 0;
    explicit Outgrown(tv_index *ix_) : ix(ix_) {}
    Outgrown(const Outgrown &) = delete;
    hipError_t release() {
        const hipError_t c = device_free(ix->device, std::exchange(codes, nullptr), codes_bytes);
        const hipError_t s = device_free(ix->device, std::exchange(scales, nullptr), scales_bytes);
        return c != hipSuccess ? c : s;
    }
    ~Outgrown() {
        if (codes == nullptr && scales == nullptr) return;
        (void)hipStreamSynchronize(ix->stream);
        (void)release();
    }
};
// What an allocation in the making holds beyond growing by half: the index's from keep() on, in the place of what its old one held.
struct AheadHold {
    tv_index *ix;
    DevicePool &pool;
    size_t bytes = 0;
    explicit AheadHold(tv_index *ix_) : ix(ix_), pool(g_pool[ix_->device]) {}
    AheadHold(const AheadHold &) = delete;
    bool take(size_t more) {
        std::lock_guard<std::mutex> lock(pool.mu);
        if (pool.ahead - ix->ahead + more > kAheadBytes) return false;
        pool.ahead += more;
        bytes = more;
        return true;
    }
    void keep() {
        std::lock_guard<std::mutex> lock(pool.mu);
        pool.ahead -= std::exchange(ix->ahead, std::exchange(bytes, 0));
    }
    void drop() {
        std::lock_guard<std::mutex> lock(pool.mu);
        pool.ahead -= std::exchange(bytes, 0);
    }
    ~AheadHold() { drop(); }
};
// Room for n_vectors rows.  An index grows to twice its size while the device's indexes hold no more than kAheadBytes for that, and by half
// beyond: 100K rows of 1536 dimensions added four times move 231 MB on the way (461 MB by half each time).  Where there is no
// memory for either it grows by what is needed, and only that is worth giving up what others keep.
// What is beyond the rows is zero -- but for the blocks that rows from the index's last to n_vectors fill, where the
// caller says that it is about to write all of those on the index's stream (`whole`), and not before it has waited for the
// stream, which it does before `outgrown` goes.
int ensure_capacity(tv_index *ix, size_t n_vectors, Outgrown &outgrown, bool whole) {
    const size_t blocks = (n_vectors + tv::kVecBlock - 1) / tv::kVecBlock;
    if (blocks <= ix->cap_blocks) return TV_OK;
    const size_t bb = ix->geo.block_bytes();
    const size_t needed = std::max<size_t>(blocks, 64), half = std::max(needed, ix->cap_blocks + ix->cap_blocks / 2);
    size_t cap = std::max(half, 2 * ix->cap_blocks);
    AheadHold ahead(ix);
    if (cap > half && !ahead.take((cap - half) * (bb + tv::kVecBlock * sizeof(float)))) cap = half;
    uint8_t *codes = nullptr;
    float *scales = nullptr;
    size_t codes_bytes = 0, scales_bytes = 0;
    hipError_t e = hipSuccess;
    for (;; cap = cap > half ? half : needed) {
        if (cap <= half) ahead.drop();
        e = device_alloc(ix->device, cap * bb, reinterpret_cast<void **>(&codes), &codes_bytes, cap == needed);
        if (e == hipSuccess) {
            e = device_alloc(ix->device, cap * tv::kVecBlock * sizeof(float), reinterpret_cast<void **>(&scales), &scales_bytes, cap == needed);
            if (e == hipSuccess) break;
            (void)device_free(ix->device, codes, codes_bytes);
        }
        if (cap == needed) return fail_hip(e, "device_alloc(rows)");
    }
    const size_t old_blocks = (ix->n + tv::kVecBlock - 1) / tv::kVecBlock;
    const size_t clear = whole ? std::max(old_blocks, n_vectors / tv::kVecBlock) : old_blocks;
    // fresh bytes are zero so padding lanes match a from-scratch upload
    e = hipMemsetAsync(codes + clear * bb, 0, (cap - clear) * bb, ix->stream);
    if (e == hipSuccess) e = hipMemsetAsync(scales + clear * tv::kVecBlock, 0, (cap - clear) * tv::kVecBlock * sizeof(float), ix->stream);
    if (e == hipSuccess && old_blocks) {
        e = hipMemcpyAsync(codes, ix->d_codes, old_blocks * bb, hipMemcpyDeviceToDevice, ix->stream);
        if (e == hipSuccess) e = hipMemcpyAsync(scales, ix->d_scales, old_blocks * tv::kVecBlock * sizeof(float), hipMemcpyDeviceToDevice, ix->stream);
    }
    if (e != hipSuccess) {
        (void)hipStreamSynchronize(ix->stream);
        (void)device_free(ix->device, codes, codes_bytes);
        (void)device_free(ix->device, scales, scales_bytes);
        return fail_hip(e, "growing the index");
    }
    outgrown.codes = std::exchange(ix->d_codes, codes);
    outgrown.scales = std::exchange(ix->d_scales, scales);
    outgrown.codes_bytes = std::exchange(ix->codes_bytes, codes_bytes);
    outgrown.scales_bytes = std::exchange(ix->scales_bytes, scales_bytes);
    ix->cap_blocks = cap;
    ahead.keep();
    return TV_OK;
}
int ensure_capacity(tv_index *ix, size_t n_vectors) {
    Outgrown outgrown(ix);
    const size_t before = ix->cap_blocks;
    const int rc = ensure_capacity(ix, n_vectors, outgrown, false);
    if (rc != TV_OK || ix->cap_blocks == before) return rc;
    TV_HIP(hipStreamSynchronize(ix->stream));
    TV_HIP(outgrown.release());
    return TV_OK;
}

// An upload replaces the contents: blocks of the old contents beyond the new end are cleared, so
// that rows appended later land in zeroed blocks (padding lanes zero, as in a from-scratch
// upload; pack.rs:235-243, :354).
int clear_tail_blocks(tv_index *ix, size_t n_blocks) {
    if (n_blocks >= ix->cap_blocks) return TV_OK;
    const size_t bb = ix->geo.block_bytes();
    TV_HIP(hipMemsetAsync(ix->d_codes + n_blocks * bb, 0, (ix->cap_blocks - n_blocks) * bb, ix->stream));
    TV_HIP(hipMemsetAsync(ix->d_scales + n_blocks * tv::kVecBlock, 0,
                          (ix->cap_blocks - n_blocks) * tv::kVecBlock * sizeof(float), ix->stream));
    return TV_OK;
}

// turbovec/src/search.rs:2812-2820: the codebook as int8 levels, one scale.
void derive_levels(tv_index *ix) {
    float cmax = 0.0f;
    for (float c : ix->cb.centroids) cmax = std::fmax(cmax, std::fabs(c));
    ix->cs = cmax > 0.0f ? cmax / 127.0f : 1.0f;
    std::memset(ix->levels, 0, sizeof ix->levels);
    for (size_t i = 0; i < ix->cb.centroids.size() && i < 16; ++i) {
        float v = std::round(ix->cb.centroids[i] / ix->cs);
        v = v < -127.0f ? -127.0f : (v > 127.0f ? 127.0f : v);
        ix->levels[i] = int8_t(v);
    }
    // (the scan in front of the tables: 2-bit codebooks are 3 : 10 to within 0.002 at every dimension, and the smaller and the
    // fewer-signed the operands, the higher the clock under the matrix unit's load: 0, 14, 26, 40 for -20, -6, 6, 20; 10M x 1536, 1024 queries 15.95 ms a
    // search with levels up to 127 in size, 15.65 up to 20, 15.55 up to 20 and lifted)
    const bool two = ix->geo.bits == 2;
    ix->near_cs = cmax > 0.0f ? cmax / (two ? 20.0f : 127.0f) : 1.0f;
    std::memset(ix->near_levels, 0, sizeof ix->near_levels);
    for (size_t i = 0; i < ix->cb.centroids.size() && i < 8; ++i) {
        const float v = std::round(ix->cb.centroids[i] / ix->near_cs) + (two ? 20.0f : 0.0f);
        ix->near_levels[i] = int8_t(std::fmin(std::fmax(v, -127.0f), 127.0f));
    }
}

// The tables that only the dimension decides, with the encoder's form of them: as an index's device tables begin (signs, gathers,
// packed words, two rounds each).  Drawing and packing them took 48 us of 1536 dimensions' 110 an index, 129 at 3072: the last kTableMemo are kept.
struct TableImage {
    tv::RotationTables rot;
    std::vector<uint32_t> words;
    bool packed_ok = false;
};
constexpr size_t kTableMemo = 8;
void lay_out_tables(const tv::RotationTables &rot, TableImage &t) {
    const size_t d2 = 2 * size_t(rot.dim);
    t.words.assign(3 * d2, 0u);
    std::memcpy(t.words.data(), rot.signs.data(), d2 * sizeof(float));
    std::memcpy(t.words.data() + d2, rot.perms.data(), d2 * sizeof(uint32_t));
    t.packed_ok = tv::encode_pack_tables(rot.signs.data(), rot.perms.data(), rot.dim, rot.block, t.words.data() + 2 * d2);
}
std::shared_ptr<const TableImage> default_tables(int dim) {
    static std::mutex mu;
    static std::vector<std::shared_ptr<const TableImage>> memo;      // the one used last first
    std::lock_guard<std::mutex> lock(mu);
    for (size_t i = 0; i < memo.size(); ++i)
        if (memo[i]->rot.dim == dim) {
            std::rotate(memo.begin(), memo.begin() + i, memo.begin() + i + 1);
            return memo[0];
        }
    auto t = std::make_shared<TableImage>();
    t->rot = tv::make_rotation_tables(dim);
    lay_out_tables(t->rot, *t);
    if (memo.size() == kTableMemo) memo.pop_back();
    memo.insert(memo.begin(), t);
    return t;
}

constexpr size_t kChunkQueries = 1024;
// a chunk's floors are laid out tile by tile, kQTile slots per tile, and a tile may hold one query
constexpr size_t kTauOpenInts = kChunkQueries * tv::kQTile;

// On the index's stream, from pinned memory of its own, which the device reads where it lies (four copies from pageable memory took 40 us
// of an index's 90).  The caller waits before its call ends, so that the tables are there and an error is that call's own.
int upload_tables(tv_index *ix, const TableImage &t) {
    const size_t words = t.words.size();
    std::memcpy(ix->h_tables, t.words.data(), words * sizeof(uint32_t));
    float *cen = reinterpret_cast<float *>(ix->h_tables + words);
    std::fill_n(cen, 16, 0.0f);
    for (size_t i = 0; i < ix->cb.centroids.size(); ++i) cen[i] = ix->cb.centroids[i];
    ix->packed_ok = t.packed_ok;
    // (and the floors of a search's first sampling level: the order key of -inf for every query)
    TV_HIP(tv::launch_lay_tables(ix->d_flags_host + (ix->h_tables - ix->h_flags), reinterpret_cast<uint32_t *>(ix->d_signs), words + 16, ix->d_tau_open, int(0x807fffffu), kTauOpenInts, ix->stream));
    return TV_OK;
}
int effective_mode(const tv_index *ix);
// Queries one LUT-scan launch serves: the scalar definition's float chain runs one query at a time.
int lut_tile_q(const tv_index *ix, int k) { return effective_mode(ix) == TV_SCORE_L_SCALAR ? 1 : tv::lut_tile_queries(ix->geo.nch, k); }
// Batches of u8-LUT queries beyond what the whole-table scan serves in one pass (eight queries, fewer
// where the rows are long) go sixteen queries per pass through k_scan_lut16 or, with the u32
// epilogue, all in one launch of the sparse matrix-unit scan; the scalar definition's chain of adds
// takes one query at a time.  One pass for up to sixteen queries beats the matrix-unit scan's
// half-empty tile (1M x 1536 2-bit, 16 queries: 0.26 ms a search against 0.30); from 17 on it
// would be two (33 queries: 0.56 against 0.40 ms; 400: 4.6 against 2.2).  Below about 4096 (block,
// query tile) pairs most of the matrix-unit scan's waves have no block, and up to three sixteen-query passes
// are the faster ones (20K x 1536 2-bit, 33 queries, 1250 pairs: 153 us against 155; 65K rows, 4096
// pairs: 165 against 131).  From four passes on (us a search, the passes and the matrix-unit scan):
//  - 1400 pairs: 12K x 1536 2-bit, 100 queries 75 and 62, 15K x 3072, 96 queries 106 and 91; 1000 pairs are level or worse (15K x 3072, 49 queries 83 and 90).
//  - 3-bit codes, half the products per byte: 2000 x 3072, 65 queries 123 and 115, 700 x 1536, 65 queries, k = 100 183 and 79; 49 queries
//    over 1000 x 3072 120 and 113, 10K x 1536 80 and 72.
//  - up to six chunks: 1000 x 768 2-bit, 129 queries 44.5 and 43.1, x 128 37.5 and 32.1; twelve 57.5 and 59.2.
//  - many passes, one after the other where the search is sampled: 6000 x 3072 2-bit, 1000 queries 197 either way, 3000 1430 and 166, without
//    sampling 222 and 160; 4000, 400 queries 131 and 112, but 129 queries 86 and 92.
constexpr size_t kMxMinPairs = 4096, kMxMinPairsMany = 1400, kMxMany = 3 * tv::kLut16Queries, kMxAlways = 384;
bool lut_mx_serves(const tv_index *ix, size_t cq) {
    const size_t n_blocks = (ix->rows().n + tv::kVecBlock - 1) / tv::kVecBlock, tiles = (cq + tv::kQTile - 1) / tv::kQTile, pairs = n_blocks * tiles;
    if (effective_mode(ix) != TV_SCORE_L_U32 || ix->no_lut16 || ix->no_lut_mx || cq <= size_t(tv::kLut16Queries)) return false;
    return pairs >= kMxMinPairs || (cq > kMxMany && (pairs >= kMxMinPairsMany || ix->geo.bits == 3 || ix->geo.nch <= 6 || cq > kMxAlways));
}
bool lut16_serves(const tv_index *ix) {
    return (effective_mode(ix) == TV_SCORE_L_U32 || effective_mode(ix) == TV_SCORE_L_CLASSIC) && !ix->no_lut16;
}
// Tiles of fewer queries than this keep the whole-table scan (its pass is as long for 8 queries as for 1).
int lut16_min_queries(const tv_index *ix) { return tv::lut_append_queries(ix->geo.nch) + 1; }
int lut_append_q(const tv_index *ix, size_t cq) {
    if (effective_mode(ix) == TV_SCORE_L_SCALAR) return 1;
    return lut_mx_serves(ix, cq) ? tv::kQTile : lut16_serves(ix) ? tv::kLut16Queries : tv::lut_append_queries(ix->geo.nch);
}

int effective_mode(const tv_index *ix) {
    int m = ix->score_mode;
    if (m == TV_SCORE_AUTO) m = ix->geo.bits == 4 ? TV_SCORE_P : TV_SCORE_L_U32;
    return m;
}

struct Prepared {
    float *d_qrot = nullptr;   // rotated (and calibrated) rows
    uint8_t *d_tables = nullptr;
    uint8_t *d_tables16 = nullptr;   // mode L: the same tables entry-major for the sixteen-query scan (or null)
    uint8_t *d_tables_mx = nullptr;  // mode L: the same tables as matrix operands for the sparse scan (or null)
    float *d_qscale = nullptr, *d_qbias = nullptr;
    uint8_t *d_near = nullptr;       // mode L: int8 weights of the scan in front of the tables (or null) ...
    float *d_near_unit = nullptr, *d_near_err = nullptr;
    size_t table_bytes_per_tile = 0;
};

// Query preparation for one chunk: rotation, TQ+ inverse, table build
// (turbovec/src/search.rs:3237-3269).  d_q holds nq*dim floats on the device.
// `split`: permute-dot weights in the order k_scan_p4 reads them (the batched scans take plane order)
// `keep_rotated`: the rotated rows are wanted in device memory too (the debug read-back).
// `for_append`: u8-LUT tables are wanted in the order of the batch's append scan too.
// `cleared`: a word per query to set to zero.
// `near`: what the two-step table scan reads as well (where the matrix-unit scan serves).
int prepare_queries(tv_index *ix, Arena &ar, const float *d_q, size_t nq, Prepared &out, bool split = true,
                    bool keep_rotated = false, bool for_append = false, uint64_t *stamp = nullptr, uint64_t *cleared = nullptr, bool near = false) {
    const tv::Geometry &g = ix->geo;
    const size_t nq_pad = round_up(nq, tv::kQTile);
    const int mode = effective_mode(ix);
    const bool cal = !ix->tq_shift.empty(), mode_p = mode == TV_SCORE_P;
    tv::PrepRequest r{};
    r.q = d_q;
    r.signs = ix->d_signs;
    r.perms = ix->d_perms;
    r.block = ix->rot.block;
    r.inv_sqrt_block = ix->rot.inv_sqrt_block;
    r.shift = cal ? ix->d_tq_shift : nullptr;
    r.scale = cal ? ix->d_tq_scale : nullptr;
    r.permute_dot = mode_p;
    r.split = split;
    r.cs = ix->cs;
    r.centroids = ix->d_centroids;
    r.rot_out = out.d_qrot = keep_rotated ? ar.take<float>(nq * g.dim) : nullptr;
    r.qscale = out.d_qscale = ar.take<float>(nq_pad);
    r.qbias = out.d_qbias = ar.take<float>(nq_pad);
    out.table_bytes_per_tile = mode_p ? size_t(g.nch) * 2048 : size_t(g.nch) * 1024 * tv::kQTile;
    r.tables = out.d_tables = ar.take<uint8_t>(nq_pad / tv::kQTile * out.table_bytes_per_tile);
    const bool mx = !mode_p && for_append && lut_mx_serves(ix, nq);
    if (mx) r.tables_mx = out.d_tables_mx = ar.take<uint8_t>(tv::mx_table_bytes(g.nch, g.bits, nq));
    r.stamp = stamp;
    r.cleared = cleared;
    if (near) {
        r.near = out.d_near = ar.take<uint8_t>(nq_pad * size_t(tv::near_nch(g.nch, g.bits)) * 32 * size_t(8 / g.bits));
        r.near_unit = out.d_near_unit = ar.take<float>(nq_pad);
        r.near_err = out.d_near_err = ar.take<float>(nq_pad);
        r.near_cs = ix->near_cs;
        std::memcpy(r.lv, ix->near_levels, sizeof r.lv);
    }
    TV_HIP(tv::launch_prep(r, g, nq, nq_pad, ix->stream));
    if (!mode_p && !mx && for_append && lut16_serves(ix) && nq >= size_t(lut16_min_queries(ix))) {
        out.d_tables16 = ar.take<uint8_t>(tv::lut16_table_bytes(g.nch, nq));
        TV_HIP(tv::launch_lut_interleave16(out.d_tables, out.d_tables16, g.nch, nq, ix->stream));
    }
    return TV_OK;
}

size_t prepare_bytes(const tv_index *ix, size_t nq) {
    const tv::Geometry &g = ix->geo;
    const size_t nq_pad = round_up(nq, tv::kQTile);
    size_t b = 2 * round_up(nq * g.dim * 4, 256) + 3 * round_up(nq_pad * 4, 256);
    b += round_up(nq_pad * size_t(g.nch) * 1024, 256) + 4096;
    if (lut_mx_serves(ix, nq)) b += round_up(tv::mx_table_bytes(g.nch, g.bits, nq), 256);
    else if (lut16_serves(ix)) b += round_up(tv::lut16_table_bytes(g.nch, nq), 256);
    return b;
}

void fill_scan_args(const tv_index *ix, tv::ScanArgs &a) {
    std::memset(&a, 0, sizeof a);
    const tv_rows rows = ix->rows();
    a.codes = rows.codes;
    a.scales = rows.scales;
    a.n = uint32_t(rows.n);
    a.rows = rows.in_place ? rows.slots : nullptr;
    a.n_blocks = uint32_t((rows.n + tv::kVecBlock - 1) / tv::kVecBlock);
    a.nch = ix->geo.nch;
    std::memcpy(a.lv, ix->levels, 16);
    a.classic = effective_mode(ix) == TV_SCORE_L_CLASSIC ? 1 : effective_mode(ix) == TV_SCORE_L_SCALAR ? 2 : 0;
    a.n_groups = ix->geo.G;
    a.b_step = 1;
}

constexpr int kMaxTimedTiles = int(kChunkQueries / tv::kQTile);

static_assert(kMaxTimedTiles == tv::kTimedLaunches, "the index holds one event pair per timed launch");

// The events that time scan launches belong to the index (created on first use under its lock,
// destroyed with it).
int ensure_events(tv_index *ix) {
    if (ix->events_ready) return TV_OK;
    for (int i = 0; i < kMaxTimedTiles; ++i) {
        TV_HIP(hipEventCreate(&ix->ev_start[i]));
        TV_HIP(hipEventCreate(&ix->ev_stop[i]));
    }
    ix->events_ready = true;
    return TV_OK;
}

// The two-step table scan: two tiles of queries are level at best, three ahead (us a search without and so: 2.3M x 384 2-bit, 47 queries 240 and 299; 6.2M x 768, 59
// 975 and 901; 4.1M x 384, 64 397 and 378; 7.1M x 456, 84 1431 and 826; 2.8M x 1360, 75 1530 and 943; 2.4M x 512 3-bit, 76 587
// and 480, 752 dimensions, 52 450 and 532; 1M x 1128, 86 557 and 485; 10M x 1536, 1024 45 900 and 15 900).
constexpr size_t kNearMinQueries = 65;
// Bytes of the operands it takes beside the tables; 0 where a chunk of so many queries cannot go that way, as on scratch of a fixed
// size, whose limits they would lower.
size_t near_bytes(const tv_index *ix, size_t cq) {
    const tv::Geometry &g = ix->geo;
    if (ix->ws_fixed || (!ix->force_near && cq < kNearMinQueries) || !lut_mx_serves(ix, cq) || tv::near_chunks(g.nch, g.bits) == 0) return 0;
    const size_t nq_pad = round_up(cq, tv::kQTile);
    return round_up(nq_pad * size_t(tv::near_nch(g.nch, g.bits)) * 32 * size_t(8 / g.bits), 256) + 2 * round_up(nq_pad * 4, 256);
}

// Workspace bytes one chunk of cq queries needs on the exact path (search_robust) ...
size_t robust_need(const tv_index *ix, size_t cq, size_t k_eff) {
    const tv::Geometry &g = ix->geo;
    const bool mode_p = effective_mode(ix) == TV_SCORE_P;
    const bool lists = k_eff <= size_t(tv::kMaxListK);
    const int kl = lists ? int(k_eff) : 1;
    const size_t tile_q = mode_p ? size_t(tv::kQTile) : size_t(lut_tile_q(ix, kl));
    const size_t n_tiles = (cq + tile_q - 1) / tile_q;
    const int grid = tv::scan_grid_blocks(ix->device, mode_p, g.nch, kl, int(tile_q));
    const size_t total_threads = size_t(grid) * tv::kScanThreads;
    size_t need = prepare_bytes(ix, cq) + round_up(n_tiles * tv::kQTile * 4, 256);
    if (lists) need += 2 * round_up(k_eff * total_threads * 4, 256) + round_up(total_threads * 4, 256);
    else need += round_up(size_t(tv::kQTile) * ix->rows().n * 4, 256) + round_up(tv::select_tmp_keys(k_eff) * 8 * tv::kQTile, 256) +
                 round_up(size_t(tv::kQTile) * 4096 * 4, 256);
    return need + 65536;
}

// ... and on the sampled path (search_device): prepared queries, floors, candidate segments.
struct SampledPlan {
    size_t tile_q, n_tiles, cq_pad, seg_stride, need;
    bool wide;
    bool lut_mx;        // u8-LUT queries of this chunk take the sparse matrix-unit scan, all in one launch
    bool lut16;         // u8-LUT tiles of this chunk take the sixteen-query scan
    int grid_near;      // workgroups of the int8 scan in front of the tables
    bool lut_single;    // one u8-LUT query, served by the byte-table scan
    int nt_batched;     // query tiles one launch of the tile-group kernels serves (0: one tile per launch)
    int grid;
};
SampledPlan sampled_plan(const tv_index *ix, size_t cq) {
    const tv::Geometry &g = ix->geo;
    const bool mode_p = effective_mode(ix) == TV_SCORE_P;
    SampledPlan p;
    p.tile_q = mode_p ? size_t(tv::kQTile) : size_t(lut_append_q(ix, cq));
    p.n_tiles = (cq + p.tile_q - 1) / p.tile_q;
    p.cq_pad = p.n_tiles * p.tile_q;
    // large chunks of high-dimensional queries take the wide kernel: all of them in one pass per level
    const int wide_min = tv::wide_min_queries(g.nch);
    p.wide = mode_p && !ix->no_batched && !ix->no_wide && wide_min > 0 && cq >= size_t(wide_min);
    p.lut_mx = !mode_p && lut_mx_serves(ix, cq);
    p.lut16 = !mode_p && !p.lut_mx && lut16_serves(ix) && cq >= size_t(lut16_min_queries(ix));
    p.nt_batched = (mode_p && cq > size_t(tv::kQTile) && !ix->no_batched) ? tv::batched_tiles(g.nch) : 0;
    p.grid = p.wide ? tv::wide_grid_blocks(ix->device)
           : mode_p ? tv::scan_grid_blocks(ix->device, mode_p, g.nch, 0, int(p.tile_q))
                    : tv::lut_append_grid(ix->device, g.nch);
    p.grid_near = tv::wide_grid_blocks(ix->device);
    p.lut_single = !mode_p && cq == 1 && effective_mode(ix) != TV_SCORE_L_SCALAR && tv::lut_single_uses_byte_tables(g.nch, p.grid);
    p.seg_stride = p.lut_mx ? size_t(tv::mx_segments()) : size_t(p.grid);
    // (a query keeps one candidate segment per workgroup of the launches that serve it: every launch
    // of a chunk the tile-group kernels serve is one of theirs, and their grid is not the single-tile scan's)
    if (p.nt_batched > 0 && !p.wide) p.seg_stride = size_t(tv::batched_grid_blocks(ix->device, g.nch));
    p.need = prepare_bytes(ix, cq) + near_bytes(ix, cq) + round_up(p.n_tiles * tv::kQTile * 4, 256) +
             round_up(p.cq_pad * p.seg_stride * tv::kSegCap * 8, 256) + round_up(p.cq_pad * p.seg_stride * 4, 256) +
             round_up(p.cq_pad * 4, 256) + 65536;
    return p;
}

// Sampling plan of a search: block strides of the successive append-mode scans,
// the last one being 1 (the full scan).  The first level reads about `first`
// slots and, having no floor yet, appends all of them (one short sort); level
// sizes then grow geometrically to the full index, by a factor chosen so that
// a level filtered by the floor of the one before appends at most about 4096
// candidates per query (the floor is the k_floor-th best of the level before,
// so a level `ratio` times larger keeps about ratio * k_floor).  The sampling
// levels together read about 1/ratio of the index.
struct SamplingSteps {
    static constexpr int kMax = 32;   // levels grow at least fourfold: 2^31 slots need 16 at most
    uint32_t step[kMax];
    size_t count = 0;
    bool best_first = false;   // the first level runs without floors and hands over the best row of every block it reads ...
    bool best_words = false;   // ... as a score word, from a launch of the unsampled search's scan (launch_floor takes the floors)
    size_t size() const { return count; }
    uint32_t operator[](size_t i) const { return step[i]; }
};
// `round_blocks` > 0: the scan kernel works through the blocks in rounds of that many (one per
// wave of the grid) and a level costs whole rounds whatever it fills of the last one; a level
// larger than a round is trimmed to whole rounds (its floor gets a little lower, the next level
// a little longer: at 10M rows 3157 blocks become 2048, one round instead of two).
SamplingSteps sampling_steps(size_t n_blocks, size_t k_floor, size_t round_blocks = 0) {
    const double n_slots = double(n_blocks * tv::kVecBlock);
    const double first = double(std::max<size_t>(1024, 8 * k_floor));
    SamplingSteps steps;
    if (n_slots > 2.0 * first) {
        const double max_ratio = std::max(4.0, double(tv::kFinalCap / 2) / double(k_floor));
        const int levels = std::max(1, int(std::ceil(std::log(n_slots / first) / std::log(max_ratio))));
        const double ratio = std::pow(n_slots / first, 1.0 / double(levels));
        double sample = first;
        for (int lv = 0; lv < levels && steps.count + 1 < size_t(SamplingSteps::kMax); ++lv, sample *= ratio) {
            size_t sample_blocks = std::max<size_t>(1, size_t(sample) / tv::kVecBlock);
            if (round_blocks > 0 && sample_blocks > round_blocks) sample_blocks -= sample_blocks % round_blocks;
            // a trimmed level must not spill into one more round: step rounded up
            const size_t step = round_blocks > 0 && sample_blocks >= round_blocks ? (n_blocks + sample_blocks - 1) / sample_blocks
                                                                                  : n_blocks / sample_blocks;
            if (step > 1 && (steps.count == 0 || step < steps.step[steps.count - 1])) steps.step[steps.count++] = uint32_t(step);
        }
    }
    steps.step[steps.count++] = 1;
    return steps;
}

// The all-queries-per-pass kernel holds 16 bytes of LDS per query beside its slice ring: a call with
// more than kChunkQueries queries left takes them up to kWideChunkQueries at a time there -- a block
// is then loaded and decoded once per 64 query tiles instead of once per 32.
constexpr size_t kWideChunkQueries = 2 * kChunkQueries;      // (where the instance for the row length fits that many)
bool wide_serves(const tv_index *ix) {
    return effective_mode(ix) == TV_SCORE_P && !ix->no_batched && !ix->no_wide && tv::wide_min_queries(ix->geo.nch) > 0;
}
size_t chunk_len(const tv_index *ix, size_t remaining) {
    if (remaining > kChunkQueries && wide_serves(ix))
        return std::min(remaining, std::min<size_t>(kWideChunkQueries, size_t(tv::wide_max_queries(ix->geo.nch))));
    return std::min(remaining, kChunkQueries);
}

// Queries of one call are processed in chunks (chunk_len); the chunks of a group are enqueued
// back to back and the host reads their overflow flags once, after the group's last chunk.
constexpr size_t kGroupQueries = 8 * kChunkQueries;
constexpr size_t kLevelFlagWords = (kGroupQueries / kChunkQueries) * SamplingSteps::kMax;   // per chunk, one word per level

// What a group keeps at the head of the workspace across its passes: per query the overflow flag and
// the raised floor of the first pass; for the repeated pass the rows to repeat and their queries
// packed (one chunk's worth at a time); the per-level "candidates did not fit" flags of the pass in
// flight.
size_t group_header_bytes(const tv_index *ix, size_t gq) {
    const size_t cq = std::min(gq, kWideChunkQueries);
    return 2 * round_up(gq * 4, 256) + round_up(cq * 4, 256) + round_up(cq * size_t(ix->geo.dim) * 4, 256) +
           round_up(kLevelFlagWords * 4, 256);
}

// Workspace the sampled path needs for a call of nq queries: the header of its largest group, the
// working set of a full chunk (or of the only, smaller one), and room for the repeated pass to run
// at least a tile of queries at a time (a smaller packed batch may fall to another kernel with
// more candidate segments per query; it is then cut into pieces that fit).
constexpr size_t kRepeatPieces[] = {1024, 512, 256, 128, 96, 64, 32};
size_t sampled_need_worst(const tv_index *ix, size_t nq) {
    const size_t gq = std::min(nq, kGroupQueries);
    size_t need = 0;
    auto chunks_of_group = [&](size_t group_queries) {
        for (size_t c0 = 0; c0 < group_queries;) {
            const size_t cq = chunk_len(ix, group_queries - c0);
            need = std::max(need, sampled_plan(ix, cq).need);
            c0 += cq;
        }
    };
    chunks_of_group(gq);                                                              // a full group, or the only one
    if (nq > kGroupQueries && nq % kGroupQueries != 0) chunks_of_group(nq % kGroupQueries);   // and the last, shorter one
    need = std::max(need, sampled_plan(ix, std::min<size_t>(nq, tv::kQTile)).need);
    return need + group_header_bytes(ix, gq);
}

// Full-range search without sampling: per-lane lists with shared thresholds for
// k <= 32, dense scores + radix select beyond.  Always exact; used for the
// queries whose candidate buffer overflowed and for very large k.
int search_robust(tv_index *ix, const float *d_queries, size_t nq, size_t k_eff, const uint64_t *d_mask,
                  float *d_out_scores, int64_t *d_out_idx, bool timed_run) {
    const size_t n = ix->rows().n;
    const tv::Geometry &g = ix->geo;
    const int mode = effective_mode(ix);
    const bool mode_p = mode == TV_SCORE_P;
    const bool lists = k_eff <= size_t(tv::kMaxListK);
    int rc = TV_OK;
    for (size_t q0 = 0; q0 < nq; q0 += kChunkQueries) {
        const size_t cq = std::min(kChunkQueries, nq - q0);
        const int kl = lists ? int(k_eff) : 1;
        const size_t tile_q = mode_p ? size_t(tv::kQTile) : size_t(lut_tile_q(ix, kl));
        const size_t n_tiles = (cq + tile_q - 1) / tile_q;
        const int grid = tv::scan_grid_blocks(ix->device, mode_p, g.nch, kl, int(tile_q));
        const size_t total_threads = size_t(grid) * tv::kScanThreads;
        rc = ensure_workspace(ix, robust_need(ix, cq, k_eff));
        if (rc != TV_OK) return rc;
        Arena ar;
        ar.base = static_cast<uint8_t *>(ix->ws);
        Prepared pq;
        rc = prepare_queries(ix, ar, d_queries + q0 * g.dim, cq, pq);
        if (rc != TV_OK) return rc;
        int *d_tau = ar.take<int>(n_tiles * tv::kQTile);
        TV_HIP(tv::launch_fill_i32(d_tau, int(0x807fffffu) /* order key of -inf */, n_tiles * tv::kQTile, ix->stream));
        float *d_part_s = nullptr, *d_dense = nullptr;
        uint32_t *d_part_i = nullptr, *d_hist = nullptr;
        int *d_part_c = nullptr;
        uint64_t *d_keys = nullptr;
        if (lists) {
            d_part_s = ar.take<float>(k_eff * total_threads);
            d_part_i = ar.take<uint32_t>(k_eff * total_threads);
            d_part_c = ar.take<int>(total_threads);
        } else {
            d_dense = ar.take<float>(size_t(tv::kQTile) * n);
            d_keys = ar.take<uint64_t>(tv::select_tmp_keys(k_eff) * tv::kQTile);
            d_hist = ar.take<uint32_t>(size_t(tv::kQTile) * 4096);
        }
        for (size_t t = 0; t < n_tiles; ++t) {
            tv::ScanArgs a;
            fill_scan_args(ix, a);
            a.mask = d_mask;
            a.tables = pq.d_tables + t * (mode_p ? pq.table_bytes_per_tile : tile_q * size_t(g.nch) * 1024);
            a.qscale = pq.d_qscale + t * tile_q;
            a.qbias = pq.d_qbias + t * tile_q;
            a.nq_tile = int(std::min<size_t>(tile_q, cq - t * tile_q));
            a.k = kl;
            a.gtau = d_tau + t * tv::kQTile;
            a.part_scores = d_part_s; a.part_idx = d_part_i; a.part_cnt = d_part_c;
            a.score_out = d_dense;
            a.share_tau = 1;
            if (!lists && d_mask)  // blocks without an allowed slot are skipped by the scan: mark them excluded
                TV_HIP(tv::launch_fill_i32(reinterpret_cast<int *>(d_dense), 0x7fc00000, size_t(a.nq_tile) * n, ix->stream));
            const bool timed = timed_run && int(t) < kMaxTimedTiles;
            const int smode = lists ? tv::kModeLists : tv::kModeDump;
            if (timed) TV_HIP(hipEventRecord(ix->ev_start[t], ix->stream));
            if (mode_p) TV_HIP(tv::launch_scan_p4(a, grid, smode, ix->stream));
            else TV_HIP(tv::launch_scan_lut(a, grid, smode, ix->stream));
            if (timed) TV_HIP(hipEventRecord(ix->ev_stop[t], ix->stream));
            float *os = d_out_scores + (q0 + t * tile_q) * k_eff;
            int64_t *oi = d_out_idx + (q0 + t * tile_q) * k_eff;
            if (lists) {
                const int qmod = mode_p ? tv::kQTile : mode == TV_SCORE_L_SCALAR ? 1 : tv::lut_launch_ql(g.nch, kl, a.nq_tile);
                TV_HIP(tv::launch_merge(d_part_s, d_part_i, d_part_c, int(total_threads), qmod, int(k_eff), int(k_eff),
                                        a.nq_tile, os, oi, nullptr, ix->stream));
            } else {
                TV_HIP(tv::launch_select_topk(d_dense, n, a.nq_tile, k_eff, d_keys, d_hist, os, oi, ix->stream));
            }
            if (ix->rows().slots) TV_HIP(tv::launch_map_slots(oi, size_t(a.nq_tile) * k_eff, ix->rows().slots, n, ix->stream));
        }
        TV_HIP(hipStreamSynchronize(ix->stream));
        for (size_t t = 0; timed_run && t < n_tiles && int(t) < kMaxTimedTiles; ++t) {
            float ms = 0.0f;
            TV_HIP(hipEventElapsedTime(&ms, ix->ev_start[t], ix->ev_stop[t]));
            ix->last_scan_ms += ms;
            ix->last_scan_launches += 1;
        }
    }
    return TV_OK;
}

// Block strides of the sampling ladder a first pass over cq queries runs (the last one is 1).  The
// all-queries-per-pass kernel works through the blocks in rounds of its grid, and its levels are
// trimmed to whole rounds.
//
// A first pass served by the single-tile permute-dot kernel (up to 32 queries), the all-queries
// kernel or the single-query byte-table LUT scan runs one sampling level only, without a floor:
// the scan hands over the best row of every block it reads (kModeBest), and the k_floor-th best
// of those is the floor of the full scan.  The level is sized so that the full scan then appends
// about 2048 rows per query (1024 on the all-queries kernel), and reads at least 8 * k_floor
// blocks; a quarter of the index or more is not worth sampling.
constexpr size_t kBestLevelMaxK = 64;
constexpr size_t kBestLevelMaxKLut = 128;   // (the single-query byte-table scan: configuration 3 asks for k = 100)
constexpr int kRowLadderSearches = 64;   // searches that keep to the row-level ladder after the floorless level failed
bool first_level_is_best_of_block(const tv_index *ix, const SampledPlan &plan, size_t k_floor) {
    if (ix->row_ladder_left != 0) return false;
    if (effective_mode(ix) != TV_SCORE_P) return plan.lut_single && k_floor <= kBestLevelMaxKLut;   // u8 LUT: the single-query byte-table scan has the mode
    if (k_floor > kBestLevelMaxK) return false;
    return plan.wide ? tv::wide_serves_best_of_block(ix->geo.nch) : plan.nt_batched == 0;
}
// The other kernels have no floorless mode -- a second epilogue does not fit their registers -- but the scans of the unsampled
// search keep every block's best score, and on a sample of the blocks those give a floor as good: one launch of
// them and k_floor_of_best instead of two row-level samples, their selections and the second one's conditional
// repeat.  On indexes of any size that the unsampled search does not take, as long as the sample holds k_floor blocks with a row
// that may be returned (us a search with the ladder, and so: 500K x 1536, 64 queries 175 and 137; 60K x 1536, 64 queries, k = 50 83
// and 66; 16K x 1536, k = 100 70 and 58; 100K x 1536, 1000 queries, k = 100 541 and 340; 500K x 3072, 100 queries 415 and 294; 20K x
// 1000 3-bit, 8 queries, k = 100 75 and 64; from fewer blocks floors stay open and queries are repeated: 20K x 640, 500 queries, k = 128).
// Large or filtered batches of the matrix-unit scan keep the row-level ladder: its floors cost them less than a sample of whole (block, tile)
// epilogues (889K x 920 2-bit, 640 queries: 1842 us with the ladder, 1884 without; 3M x 512 3-bit, 50 queries, 1 % allowed: 249 and 279).
bool first_level_is_best_words(const tv_index *ix, const SampledPlan &plan, size_t n_blocks, size_t k_floor, bool masked) {
    if (ix->row_ladder_left != 0 || k_floor > size_t(tv::kMaxPickK) || n_blocks < 4 || (ix->no_direct && n_blocks <= 16384)) return false;
    if (ix->allowed.in_place) return false;      // (the best-of-block scans read whole blocks)
    if (effective_mode(ix) == TV_SCORE_P) return tv::best_serves(ix->geo.nch) && (plan.wide || plan.nt_batched > 0);
    return effective_mode(ix) == TV_SCORE_L_U32 && !ix->no_lut16 && (!plan.lut_mx || (plan.cq_pad <= 160 && k_floor <= 64 && !masked));
}
// Rows per query the full scan then appends, about: a smaller sample against more appends, which weigh most on short rows
// and on the matrix-unit scan (3M x 128, 1000 queries: 256 rows 657 us a search, 512 741, 1024 888, without this level 1223;
// 1M x 1536, 64 queries: 212, 223, 204, 237; 3M x 384 2-bit, 141 queries: 878, 878, 958, 946).
size_t floor_rows(const tv_index *ix, const SampledPlan &plan) {
    return plan.lut_mx ? 512 : effective_mode(ix) == TV_SCORE_P && ix->geo.nch < 12 ? 256 : 1024;
}
// sure: of every `step` blocks in turn, sure / step hold a row the search may return, whatever its mask looks like.
SamplingSteps level_strides(const tv_index *ix, const SampledPlan &plan, size_t n_blocks, size_t sure, size_t k_floor, bool repeat, bool masked) {
    if (!repeat && first_level_is_best_of_block(ix, plan, k_floor)) {
        SamplingSteps steps;
        // (the all-queries kernel pays for every candidate of the full scan -- a tile with one in it
        // leaves the integer fast path -- and samples twice as many blocks for a floor that lets half
        // as many through: 10M x 1536, 1024 queries: two rounds of its grid instead of one, +0.12 ms
        // of sampling, -0.25 ms of scan)
        const size_t per = plan.wide ? 1024 : 2048;
        size_t sample = std::max<size_t>((n_blocks * k_floor + per - 1) / per, 8 * k_floor);
        sample = std::min<size_t>(sample, size_t(plan.grid) * (tv::kSegCap / 2));   // a workgroup's blocks fit its segment
        size_t step = sample ? n_blocks / sample : 0;
        if (plan.wide) {
            // the all-queries-per-pass kernel works through the blocks in rounds of its grid and a
            // level costs whole rounds: trimmed to whole rounds, at least one, and never spilling into another
            const size_t round = size_t(plan.grid) * tv::wide_blocks_per_workgroup(ix->geo.nch);
            if (sample > round) sample -= sample % round;
            step = sample >= round ? (n_blocks + sample - 1) / sample : n_blocks / sample;
        }
        if (sample * 4 <= n_blocks && step > 1) {
            steps.step[steps.count++] = uint32_t(step);
            steps.step[steps.count++] = 1;
            steps.best_first = true;
            return steps;
        }
        // (an index too small for that level -- it would read a quarter of it or more -- takes the
        // row-level ladder below: a full scan from open floors alone would append every row)
    }
    if (!repeat && first_level_is_best_words(ix, plan, n_blocks, k_floor, masked)) {
        SamplingSteps steps;
        const size_t sample = std::min<size_t>({std::max<size_t>(n_blocks * k_floor / floor_rows(ix, plan), 8 * k_floor), size_t(tv::kMaxFloorBlocks), n_blocks / 4,
                                                 plan.seg_stride * tv::kSegCap * 2});      // (the words lie in the candidates' place)
        const size_t step = (n_blocks + sample - 1) / sample;
        if (sure / step >= k_floor) {      // (fewer would leave the floor open)
            steps.step[steps.count++] = uint32_t(step);
            steps.step[steps.count++] = 1;
            steps.best_first = steps.best_words = true;
            return steps;
        }
    }
    // (the sixteen-query LUT scan works in rounds too: every wave of the grid carries two blocks through the row)
    return plan.wide    ? sampling_steps(n_blocks, k_floor, size_t(plan.grid) * tv::wide_blocks_per_workgroup(ix->geo.nch))
           : plan.lut_mx ? sampling_steps(n_blocks, k_floor, size_t(tv::mx_round_blocks(ix->device, plan.cq_pad)))
           : plan.lut16 ? sampling_steps(n_blocks, k_floor, size_t(plan.grid) * tv::lut16_blocks_per_workgroup(effective_mode(ix) == TV_SCORE_L_CLASSIC))
                        : sampling_steps(n_blocks, k_floor);
}
// ---- u8-LUT batches over large indexes: an int8 scan in front of the tables (tv_kernels3.hip: NEAR, tv_kernels7.hip) ----
// The index is passed over in stages, each spread over all of it: the int8 scan, the rows it leaves in from the tables, the
// k_floor-th best so far as the next stage's floor.  A stage is about as large as everything before it, whole rounds of the
// scan's grid, and its rows and masks fit kNearBytes.  The first floor comes from a sample of blocks on the matrix-unit scan.
constexpr size_t kNearBytes = size_t(1) << 30;
constexpr size_t kNearSample = 512;      // blocks
constexpr int kNearMaxStages = 32;
// ... and so many (block, query tile, chunk) triples of 2-bit codes (390K x 144, 636 queries, 480 000 triples, 459 and 220; 87K x 1536, 223,
// k = 86, 230 000: 271 and 242), and of 3-bit ones, whose one-hot products are half as many (430K x 256, 349 queries, 590 000: 225 and 282; 890K x 280, 129,
// 700 000: 272 and 284; 1.2M x 248, 319, 1.5e6: 705 and 329).
constexpr size_t kNearMinWork2 = 200000, kNearMinWork3 = 1200000;
// Rows that have to be looked up for nothing cost the rest: the share of an index within the margin of the last result (long rows,
// many results, few rows).  3072 dimensions 2-bit: 2.2M rows, 127 queries, k = 71, 1.1 % 2810 and 3623; 1.2M, 389 queries, k = 24, 0.8 % 4831
// and 4070; 3.8M, 437 queries, k = 21, 0.5 % 14 583 and 6371; 3-bit: 2M x 976, 373 queries, k = 91, 1 % 2859 and 2480; 3M x 760, 225 queries,
// k = 92, 0.5 % 2347 and 1271.
// Less of them where queries are few and the one-hot products cheap: 3-bit, 954K x 1536, 94 queries, k = 3, 0.5 % 681 and 839; 838K x 768, 177, k =
// 15, 0.3 % 477 and 537; 2.6M x 768, 175, k = 7, 0.1 % 1421 and 1060.
constexpr double kNearShare2 = 0.01, kNearShare3 = 0.008, kNearShareTile2 = 0.0025, kNearShareTile3 = 0.0005;
struct NearPlan {
    size_t stages = 0;                    // 0: the search does not go this way
    uint32_t groups[kNearMaxStages] = {};
    int rank[kNearMaxStages + 1] = {};    // the floor of the sample, and of each stage: the so-manieth best
    bool guessed = false;                 // ... of which k rows may fall short
    uint32_t total = 0, mul = 1, step = 1, splits = 1, sub = 1;
    size_t rows_bytes = 0, bytes = 0;     // of the largest stage
};
// A floor need not be one that k rows are sure to reach, if the end shows that k did: the r-th best of a share f of the rows is above the
// k-th best of all only where r or more of the k best are among them -- a Poisson variable of mean f * k.  The least r that is
// so with a chance of one in a million: 8 for k = 100 and a 150th of the rows, in place of 100.
int guessed_rank(double share, size_t k) {
    const double mean = share * double(k);
    double term = std::exp(-mean), below = term;
    int r = 1;
    for (; r < int(k) && 1.0 - below > 1e-6; ++r) below += term *= mean / r;
    return r;
}
// rows: those the search may return, in at least `sure` of the blocks.
NearPlan near_plan(const tv_index *ix, const SampledPlan &plan, size_t cq, size_t k_eff, size_t n_blocks, size_t rows, size_t sure) {
    NearPlan p;
    const size_t k_floor = std::max<size_t>(k_eff, 16);
    const int nch = ix->geo.nch, bits = ix->geo.bits;
    if (near_bytes(ix, cq) == 0 || ix->no_wide || ix->no_batched || ix->row_ladder_left != 0 || ix->allowed.in_place || k_floor > size_t(tv::kMaxPickK)) return p;
    if (tv::near_rescore_queries(nch) == 0 || ix->rows().n >= (size_t(1) << 31)) return p;
    const size_t round = size_t(plan.grid_near) * size_t(tv::near_blocks_per_workgroup(nch, bits)) / tv::kNearBlocks;      // groups
    const size_t total = (n_blocks + tv::kNearBlocks - 1) / tv::kNearBlocks, tiles = (cq + tv::kQTile - 1) / tv::kQTile;
    if (ix->no_direct && n_blocks <= 16384) return p;
    if (n_blocks < 4) return p;      // (a sample is a quarter of the blocks at most, and one at least)
    if (!ix->force_near && n_blocks * tiles * size_t(nch) < (bits == 2 ? kNearMinWork2 : kNearMinWork3)) return p;
    // how far above the int8 product a table sum may lie, in standard deviations of the score, about (measured at 128 to 3072 dimensions),
    // and the share of rows that close to the last result's score, were scores normal
    const double margin = (bits == 2 ? 0.028 : 0.045) * std::sqrt(double(ix->geo.dim));
    const double tail = std::log(double(rows) / double(2 * k_eff));
    double z = std::sqrt(2.0 * std::max(tail, 1.0));
    for (int i = 0; i < 2; ++i) z = std::sqrt(2.0 * std::max(tail - 0.919 - std::log(z), 0.5));
    if (!ix->force_near && 0.5 * std::erfc((z - margin) * 0.70710678) > (bits == 2 ? std::min(kNearShare2, kNearShareTile2 * double(tiles)) : std::min(kNearShare3, kNearShareTile3 * double(tiles)))) return p;
    const size_t group_rows = size_t(tv::kNearBlocks) * ix->geo.block_bytes(), group_masks = tiles * tv::kQTile * tv::kNearBlocks * 4;
    const size_t most = std::max(round, kNearBytes / (group_rows + group_masks) / round * round);
    const size_t per_group = size_t(tv::near_rescore_queries(nch)), query_groups = (cq + per_group - 1) / per_group;
    // workgroups of the rescore: up to two a CU at once, and none that wait for a place among those (us a search rounded up and so, all 2-bit: 4M x 256, 800
    // queries 1338 and 1254, 3M x 384, 500 944 and 871, 2M x 768, 300 842 and 794, 2M x 1536, 500 1926 and 1906; the one the other way 1.5M x 1536, 200, k = 50, 975 and 990)
    p.splits = uint32_t(std::clamp<size_t>(std::max((6 * k_floor + tv::kSegCap - 1) / tv::kSegCap, 512 / query_groups), 4, 16));
    p.guessed = ix->near_sure_left == 0;
    const size_t sample = std::min<size_t>({p.guessed ? std::max<size_t>(kNearSample, size_t(tv::mx_round_blocks(ix->device, cq))) : std::max({4 * kNearSample, 8 * k_floor, round * tv::kNearBlocks / 2}),
                                            size_t(tv::kMaxFloorBlocks), n_blocks / 4});
    p.step = uint32_t((n_blocks + sample - 1) / sample);
    auto rank_of = [&](double share) { return p.guessed ? guessed_rank(share, k_eff) : int(k_floor); };
    p.rank[0] = rank_of(1.0 / double(p.step));
    if (sure / p.step < 2 * size_t(p.rank[0])) return p;
    size_t seen = sample / tv::kNearBlocks, largest = 0;
    const double grow = p.guessed ? (margin < 0.9 ? 6.0 : margin < 1.15 ? 4.0 : 2.0) : 2.0;
    for (size_t done = 0; done < total;) {
        const size_t left = total - done;
        size_t g = std::min(most, std::max<size_t>(1, size_t(double(seen) * (grow - 1.0) / double(round) + 0.5)) * round);
        if (left <= most && left <= g + g / 2) g = left;
        else if (left < 2 * g) g = std::min(g, (left / 2 + round - 1) / round * round);
        g = std::min(g, left);
        if (p.stages == size_t(kNearMaxStages) || (p.stages + 1) * p.splits > plan.seg_stride) { p.stages = 0; return p; }
        p.groups[p.stages++] = uint32_t(g);
        largest = std::max(largest, g);
        done += g;
        seen += g;
        p.rank[p.stages] = rank_of(double(done) / double(total));
    }
    while (p.sub < 8 && p.stages * p.splits * p.sub * 2 <= plan.seg_stride) p.sub *= 2;      // (room for neighbours that lie together)
    p.total = uint32_t(total);
    // (consecutive multiples of the golden section of the total, modulo it, lie evenly over it; coprime, so that each group comes up once)
    auto gcd = [](size_t a, size_t b) { while (b) { const size_t t = a % b; a = b; b = t; } return a; };
    size_t mul = std::max<size_t>(1, size_t(double(total) * 0.6180339887498949));
    while (gcd(mul, total) != 1) ++mul;
    p.mul = uint32_t(mul % total);
    p.rows_bytes = round_up(largest * group_rows, 256);
    p.bytes = p.rows_bytes + largest * group_masks;
    return p;
}
// rows: those of the n_blocks blocks that the search may return.
bool near_takes(const tv_index *ix, size_t nq, size_t k_eff, size_t n_blocks, size_t rows) {
    const size_t cq = chunk_len(ix, nq);
    return near_plan(ix, sampled_plan(ix, cq), cq, k_eff, n_blocks, rows, rows / tv::kVecBlock).stages > 0;
}
// Block offset of a repeated pass's level of stride `step`: it samples other blocks than the pass
// that misjudged the floor, half a stride in (an even number of blocks, so that mask words stay
// aligned).
uint32_t repeat_offset(uint32_t step) { return step >= 4 ? (step / 2) & ~1u : 0u; }

// ---- small indexes: no sampling (tv_kernels6.hip) ----
constexpr size_t kDirectWideBlocks = 20480;

// Which scan the search of nq queries without sampling takes: the all-queries kernel keeps a decoded block
// for all of them, from where its grid of eight waves per CU has blocks to hold (157 blocks of 1536
// dimensions, 1000 queries: 126 us a search against 103; 938: 149 against 179).
bool direct_wide(const tv_index *ix, size_t nq, size_t n_blocks) {
    const int nch = ix->geo.nch;
    return tv::wide_min_queries(nch) > 0 && nq >= size_t(tv::wide_min_queries(nch)) && tv::wide_serves_best_of_block(nch) && n_blocks > 512;
}
// Whether the scan of that search keeps every row's score: few rows, on the kernel that can, and memory of the index's own.  A score per
// row and query against whole blocks scored again (us a search, blocks and rows): 2000 x 3072, 1024 queries 129 and 63, k = 1 71 and 62; 4096 x
// 1536, 300 queries 61 and 39, 8 queries, k = 100 69 and 35; 4000 x 384, 1024 queries 42.4 and 41.8, x 256 38.3 and 40.8, x 128
// 34.5 and 39.8, k = 50 49 and 44; 2000 x 128 32.6 and 33.5, 1000 x 128 32.2 and 31.0; 4000 x 128, one query 27.9 and 24.4, 128 queries 28.9 and 26.6.
bool direct_rows(const tv_index *ix, size_t nq, size_t n_blocks, size_t k_eff) {
    const size_t rows = n_blocks * tv::kVecBlock;
    return !ix->ws_fixed && effective_mode(ix) == TV_SCORE_P && rows <= tv::kMaxPickRows && !direct_wide(ix, nq, n_blocks) &&
           (nq <= 256 || rows <= 75 * k_eff * size_t(ix->geo.nch));
}
// (a fixed scratch array has no room set aside for it)
int direct_shares(const tv_index *ix, size_t cq, size_t k_eff) {
    return ix->ws_fixed ? 1 : tv::pick_shares(ix->device, ix->geo.nch, k_eff, cq, effective_mode(ix) != TV_SCORE_P);
}
// (enough for a call's shorter last chunk too, which may keep rows' scores, or share, where the others do not)
size_t direct_need(const tv_index *ix, size_t cq, size_t n_blocks, size_t k_eff) {
    const size_t sharing = std::min(cq, size_t(tv::device_cus(ix->device)) / 2);
    return prepare_bytes(ix, cq) + round_up(cq * round_up(n_blocks, 64) * (direct_rows(ix, 1, n_blocks, k_eff) ? tv::kVecBlock : 1) * sizeof(uint32_t), 256) +
           (direct_shares(ix, 1, k_eff) > 1 ? round_up(tv::pick_shared_bytes(k_eff, sharing), 256) : 0) + 65536;
}
// Where the search without sampling is the faster one.  Device buffers, k = 10, us a search, each pair
// without sampling and with it: 100K x 128, 1 query 30 and 45, 64 queries 32 and 61, 1000 queries 67 and 493; x 64, 5 queries
// 29 and 45 (1.04M: 45 and 59); 260K x 768, 32 queries 54 and 71; 100K x 1536, 1000 queries 246 and 304.
//  - It scores k blocks a second time: in one workgroup k = 100 at 768 dimensions (12 chunks) costs one
//    query 77 us against 64, at 128 dimensions 40 against 72; in up to eight of them, where queries are few (pick_shares), 20K rows x 768
//    41.5 and 57.2, 400K 64 and 105, 100K x 3072 92 and 137, 32 queries over 100K x 1536 74 and 106; but 60 queries over 100K x 1024 73 and 63.
//  - k_pick keeps a word per block in registers: 32768 blocks at most (twice that spills: 2M x 128, one query
//    121 and 77).
//  - One tile of queries: a full scan of so many bytes that two more launches no longer show.  1.04M rows x 128
//    51 and 63, x 512 80 and 92, x 640 99 and 101, x 768 113 and 115, x 1024 140 and 140; 600K x 1024 95 and 105, x 1536 132 and 131.
//  - More tiles on k_scan_p4_best, which decodes a block once per tile group: won up to a number of (block,
//    tile, chunk) triples that depends on the kernel it replaces -- rows whose tiles
//    stay in LDS and that this kernel too keeps two tiles of (1.04M x 1024, 64 queries, 1.04e6: 172 and 193) or only one (100K x 1536,
//    100 queries, 3e5: 100 and 99; 600K x 1536, 64 queries, 9e5: 211 and 185), rows whose tiles are streamed (260K x 3072, 100 queries, 1.6e6:
//    308 and 528; 500K, 3e6: 489 and 437).
//  - Rows of 3 to 11 chunks: this kernel decodes a block once for every four tiles and scores k blocks a query again, the all-queries kernel decodes it
//    once for all tiles, but needs a sample's floors first and takes whole rounds of blocks.  By 22 000 searches both ways (3 to 10 chunks, 129 to 1024 queries, 4200 to
//    1.04M rows, k = 1 to 120, Gaussian and clustered), in the time of one (block, chunk) pair decoded once more, about 0.1 ns: a block scored again 176 a
//    chunk for every 256 queries, which is one a CU; the floors 160 000 and 4000 a tile; a place of the last round that no block takes, a quarter a chunk and tile.  0.6 % off the
//    faster way on the mean, 4.8 % of the searches by more than 4 %; without the second and the last of these 1.2 % and 8.4 %.  k = 10:
//    491K x 176, 182 queries 70 and 83; 164K x 616, 562 137 and 147; 130K x 264, 964 99 and 133; 864K x 608, 329 302 and 273; 638K x 488, 505 246 and 221.  More
//    results: 729K x 136, 397, k = 59 193 and 174; 389K x 368, 928, k = 75 319 and 255; 319K x 168, 387, k = 100 116 and 131, k = 33 98 and 114.
//    Of one or two chunks: 1M x 128, 300 queries 128 and 135, 1000 296 and 283, 750K x 64, 1000 237 and 402.  Up to four tiles the other
//    kernel is k_scan_p4_multi: 100 queries 1M x 256 86 and 98, x 640 143 and 137.
//  - On the all-queries kernel its epilogue over every pair costs as much as sampling saves at about 700K
//    rows (1000 queries: 600K x 768 570 and 621, x 1536 972 and 999; 1.04M x 768 935 and 895, x 1536 1611 and 1523),
//    earlier where many rows are scored again (500K x 768, k = 45: 556 and 540).
// The same for u8-LUT queries with the u32 epilogue.  k = 10, us a search without sampling and with it, 2 bits: 100K x 128, 1 query
// 32 and 42, 12 queries 42 and 62, 100 queries 61 and 96; 400K x 64, 100 queries 84 and 146; 400K x 512, 4 queries 52 and 86; 20K x 1536,
// 100 queries 89 and 164; 1M x 1536, 12 queries 198 and 236.
//  - Rows are scored a second time at two table reads a byte: 100 blocks of 12 chunks take 50 us (400K x 768 3-bit, one
//    query, k = 60: 95 and 85; 60K x 1536, 8 queries, k = 100: 99 and 97; 400K: 133 and 138; 64 queries: 147 and
//    177; 60K, 400 queries: 309 and 285) in one workgroup; shared, one query, k = 100: 100K x 768 44 and 53, 400K x 1536 76 and 86; 60 queries
//    over 100K x 1536 3-bit 117 and 174, 100 over 100K x 768 3-bit, k = 100 112 either way.  One query over up to 64 blocks would be scanned once, without a level in front (1000 rows x
//    512 34 and 40; x 1536 49 and 50; x 1024 3-bit 54.3 and 53.6; x 3072 71 and 66, k = 1 65.7 and 65.3).
//  - The matrix-unit scan pays its epilogue on every (block, tile) pair: 400K x 1536, 500 queries (200K pairs) 983 and 1038, 1M x
//    512 (500K pairs) 1060 and 955.
constexpr size_t kSharedMost = 6000;      // (k times the chunks of a row, shared by eight: 100K x 3072, k = 100 is 4800)
bool direct_serves_lut(const tv_index *ix, size_t nq, size_t k_eff, size_t n_blocks, bool masked) {
    const size_t nch = size_t(ix->geo.nch), rescored = k_eff * nch, tiles = (std::min(nq, kChunkQueries) + tv::kQTile - 1) / tv::kQTile;
    if (effective_mode(ix) != TV_SCORE_L_U32 || ix->no_lut16 || tv::pick_lds_bytes(int(nch), k_eff, true) > tv::kPickLds) return false;
    const size_t shares = size_t(direct_shares(ix, nq, k_eff));
    if (nq == 1) return rescored <= (n_blocks > 64 ? (shares > 1 ? kSharedMost : 400u) : nch <= 16 ? 120u : 0u);
    if (nq <= size_t(tv::kLut16Queries)) return rescored <= (n_blocks >= 4096 ? 1200u : 720u);
    // (the two-step scan, whose stages cost some 80 us at least, from so many triples: 560K x 1536, 287 queries, 1.9e6 875 and 546; 180K x 1024,
    // 389, 6e5 299 and 239; 720K x 768, 188, 8e5 369 and 352; 530K x 384, 273, 4.5e5 296 and
    // 262, 130K x 512, 870, 4.5e5 258 and 207, 120K x 1024, 481, 4.8e5 270 and 241, 460K x 1536, 87, 5.2e5 308 and 288, 98K x 1536, 472, 5.5e5 284 and 294, 99K x 768, 890, 5.2e5 264 and 292; but 116K x 1536, 298, 4.4e5 241 and 264, 650K x 384, 168,
    // 3.7e5 222 and 249, 280K x 664, 155, 2.6e5 170 and 193; longer rows: 140K x 2048, 621, 1.4e6 610 and 642)
    if (!masked && ix->geo.bits == 2 && nch <= 12 && tiles >= 3 && n_blocks * tiles * nch >= (nch <= 8 && n_blocks >= 3500 ? 450000u : 600000u) && near_takes(ix, nq, k_eff, n_blocks, n_blocks * tv::kVecBlock)) return false;
    return n_blocks * tiles <= 200000 && rescored <= std::max<size_t>(tiles <= 4 ? 1200u : 600u, 600u * shares);
}
bool direct_serves(const tv_index *ix, size_t nq, size_t k_eff, size_t n_blocks, bool masked) {
    const int nch = ix->geo.nch;
    if (ix->force_robust || ix->no_batched || ix->no_wide || ix->no_direct || ix->force_near) return false;
    if (k_eff > size_t(tv::kMaxPickK) || n_blocks > tv::kMaxPickBlocks) return false;
    const size_t cq = chunk_len(ix, nq), tiles = (cq + tv::kQTile - 1) / tv::kQTile, triples = n_blocks * tiles * nch;
    if (ix->ws_fixed && direct_need(ix, cq, n_blocks, k_eff) > ix->ws_bytes) return false;
    if (effective_mode(ix) != TV_SCORE_P) return direct_serves_lut(ix, nq, k_eff, n_blocks, masked);
    if (!tv::best_serves(nch)) return false;
    // (no block is scored again where rows' scores are kept)
    if (!direct_rows(ix, cq, n_blocks, k_eff) &&
        (k_eff * nch > (tiles == 1 && direct_shares(ix, nq, k_eff) > 1 ? kSharedMost : 600u) || tv::pick_lds_bytes(nch, k_eff, false) > tv::kPickLds)) return false;
    if (direct_wide(ix, cq, n_blocks)) return n_blocks <= (k_eff * nch <= 300 ? kDirectWideBlocks : kDirectWideBlocks / 2);
    if (tiles == 1) return n_blocks <= (nch <= 24 ? 16384u : 8192u) || triples <= 327680;
    if (nch <= 2) return true;
    if (nch < 12) {
        const size_t round = size_t(tv::wide_grid_blocks(ix->device)) * size_t(tv::wide_blocks_per_workgroup(nch)), empty = (n_blocks + round - 1) / round * round - n_blocks;
        const size_t again = direct_rows(ix, cq, n_blocks, k_eff) ? 0 : 176 * k_eff * ((cq + 255) / 256);
        return (n_blocks * ((tiles + 3) / 4 - 1) + again) * size_t(nch) <= 160000 + 4000 * tiles + empty * tiles * size_t(nch) / 4;
    }
    return triples <= (!tv::batched_weights_split(nch) ? 1600000 : nch <= 16 ? 1050000 : 250000) || n_blocks <= 512;
}
// The best score of every scanned block for u8-LUT queries, on the kernel that serves so many in a full scan: byte tables for one,
// whole tables in LDS for a few, tables streamed for up to sixteen (tiles side by side beyond) or the
// sparse matrix instruction; a few queries over few blocks with each block's chunks on several waves (tv_kernels8.hip).
int best_scan_lut(tv_index *ix, tv::ScanArgs a, const Prepared &pq, size_t cq) {
    const int nch = a.nch;
    const size_t blocks = (a.n_blocks + a.b_step - 1) / a.b_step;
    a.k = 1;
    a.gtau = ix->d_tau_open;
    if (pq.d_tables_mx != nullptr) {
        a.tables = pq.d_tables_mx;
        if (a.mask) TV_HIP(tv::launch_fill_i32(reinterpret_cast<int *>(a.best_out), 0, cq * a.best_stride, ix->stream));   // (it skips blocks without an allowed row)
        TV_HIP(tv::launch_scan_lut_mx(a, tv::mx_shape(ix->device, cq, blocks, false), ix->geo.bits, ix->stream));
    } else if (pq.d_tables16 != nullptr) {
        a.tables = pq.d_tables16;
        const int tiles = int((cq + tv::kLut16Queries - 1) / tv::kLut16Queries);
        const int grid = int(std::min<size_t>(size_t(tv::device_cus(ix->device)), (blocks + 7) / 8));
        TV_HIP(tv::launch_scan_lut16(a, grid, tiles, ix->stream));
    } else if (const int parts = a.classic == 0 ? tv::lut_parts(nch, int(cq), blocks, tv::device_cus(ix->device)) : 1; parts > 1) {
        TV_HIP(tv::launch_scan_lut_parts(a, parts, ix->device, ix->stream));
    } else {
        const int grid = int(std::min<size_t>(size_t(tv::lut_append_grid(ix->device, nch)), (blocks + 1) / 2));
        TV_HIP(tv::launch_scan_lut(a, grid, tv::kModeAppend, ix->stream));
    }
    return TV_OK;
}
// The milliseconds between the two stamps.
int take_stamps(tv_index *ix, int launches) {
    int khz = 0;
    TV_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, ix->device));
    const uint64_t before = *std::max_element(ix->h_stamps, ix->h_stamps + tv::kStampsBefore);      // (those of earlier searches are lower)
    if (khz > 0) ix->last_scan_ms += float(double(ix->h_stamps[tv::kStampsBefore] - before) / khz);
    ix->last_scan_launches += launches;
    return TV_OK;
}
int search_direct(tv_index *ix, const float *d_queries, size_t nq, size_t k_eff, const uint64_t *d_mask, float *d_out_scores,
                  int64_t *d_out_idx, bool timing) {
    const tv::Geometry &g = ix->geo;
    const size_t n_blocks = (ix->rows().n + tv::kVecBlock - 1) / tv::kVecBlock, stride = round_up(n_blocks, 64);
    int rc = ensure_workspace(ix, direct_need(ix, chunk_len(ix, nq), n_blocks, k_eff));
    if (rc != TV_OK) return rc;
    ix->last_queries_per_launch = int(chunk_len(ix, nq));
    if (effective_mode(ix) != TV_SCORE_P && !lut_mx_serves(ix, chunk_len(ix, nq)))
        ix->last_queries_per_launch = std::min(ix->last_queries_per_launch, tv::kLut16Queries);     // (a pass serves so many; passes share a launch)
    for (size_t g0 = 0; g0 < nq; g0 += kGroupQueries) {
        const size_t gq = std::min(kGroupQueries, nq - g0);
        for (size_t c0 = 0, cq; c0 < gq; c0 += cq) {
            cq = chunk_len(ix, gq - c0);
            const size_t q0 = g0 + c0;
            const bool mode_p = effective_mode(ix) == TV_SCORE_P, timed = timing && q0 == 0;
            const bool wide = mode_p && direct_wide(ix, cq, n_blocks), split = wide && tv::wide_weights_split(g.nch);
            Arena ar;
            ar.base = static_cast<uint8_t *>(ix->ws);
            Prepared pq;
            const int shares = direct_rows(ix, cq, n_blocks, k_eff) ? 1 : direct_shares(ix, cq, k_eff);
            uint64_t *shared = shares > 1 ? ar.take<uint64_t>(tv::pick_shared_bytes(k_eff, cq) / sizeof(uint64_t)) : nullptr;
            const bool parts = effective_mode(ix) == TV_SCORE_L_U32 && !lut_mx_serves(ix, cq) && tv::lut_parts(g.nch, int(cq), n_blocks, tv::device_cus(ix->device)) > 1;
            rc = prepare_queries(ix, ar, d_queries + q0 * g.dim, cq, pq, split, false, !parts, timed ? ix->d_stamps : nullptr, shared);
            if (rc != TV_OK) return rc;
            tv::ScanArgs a;
            fill_scan_args(ix, a);
            a.mask = d_mask;
            a.tables = pq.d_tables;
            a.qscale = pq.d_qscale;
            a.qbias = pq.d_qbias;
            a.nq_tile = int(cq);
            a.best_rows = direct_rows(ix, cq, n_blocks, k_eff) ? 1 : 0;
            a.best_stride = uint32_t(stride * (a.best_rows ? tv::kVecBlock : 1));
            a.best_out = ar.take<uint32_t>(cq * a.best_stride);
            if (wide) {
                a.gtau = ix->d_tau_open;
                a.best_of_block = 1;
                if (d_mask) TV_HIP(tv::launch_fill_i32(reinterpret_cast<int *>(a.best_out), 0, cq * stride, ix->stream));   // (it skips blocks without an allowed row)
                TV_HIP(tv::launch_scan_p4_wide(a, tv::wide_grid_blocks(ix->device), ix->stream));
            } else if (mode_p) {
                TV_HIP(tv::launch_scan_p4_best(a, split, ix->device, ix->stream));
            } else {
                rc = best_scan_lut(ix, a, pq, cq);
                if (rc != TV_OK) return rc;
            }
            if (a.best_rows)
                TV_HIP(tv::launch_pick_rows(reinterpret_cast<const float *>(a.best_out), a.best_stride, a.n, int(k_eff), int(cq), d_out_scores + q0 * k_eff,
                                            d_out_idx + q0 * k_eff, ix->rows().slots, ix->d_flags_host + c0, timed ? ix->d_stamps + tv::kStampsBefore : nullptr, ix->stream));
            else TV_HIP(tv::launch_pick(a, !mode_p, split, int(k_eff), d_out_scores + q0 * k_eff, d_out_idx + q0 * k_eff, ix->rows().slots, ix->d_flags_host + c0,
                                   shares, shared, timed ? ix->d_stamps + tv::kStampsBefore : nullptr, ix->stream));
        }
        TV_HIP(hipStreamSynchronize(ix->stream));
        if (timing && g0 == 0) {
            rc = take_stamps(ix, 1);
            if (rc != TV_OK) return rc;
        }
        // (fewer rows than wanted had a score: a mask of fewer rows than the caller's count promised)
        std::vector<uint32_t> exact_rows;
        for (size_t q = 0; q < gq; ++q)
            if (ix->h_flags[q] != 0u) exact_rows.push_back(uint32_t(q));
        ix->overflow_redos += exact_rows.size();
        ix->exact_redos += exact_rows.size();
        for (const uint32_t row : exact_rows) {
            const size_t q = g0 + row;
            rc = search_robust(ix, d_queries + q * g.dim, 1, k_eff, d_mask, d_out_scores + q * k_eff, d_out_idx + q * k_eff, false);
            if (rc != TV_OK) return rc;
        }
    }
    return TV_OK;
}

int leave_in_place(tv_index *ix, size_t nq, size_t k_eff);
constexpr size_t kLiveUnknown = ~size_t(0);

// The seam: search::search over device-resident inputs and outputs.
//
// Sample-then-filter.  Scans run in append mode: every allowed slot whose score
// reaches the query's floor is appended to a small per-query buffer, and a sort
// of that buffer yields either the next floor (sampling levels) or the answer
// (the full scan).  A floor is the k-th best score among slots actually
// scanned, hence a lower bound of the true k-th best, so the full scan appends
// every member of the true top-k; ties at the floor are kept (>=) and resolved
// by the same total order as everywhere else.
//
// Where ix->allowed has the rows `d_mask` allows, those are searched and the mask is not read -- but for queries
// whose candidates did not fit in a scan of rows in place, which alone are repeated with it (or on a copy).  live: the
// blocks of the index with a row that the mask allows, or kLiveUnknown.
int search_rows(tv_index *ix, const float *d_queries, size_t nq, size_t k, const uint64_t *d_mask,
                size_t n_allowed, size_t live, float *d_out_scores, int64_t *d_out_idx, size_t *out_k_eff) {
    const size_t n = ix->rows().n;
    // (counted blocks may lie anywhere: half of a sample's share of them; rows of a mask nobody has looked at: the fewest blocks that hold so many)
    const size_t sure = live != kLiveUnknown ? live / 2 : n_allowed / tv::kVecBlock;
    const uint64_t *mask = ix->allowed.codes ? nullptr : d_mask;
    size_t k_eff = std::min(std::min(k, n), n_allowed);  // lib.rs:1460, search.rs:3222-3225
    if (out_k_eff) *out_k_eff = k_eff;
    ix->last_scan_ms = 0.0f;
    ix->last_scan_launches = 0;
    if (k_eff == 0 || nq == 0) return TV_OK;                // search.rs:3226-3229
    if (n >= (size_t(1) << 31)) { g_last_error = "index too large for 31-bit slots"; return TV_ERR_BAD_ARGUMENT; }
    const tv::Geometry &g = ix->geo;
    const int mode = effective_mode(ix);
    if (mode == TV_SCORE_P && g.bits != 4) { g_last_error = "score mode P needs 4-bit codes"; return TV_ERR_BAD_ARGUMENT; }
    const bool mode_p = mode == TV_SCORE_P;
    // a search on a lent, fixed workspace (tv_search_dev_noalloc) creates nothing, event pool included
    const bool timing = !ix->ws_fixed;
    int rc = timing ? ensure_events(ix) : TV_OK;
    if (rc != TV_OK) return rc;
    if (k_eff > size_t(tv::kMaxSampledK) || ix->force_robust)
        return search_robust(ix, d_queries, nq, k_eff, mask, d_out_scores, d_out_idx, timing);

    size_t n_blocks = (n + tv::kVecBlock - 1) / tv::kVecBlock;
    if (direct_serves(ix, nq, k_eff, n_blocks, mask != nullptr)) return search_direct(ix, d_queries, nq, k_eff, mask, d_out_scores, d_out_idx, timing);
    // sampling levels take the k_floor-th best as the floor: a deeper order statistic is steadier
    const size_t k_floor = std::max<size_t>(k_eff, 16);
    if (ix->row_ladder_left > 0) --ix->row_ladder_left;
    if (ix->floorless_kept_left > 0) --ix->floorless_kept_left;
    if (ix->near_sure_left > 0) --ix->near_sure_left;
    uint32_t *h_over = ix->h_flags;   // pinned, one flag per query of a group, then the groups' level flags
    const bool track_levels = ix->track_levels != 0;
    // sized once for the whole call, repeated passes included: nothing is reallocated while work is in flight
    rc = ensure_workspace(ix, sampled_need_worst(ix, nq));
    if (rc != TV_OK) return rc;

    auto near_of = [&](const SampledPlan &plan, size_t cq) {
        return near_plan(ix, plan, cq, k_eff, n_blocks, mask ? n_allowed : ix->rows().n, mask ? sure : n_blocks);
    };
    // The two-step table scan's stages: memory that nothing is given up for; without it the first passes take the matrix-unit scan alone.
    struct Staged {
        tv_index *ix;
        tv_spare *there = nullptr;
        bool idle = true;      // (an error may leave launches that still use it)
        ~Staged() {
            if (there && !idle) (void)hipStreamSynchronize(ix->stream);
            if (there) staged_give(ix->device, there);
        }
    } staged{ix};
    {
        size_t bytes = 0;
        for (const size_t cq : {std::min(nq, kChunkQueries), nq % kChunkQueries})      // (a chunk, and the last one)
            if (cq != 0 && mode != TV_SCORE_P) bytes = std::max(bytes, near_of(sampled_plan(ix, cq), cq).bytes);
        if (bytes > 0) staged.there = staged_take(ix->device, bytes);
    }

    // (which rows a scan reads, and through which mask, changes between a group's first passes and its repeated ones)
    const tv_rows asked = ix->allowed;
    auto read = [&](const tv_rows &rows) {
        ix->allowed = rows;
        mask = rows.codes ? nullptr : d_mask;
        n_blocks = (ix->rows().n + tv::kVecBlock - 1) / tv::kVecBlock;
    };
    bool left_in_place = false;
    for (size_t g0 = 0; g0 < nq; g0 += kGroupQueries) {
        const size_t gq = std::min(kGroupQueries, nq - g0);
        if (left_in_place && !ix->allowed.codes) read(asked);      // (a copy, once made, serves the rest of the call)
        Arena head;
        head.base = static_cast<uint8_t *>(ix->ws);
        int *d_raise = head.take<int>(gq);
        // The overflow flags of the first passes are written by k_final straight into the pinned
        // host array (device-visible): no copy kernel between the last selection and the host's read.
        uint32_t *d_over_all = ix->d_flags_host;
        head.take<uint32_t>(gq);
        uint32_t *d_rows = head.take<uint32_t>(std::min(gq, kWideChunkQueries));
        float *d_redo_q = head.take<float>(std::min(gq, kWideChunkQueries) * g.dim);
        // the group's chunks: (first query, relative to the group; length)
        size_t chunk_at[kGroupQueries / kChunkQueries + 1], n_chunks = 0;
        for (size_t c0 = 0; c0 < gq; c0 += chunk_len(ix, gq - c0)) chunk_at[n_chunks++] = c0;
        chunk_at[n_chunks] = gq;
        uint32_t *d_level_flags_all = head.take<uint32_t>(kLevelFlagWords);
        size_t n_timed = 0;
        bool stamped = false;      // the full scan lies between two stamps (there is a level before it), not between events

        // One pass over `pq_n` queries of the chunk at q0: the ladder from open floors, or, for the
        // packed batch of queries to repeat (rows d_rows[row0 ..]), the ladder again from the floors
        // the pass before raised for them.  Enqueues only; the caller synchronises.
        auto pass = [&](size_t q0, size_t row0, size_t pq_n, bool repeat, bool timed_pass, size_t chunk_no) -> int {
            const float *d_q = d_queries + q0 * g.dim;
            float *d_os = d_out_scores + q0 * k_eff;
            int64_t *d_oi = d_out_idx + q0 * k_eff;
            const SampledPlan plan = sampled_plan(ix, pq_n);
            const size_t tile_q = plan.tile_q, n_tiles = plan.n_tiles, cq_pad = plan.cq_pad, seg_stride = plan.seg_stride;
            const bool wide = plan.wide;
            const int grid = plan.grid;
            const SamplingSteps steps = level_strides(ix, plan, n_blocks, mask ? sure : n_blocks, k_floor, repeat, mask != nullptr);
            const bool best_first = steps.best_first;
            NearPlan near = repeat || !staged.there ? NearPlan{} : near_of(plan, pq_n);
            if (near.stages > 0 && near.bytes > staged.there->bytes) near = NearPlan{};      // (a group before this one changed the plan)
            uint32_t *d_level_flags = d_level_flags_all + chunk_no * SamplingSteps::kMax;
            if (head.used + plan.need > ix->ws_bytes) {
                g_last_error = "internal: workspace smaller than the pass it was sized for";
                return TV_ERR_BAD_ARGUMENT;
            }
            Arena ar;
            ar.base = static_cast<uint8_t *>(ix->ws) + head.used;
            int *d_tau = ar.take<int>(n_tiles * tv::kQTile);
            if (repeat) {
                TV_HIP(tv::launch_gather_redo(d_q, d_rows + row0, d_raise + (q0 - g0), g.dim, int(tile_q), pq_n, d_redo_q, d_tau,
                                              ix->stream));
                // every level of a repeated pass filters by a floor: all of their flags start at zero
                TV_HIP(tv::launch_fill_i32(reinterpret_cast<int *>(d_level_flags), 0, SamplingSteps::kMax, ix->stream));
            }
            Prepared pq;
            const int nt_batched = plan.nt_batched;
            const bool split = wide ? tv::wide_weights_split(g.nch) : (nt_batched == 0 || tv::batched_weights_split(g.nch));
            int prc = prepare_queries(ix, ar, repeat ? d_redo_q : d_q, pq_n, pq, split, false, true, nullptr, nullptr, near.stages > 0);
            if (prc != TV_OK) return prc;
            uint64_t *d_cand = ar.take<uint64_t>(cq_pad * seg_stride * tv::kSegCap);
            uint32_t *d_cnt = ar.take<uint32_t>(cq_pad * seg_stride);
            uint32_t *d_over = repeat ? ar.take<uint32_t>(cq_pad) : d_over_all + (q0 - g0);
            // no per-search clears: the first level reads the index's standing array of open floors,
            // every later one the floors k_final wrote, and k_final writes every overflow flag

            const int bgrid = tv::batched_grid_blocks(ix->device, g.nch);
            const bool batched = nt_batched > 0 && !wide;
            const size_t tiles_per_launch = wide || plan.lut_mx ? n_tiles : batched ? size_t(nt_batched) : 1;
            if (!repeat && q0 == 0) ix->last_queries_per_launch = int(std::min(pq_n, tile_q * tiles_per_launch));   // the call's first chunk
            // The floors of a sample's best words (in the candidates' place, which nothing has been written to yet: 512 bytes a segment
            // against four a block).
            auto floors_of_best = [&](uint32_t step, int rank) -> int {
                const size_t level_blocks = (n_blocks + step - 1) / step;
                tv::ScanArgs a;
                fill_scan_args(ix, a);
                a.mask = mask;
                a.tables = pq.d_tables;
                a.qscale = pq.d_qscale;
                a.qbias = pq.d_qbias;
                a.nq_tile = int(pq_n);
                a.b_step = step;
                a.best_out = reinterpret_cast<uint32_t *>(d_cand);
                a.best_stride = uint32_t(round_up(level_blocks, 64));
                if (a.best_stride > seg_stride * tv::kSegCap * 2) { g_last_error = "internal: a sample larger than the candidates' place"; return TV_ERR_BAD_ARGUMENT; }
                if (mode_p) TV_HIP(tv::launch_scan_p4_best(a, split, ix->device, ix->stream));
                else if (const int lrc = best_scan_lut(ix, a, pq, pq_n)) return lrc;
                TV_HIP(tv::launch_floor(a.best_out, a.best_stride, uint32_t(level_blocks), rank, int(pq_n), d_tau, int(tile_q),
                                        timed_pass ? ix->d_stamps : nullptr, ix->stream));
                return TV_OK;
            };
            if (near.stages > 0) {
                staged.idle = false;
                if (const int frc = floors_of_best(near.step, near.rank[0])) return frc;
                tv::ScanArgs a;
                fill_scan_args(ix, a);
                a.mask = mask;
                a.tables = pq.d_near;
                std::memcpy(a.lv, ix->near_levels, sizeof ix->near_levels);
                a.qscale = pq.d_qscale;
                a.qbias = pq.d_qbias;
                a.near_unit = pq.d_near_unit;
                a.near_err = pq.d_near_err;
                a.nq_tile = int(pq_n);
                a.gtau = d_tau;
                a.near = tv::NearStage{0, 0, near.total, near.mul, reinterpret_cast<uint16_t *>(static_cast<uint8_t *>(staged.there->p) + near.rows_bytes), static_cast<uint8_t *>(staged.there->p)};
                tv::NearRescore r{};
                r.tables = pq.d_tables;
                r.scales = a.scales;
                r.qscale = pq.d_qscale;
                r.qbias = pq.d_qbias;
                r.gtau = d_tau;
                r.cand = d_cand;
                r.cand_cnt = d_cnt;
                r.seg_stride = uint32_t(seg_stride);
                r.splits = near.splits;
                r.sub = near.sub;
                r.n = a.n;
                r.nq = int(pq_n);
                r.nch = g.nch;
                for (size_t st = 0; st < near.stages; ++st, a.near.first += a.near.groups) {
                    const bool last = st + 1 == near.stages;
                    a.near.groups = near.groups[st];
                    TV_HIP(tv::launch_scan_near(a, g.bits, plan.grid_near, ix->stream));
                    r.stage = a.near;
                    r.seg0 = uint32_t(st) * near.splits * near.sub;
                    TV_HIP(tv::launch_near_rescore(r, ix->stream));
                    const uint32_t n_seg = r.seg0 + near.splits * near.sub;
                    const int rank = near.rank[st + 1];
                    if (!last)
                        TV_HIP(tv::launch_final(d_cand, d_cnt, n_seg, uint32_t(seg_stride), rank, rank, int(pq_n), d_os, d_oi, d_over, d_tau, int(tile_q), 2, nullptr, nullptr,
                                                nullptr, nullptr, nullptr, nullptr, nullptr, 0.0, ix->stream));
                    else
                        TV_HIP(tv::launch_final(d_cand, d_cnt, n_seg, uint32_t(seg_stride), int(k_eff), int(k_floor), int(pq_n), d_os, d_oi, d_over, nullptr, int(tile_q), 1,
                                                d_raise + (q0 - g0), nullptr, nullptr, nullptr, nullptr, ix->rows().slots, timed_pass ? ix->d_stamps + tv::kStampsBefore : nullptr, 0.0,
                                                ix->stream, near.guessed ? d_tau : nullptr));
                }
                if (timed_pass) {
                    stamped = true;
                    n_timed = 2 * near.stages;
                }
                return TV_OK;
            }
            for (size_t lv = 0; lv < steps.size(); ++lv) {
                const bool last = lv + 1 == steps.size();
                // Sampling levels only yield floors, never slots, so the shifted origin of a repeated
                // pass needs no correction downstream.
                const uint32_t off = repeat ? repeat_offset(steps[lv]) : 0u;
                const size_t level_blocks = (n_blocks - off + steps[lv] - 1) / steps[lv];
                // level 1 appends every slot it reads: two blocks per workgroup fill a segment exactly
                const int lgrid = int(std::min<size_t>(size_t(grid), std::max<size_t>(1, (level_blocks + 1) / 2)));
                // A sampling level behind the first filters by the floor of the level before; when
                // that floor was far too low (rows laid out against the sample) its candidates do not
                // fit, k_final says so in the level's flag, and the level runs once more from the
                // floor k_final took from what did fit -- launches that do nothing unless the flag
                // is set.  The full scan then starts from the floor the level was meant to give.
                uint32_t *lv_flag = (!last && (lv > 0 || repeat)) ? d_level_flags + lv : nullptr;
                uint32_t *next_flag = (lv + 2 < steps.size()) ? d_level_flags + lv + 1 : nullptr;
                if (lv == 0 && steps.best_words) {
                    if (const int frc = floors_of_best(steps[0], int(k_floor))) return frc;
                    continue;
                }
                for (int attempt = 0; attempt < (lv_flag ? 2 : 1); ++attempt) {
                    const uint32_t *run_if = attempt == 0 ? nullptr : lv_flag;
                    int n_seg = lgrid;
                    size_t launch_no = 0;
                    // sampling levels of the sixteen-query LUT scan: all the chunk's tiles it serves in one
                    // launch, side by side (one tile leaves most of the chip idle for a round's time)
                    const size_t side_by_side = (plan.lut16 && !last && pq.d_tables16 != nullptr)
                                                    ? pq_n / tile_q + (pq_n % tile_q >= size_t(lut16_min_queries(ix)) ? 1 : 0) : 0;
                    for (size_t t = 0; t < n_tiles; t += (t < side_by_side ? side_by_side : tiles_per_launch), ++launch_no) {
                        tv::ScanArgs a;
                        fill_scan_args(ix, a);
                        a.mask = mask;
                        a.tables = pq.d_tables + t * (mode_p ? pq.table_bytes_per_tile : tile_q * size_t(g.nch) * 1024);
                        a.qscale = pq.d_qscale + t * tile_q;
                        a.qbias = pq.d_qbias + t * tile_q;
                        a.nq_tile = int(std::min<size_t>(tile_q * tiles_per_launch, pq_n - t * tile_q));
                        a.k = 1;
                        a.gtau = ((lv == 0 && !repeat) ? ix->d_tau_open : d_tau) + t * tv::kQTile;
                        a.b_step = steps[lv];
                        a.run_if = run_if;
                        a.best_of_block = (best_first && lv == 0) ? 1 : 0;
                        if (off) {
                            a.codes += size_t(off) * g.block_bytes();
                            a.scales += size_t(off) * tv::kVecBlock;
                            if (a.mask) a.mask += off / 2;
                            a.n_blocks -= off;
                            a.n -= off * tv::kVecBlock;
                        }
                        a.cand = d_cand + t * tile_q * seg_stride * tv::kSegCap;
                        a.cand_cnt = d_cnt + t * tile_q * seg_stride;
                        a.seg_stride = uint32_t(seg_stride);
                        const bool timed = timed_pass && last && steps.size() == 1 && int(launch_no) < kMaxTimedTiles;
                        if (timed) TV_HIP(hipEventRecord(ix->ev_start[launch_no], ix->stream));
                        if (wide) {
                            n_seg = grid;
                            TV_HIP(tv::launch_scan_p4_wide(a, n_seg, ix->stream));
                        } else if (batched) {
                            n_seg = int(std::min<size_t>(size_t(bgrid), seg_stride));
                            TV_HIP(tv::launch_scan_p4_batched(a, n_seg, ix->stream));
                        } else if (mode_p) {
                            TV_HIP(tv::launch_scan_p4(a, lgrid, (best_first && lv == 0) ? tv::kModeBest : tv::kModeAppend, ix->stream));
                        } else if (plan.lut_mx) {
                            const tv::MxShape shape = tv::mx_shape(ix->device, pq_n, level_blocks, lv == 0 && !repeat);
                            n_seg = int(shape.wgs * shape.sub);
                            a.tables = pq.d_tables_mx;
                            TV_HIP(tv::launch_scan_lut_mx(a, shape, g.bits, ix->stream));
                        } else if (t < side_by_side) {
                            a.tables = pq.d_tables16;
                            a.nq_tile = int(std::min<size_t>(pq_n, side_by_side * tile_q));
                            TV_HIP(tv::launch_scan_lut16(a, lgrid, int(side_by_side), ix->stream));
                        } else if (pq.d_tables16 != nullptr && a.nq_tile >= lut16_min_queries(ix)) {
                            a.tables = pq.d_tables16 + t * tv::lut16_table_bytes(g.nch, tile_q);
                            TV_HIP(tv::launch_scan_lut16(a, lgrid, 1, ix->stream));
                        } else {
                            TV_HIP(tv::launch_scan_lut(a, lgrid, tv::kModeAppend, ix->stream));
                        }
                        if (timed) TV_HIP(hipEventRecord(ix->ev_stop[launch_no], ix->stream));
                    }
                    if (last && timed_pass) {      // (two stamps enclose every launch, events the first ones only)
                        stamped = steps.size() > 1;
                        n_timed = stamped ? launch_no : std::min<size_t>(launch_no, size_t(kMaxTimedTiles));
                    }
                    // a floor is the k_floor-th best of the level before, and of 256 segments that hold eight candidates on average one holds
                    // twice that; without a floor every slot, or every block's best, is there, dealt out evenly
                    const double longest = (lv > 0 ? 2.0 * double(k_floor) * steps[lv - 1] / steps[lv] : double(level_blocks) * (best_first ? 1 : int(tv::kVecBlock))) / n_seg;
                    // the first final pass may hand raised floors to a repeated one; the repeated pass
                    // sends what still does not fit to the exact path
                    TV_HIP(tv::launch_final(d_cand, d_cnt, uint32_t(n_seg), uint32_t(seg_stride), int(k_eff), int(k_floor),
                                            int(pq_n), d_os, d_oi, d_over, last ? nullptr : d_tau, int(tile_q),
                                            (lv > 0 || repeat) ? 1 : 0, (last && !repeat) ? d_raise + (q0 - g0) : nullptr,
                                            repeat ? d_rows + row0 : nullptr, lv_flag, attempt == 0 ? next_flag : nullptr,
                                            run_if, ix->rows().slots, !timed_pass ? nullptr : last ? ix->d_stamps + tv::kStampsBefore : lv + 2 == steps.size() ? ix->d_stamps : nullptr,
                                            longest, ix->stream));
                }
            }
            if (repeat) TV_HIP(hipMemcpyAsync(h_over, d_over, pq_n * sizeof(uint32_t), hipMemcpyDeviceToHost, ix->stream));
            return TV_OK;
        };

        // first passes of every chunk of the group, back to back; one read of the flags at the end
        for (size_t c = 0; c < n_chunks; ++c) {
            rc = pass(g0 + chunk_at[c], 0, chunk_at[c + 1] - chunk_at[c], false, timing && c == 0, c);
            if (rc != TV_OK) return rc;
        }
        if (track_levels)
            TV_HIP(hipMemcpyAsync(h_over + kGroupQueries, d_level_flags_all, kLevelFlagWords * 4, hipMemcpyDeviceToHost, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
        staged.idle = true;
        if (track_levels) {
            // flags of levels the passes above did not use hold whatever the workspace held: count only the used ones
            for (size_t c = 0; c < n_chunks; ++c) {
                const SampledPlan plan = sampled_plan(ix, chunk_at[c + 1] - chunk_at[c]);
                if (staged.there && near_of(plan, chunk_at[c + 1] - chunk_at[c]).stages > 0) continue;
                const size_t n_levels = level_strides(ix, plan, n_blocks, mask ? sure : n_blocks, k_floor, false, mask != nullptr).size();
                for (size_t lv = 1; lv + 1 < n_levels; ++lv)
                    ix->level_repeats += h_over[kGroupQueries + c * SamplingSteps::kMax + lv] != 0u;
            }
        }
        if (stamped) {
            rc = take_stamps(ix, int(n_timed));
            if (rc != TV_OK) return rc;
        }
        for (size_t t = 0; t < n_timed && !stamped; ++t) {
            float ms = 0.0f;
            TV_HIP(hipEventElapsedTime(&ms, ix->ev_start[t], ix->ev_stop[t]));
            ix->last_scan_ms += ms;
            ix->last_scan_launches += 1;
        }
        // Queries whose candidates did not fit (an unlucky sample, adversarial order).  Those that
        // came back with a raised floor (flag 1) are packed and scanned once more, a chunk's worth
        // together; what still does not fit then, and what had no floor to raise (flag 2), is
        // redone exactly.
        std::vector<uint32_t> redo_rows, exact_rows;    // group-relative query numbers
        for (size_t q = 0; q < gq; ++q) {
            if (h_over[q] == 1u) redo_rows.push_back(uint32_t(q));
            else if (h_over[q] != 0u) exact_rows.push_back(uint32_t(q));
        }
        ix->overflow_redos += redo_rows.size() + exact_rows.size();
        if ((redo_rows.size() + exact_rows.size()) * 8 >= gq) {
            const SampledPlan plan = sampled_plan(ix, chunk_at[1] - chunk_at[0]);
            const NearPlan near = staged.there ? near_of(plan, chunk_at[1] - chunk_at[0]) : NearPlan{};
            if (near.stages > 0 && near.guessed) {
                // (neighbours that lie together: a share of the rows has all of a query's best or none)
                ix->near_sure_left = kRowLadderSearches;
            } else if (near.stages > 0 ||
                level_strides(ix, plan, n_blocks, mask ? sure : n_blocks, k_floor, false, mask != nullptr).best_first) {
                // from here on, the repeated passes below included -- unless the row-level ladder has just failed too
                if (ix->floorless_kept_left == 0) ix->row_ladder_left = kRowLadderSearches;
            } else if (ix->row_ladder_left > 0) {
                // rows laid out against the row-level ladder as well: back to the floorless level, whose
                // failure is the cheaper one (its full scan gives up within a few rounds), and no
                // switching for a while
                ix->row_ladder_left = 0;
                ix->floorless_kept_left = kRowLadderSearches;
            }
        }
        if (ix->allowed.in_place && !(redo_rows.empty() && exact_rows.empty())) {     // (the passes below run on every kernel)
            left_in_place = true;
            rc = leave_in_place(ix, redo_rows.size() + exact_rows.size(), k_eff);
            if (rc != TV_OK) return rc;
            read(ix->allowed);
        }
        const size_t room = ix->ws_bytes - head.used;
        for (size_t i = 0; i < redo_rows.size();) {
            // rows of one chunk go together: all of them in one pass when the workspace holds that
            // pass, else in the largest pieces it holds
            size_t chunk = 0;
            while (chunk_at[chunk + 1] <= redo_rows[i]) ++chunk;
            size_t e = i;
            while (e < redo_rows.size() && redo_rows[e] < chunk_at[chunk + 1]) ++e;
            size_t piece = std::min<size_t>(e - i, tv::kQTile);
            for (size_t cand_piece : kRepeatPieces) {
                const size_t m = std::min(cand_piece, e - i);
                if (sampled_plan(ix, m).need <= room) { piece = m; break; }
            }
            for (size_t r = 0; r < piece; ++r) h_over[r] = redo_rows[i + r] - uint32_t(chunk_at[chunk]);   // pinned staging
            TV_HIP(hipMemcpyAsync(d_rows, h_over, piece * sizeof(uint32_t), hipMemcpyHostToDevice, ix->stream));
            TV_HIP(hipStreamSynchronize(ix->stream));
            rc = pass(g0 + chunk_at[chunk], 0, piece, true, false, chunk);
            if (rc != TV_OK) return rc;
            TV_HIP(hipStreamSynchronize(ix->stream));
            for (size_t r = 0; r < piece; ++r)
                if (h_over[r] != 0u) exact_rows.push_back(redo_rows[i + r]);
            i += piece;
        }
        std::sort(exact_rows.begin(), exact_rows.end());
        ix->exact_redos += exact_rows.size();
        for (size_t i = 0; i < exact_rows.size();) {
            size_t e = i + 1;
            while (e < exact_rows.size() && exact_rows[e] == exact_rows[e - 1] + 1) ++e;     // runs of neighbours go together
            const size_t qa = g0 + exact_rows[i], cnt = e - i;
            rc = search_robust(ix, d_queries + qa * g.dim, cnt, k_eff, mask, d_out_scores + qa * k_eff, d_out_idx + qa * k_eff,
                               false);
            if (rc != TV_OK) return rc;
            i = e;
        }
    }
    if (asked.in_place && !left_in_place) ++ix->in_place_searches;
    return TV_OK;
}

// ---- filtered searches on the allowed rows alone (tv_filter.hip) ----
// What a scan costs per block, in ns, about: its codes at 6.4 TB/s, or the products and the epilogue of each tile of 32 queries, or
// passes over u8 tables.  (P: 4M x 768, 300 queries 1.3 ms, 1024 3.3, 2M x 1536 1.2 and 3.1; tables: 1M x 1536 2-bit, 300 queries 1.7 ms,
// 1024 4.6, 4M x 256 1.8 and 5.2, 778K x 1000 3-bit 1.2 and 2.9, all with 10 % of the rows allowed.)
double scan_block_ns(const tv_index *ix, size_t nq) {
    const double tiles = double((nq + tv::kQTile - 1) / tv::kQTile), nch = double(ix->geo.nch);
    if (effective_mode(ix) == TV_SCORE_P) return std::max(0.165 * nch, tiles * (0.055 * nch + 0.25) + 0.1 * nch);
    if (effective_mode(ix) != TV_SCORE_L_U32) return std::max(0.165, 0.025 * double(nq)) * nch;
    if (nq <= size_t(tv::kLut16Queries)) return (0.165 + 0.02 * double(nq)) * nch + 0.3;
    return tiles * ((ix->geo.bits == 2 ? 0.37 : 0.22) * nch + 0.6);
}
// What any block costs a tile of a large batch, one without an allowed row too: passing it, its place among the best words (a
// range of 1 % of the rows, 1024 queries: 4M x 256 2-bit 522 us with the mask and 144 gathered, 1M x 128 215 and 86).
constexpr double kPassedBlockNs = 0.08;
// Gathering, per gathered block and chunk: the lines its rows lie in, up to eight times their bytes, and the write; and its
// launches and the wait for the count, or what is left of them once the blocks are counted, or where the host knew.  (22 us: half the rows of
// 100K x 128 at random, 1024 queries, are 20 by this count, and gathering them gains 4 of 78; 10 us from the host: a range of 1 % of
// 100K x 1536, 1024 queries, is 7.7, and 370 us with the mask and 374 gathered.)  The launches that a search without sampling saves.
constexpr double kGatherNs = 0.2, kGatherFixedNs = 22000.0, kCountedNs = 5000.0, kKnownNs = 10000.0, kUnsampledNs = 25000.0, kNearFixedNs = 80000.0;
// Rows listed while the host waits for the count, and for nothing where it then reads the mask (2M rows of 4M x 256, 40 queries: 181 us
// with the mask and 201 listed first).
constexpr size_t kListedAtOnce = size_t(1) << 18;
constexpr size_t kGatheredBytes = size_t(1) << 30;      // the largest such copy an index keeps room for
bool gather_pays(const tv_index *ix, size_t nq, size_t k, double n_blocks, double live_blocks, double n_allowed, double fixed, bool in_place) {
    const double blocks = n_allowed / tv::kVecBlock + 1.0, each = scan_block_ns(ix, nq);
    // (the two-step table scan, which skips no blocks, takes as much of that beside its stages' launches: 0.85 and 0.7 of the time for 3 and 4 tiles, 0.5 for 7, 0.38 for 32)
    const double tiles = std::min(32.0, double((nq + tv::kQTile - 1) / tv::kQTile)), part = ix->geo.bits == 2 ? 0.33 + 1.5 / tiles : std::min(1.0, 0.4 + 2.5 / tiles);
    auto scan = [&](double count, double read, bool masked) {
        const bool near = effective_mode(ix) == TV_SCORE_L_U32 && !direct_serves(ix, nq, k, size_t(count), masked) && near_takes(ix, nq, k, size_t(count), size_t(n_allowed));
        return near ? kNearFixedNs + part * count * each : read * each;
    };
    const double passed = nq > size_t(tv::kQTile) ? kPassedBlockNs * double((nq + tv::kQTile - 1) / tv::kQTile) : 0.0;
    const double gather = kGatherNs * double(ix->geo.nch) * ((in_place ? -1.0 : 1.0) + std::min(8.0, live_blocks / blocks));
    const bool shorter = direct_serves(ix, nq, k, size_t(blocks), false) && !direct_serves(ix, nq, k, size_t(n_blocks), true);
    return scan(n_blocks, live_blocks, true) + n_blocks * passed + (shorter ? kUnsampledNs : 0.0) > scan(blocks, blocks, false) + blocks * (passed + gather) + fixed;
}
size_t gathered_need(const tv_index *ix, size_t n_allowed) {
    const size_t blocks = (n_allowed + tv::kVecBlock - 1) / tv::kVecBlock;
    return round_up(blocks * ix->geo.block_bytes(), 256) + blocks * tv::kVecBlock * sizeof(float);
}
// Whether a search over n_allowed rows runs on the all-queries kernel throughout, which can read them where they lie.
bool scans_in_place(const tv_index *ix, size_t nq, size_t k_eff, size_t n_allowed) {
    const size_t blocks = (n_allowed + tv::kVecBlock - 1) / tv::kVecBlock;
    if (!wide_serves(ix) || !tv::wide_serves_best_of_block(ix->geo.nch)) return false;
    if (k_eff > size_t(tv::kMaxSampledK) || ix->force_robust || direct_serves(ix, nq, k_eff, blocks, false)) return false;
    for (size_t g0 = 0; g0 < nq; g0 += kGroupQueries) {
        const size_t gq = std::min(kGroupQueries, nq - g0);
        for (size_t c0 = 0, cq; c0 < gq; c0 += cq) {
            cq = chunk_len(ix, gq - c0);
            const SampledPlan plan = sampled_plan(ix, cq);
            if (!plan.wide || !tv::wide_reads_rows(ix->geo.nch, int(cq))) return false;
        }
    }
    return true;
}
// Spares in use, or free to be taken again.
void use_spares(tv_index *ix, bool in_use) {
    std::lock_guard<std::mutex> lock(g_pool[ix->device].mu);
    ix->slots.in_use = ix->gathered.in_use = in_use;
}
// A block, in use already, where there is memory for it.  (The search reads the mask as it scans otherwise, as it would have.)
bool have_block(tv_index *ix, tv_spare &s, size_t bytes) {
    if (ensure_block(ix, s.p, s.bytes, bytes) == TV_OK) return true;
    g_last_error.clear();
    return false;
}
int copy_allowed(tv_index *ix, const uint32_t *slots, size_t total, size_t live) {
    if (!have_block(ix, ix->gathered, gathered_need(ix, total))) return TV_OK;
    uint8_t *codes = static_cast<uint8_t *>(ix->gathered.p);
    float *scales = reinterpret_cast<float *>(codes + round_up((total + tv::kVecBlock - 1) / tv::kVecBlock * ix->geo.block_bytes(), 256));
    TV_HIP(tv::launch_gather_rows(ix->d_codes, ix->d_scales, ix->geo.nch, slots, total, codes, scales, ix->stream));
    ix->allowed = tv_rows{codes, scales, total, slots, live, false};
    return TV_OK;
}
// What queries whose candidates did not fit in a scan of rows in place are repeated on: a copy of the rows where so
// many queries pay for it, the mask otherwise.
int leave_in_place(tv_index *ix, size_t nq, size_t k_eff) {
    const tv_rows was = std::exchange(ix->allowed, tv_rows{});
    const size_t n_blocks = (ix->n + tv::kVecBlock - 1) / tv::kVecBlock;
    if (gathered_need(ix, was.n) > kGatheredBytes || !gather_pays(ix, nq, k_eff, double(n_blocks), double(was.live), double(was.n), kCountedNs, false)) return TV_OK;
    return copy_allowed(ix, was.slots, was.n, was.live);
}
// With the mask read during the scan, and gathered, us a search (k = 10): 10 % of the rows allowed at random, 4M x 256 2-bit, 1024 queries 5210 and
// 680; 4M x 768, 300 queries 1359 and 403; 1M x 768, 40 queries 131 and 105, 1 query 112 and 104; 1 %: 2M x 1536, 1024 queries 1295 and
// 165, 1 query 152 and 74; 50 %: 4M x 768, 64 queries 425 and 660.  A range of 20 % of the
// rows: 4M x 768, 300 queries 376 and 470.  Read in place (with the mask, copied, in place): 50 %, 4M x 768, 1024 queries 3337, 2030 and 1650, 300 queries 1310, 1050 and
// 700; 10M x 1536, 1024 queries 13270 and, in place, 7130; 80 % 1330 and 970 in place; 30 %, 2M x 1536, 300 queries 1181 and 754; a range of half the rows, 1024 queries 1601 and 1576.
// k = 100, 50 %, from the row-level ladder (a copy, searched from best words, and in place): 4M x 768, 300 queries 1166 and 878, 1024 queries 2204 and 2116; 80 %,
// 300 queries 1363 and 1175; with the mask and in place: 2M x 1536, 300 queries 1118 and 815.
// Gathers the rows `d_mask` allows where a search of nq queries is faster on them; ix->allowed then has them.  Whether rows
// lie scattered, which it depends on, a caller says who has seen the mask (live, the blocks with an allowed row); otherwise it is counted on
// the device and waited for, and from the number of allowed rows alone, taken to be scattered, most calls that
// it cannot pay for are told without.  A search that counts and then reads the mask, of a
// range of the rows, pays 8 us (100K x 1536, 300 queries, 20 %: 88 and 96).
int gather_allowed(tv_index *ix, const uint64_t *d_mask, size_t n_allowed, size_t &live, size_t nq, size_t k_eff) {
    const size_t n = ix->n, n_blocks = (n + tv::kVecBlock - 1) / tv::kVecBlock;
    if (ix->ws_fixed || ix->no_gather || n_allowed == 0 || n_allowed >= n || n >= (size_t(1) << 31)) return TV_OK;
    bool in_place = scans_in_place(ix, nq, k_eff, n_allowed);
    const bool large = in_place && n_blocks * ix->geo.block_bytes() > 0xffffffffull;      // rows of a block may lie too far apart
    if (!in_place && gathered_need(ix, n_allowed) > kGatheredBytes) return TV_OK;
    auto pays = [&](double blocks, double fixed) {
        return ix->force_gather || gather_pays(ix, nq, k_eff, double(n_blocks), blocks, double(n_allowed), fixed, in_place);
    };
    const bool known = live != kLiveUnknown;
    const double scattered = double(n_blocks) * (1.0 - std::pow(1.0 - double(n_allowed) / double(n), double(tv::kVecBlock)));
    if (!(known ? pays(double(live), kKnownNs) : pays(scattered, kGatherFixedNs))) return TV_OK;
    const size_t count_bytes = round_up(tv::mask_counts(n) * 2 * sizeof(uint32_t), 256);
    use_spares(ix, true);
    if (!have_block(ix, ix->slots, count_bytes + n_allowed * sizeof(uint32_t))) return TV_OK;
    uint32_t *counts = static_cast<uint32_t *>(ix->slots.p), *slots = counts + count_bytes / sizeof(uint32_t);
    static_assert(kGroupQueries >= 2 * tv::kMaxMaskTotals + 1, "the counts lie where the flags will");
    volatile uint64_t *totals = reinterpret_cast<uint64_t *>(ix->h_flags);
    const size_t n_totals = tv::mask_totals(n);
    for (size_t i = 0; i < n_totals; ++i) totals[i] = 0;
    TV_HIP(tv::launch_mask_count(d_mask, n, counts, known ? nullptr : reinterpret_cast<uint64_t *>(ix->d_flags_host), ix->stream));
    // (a short list is there by the time the host has the count and has launched what comes next)
    const bool at_once = known || n_allowed <= kListedAtOnce;
    if (at_once) TV_HIP(tv::launch_mask_slots(d_mask, n, counts, slots, n_allowed, ix->stream));
    if (!known) {
        // (a wait of a few microseconds, which through the runtime takes ten more; beyond that it is the runtime's)
        const auto until = std::chrono::steady_clock::now() + std::chrono::microseconds(200);
        size_t there = 0;
        while (there < n_totals && (totals[there] != 0 || std::chrono::steady_clock::now() < until)) there += totals[there] != 0;
        if (there < n_totals) TV_HIP(hipStreamSynchronize(ix->stream));
        uint64_t sum = 0;
        for (size_t i = 0; i < n_totals; ++i) sum += totals[i] & ~tv::kMaskCounted;
        if ((sum & 0x7fffffffu) != n_allowed) return TV_OK;      // (the caller's count is not the mask's)
        live = size_t(sum >> 31);
        if (!pays(double(live), kCountedNs)) return TV_OK;
    }
    if (!at_once) TV_HIP(tv::launch_mask_slots(d_mask, n, counts, slots, n_allowed, ix->stream));
    if (large) {
        volatile uint32_t *far = ix->h_flags + 2 * tv::kMaxMaskTotals;
        *far = 0;
        TV_HIP(tv::launch_rows_apart(slots, n_allowed, ix->geo.block_bytes(), ix->d_flags_host + 2 * tv::kMaxMaskTotals, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
        if (*far != 0) {
            in_place = false;
            if (gathered_need(ix, n_allowed) > kGatheredBytes || !pays(double(live), kCountedNs)) return TV_OK;
        }
    }
    if (in_place) ix->allowed = tv_rows{ix->d_codes, ix->d_scales, n_allowed, slots, live, true};
    else if (const int rc = copy_allowed(ix, slots, n_allowed, live)) return rc;
    if (ix->allowed.codes) ++ix->gathered_searches;
    return TV_OK;
}
// live: the blocks of 32 rows with one that the mask allows, where the caller knows.
int search_device(tv_index *ix, const float *d_queries, size_t nq, size_t k, const uint64_t *d_mask,
                  size_t n_allowed, size_t live, float *d_out_scores, int64_t *d_out_idx, size_t *out_k_eff) {
    struct Back {
        tv_index *ix;
        void give() {
            ix->allowed = tv_rows{};
            if (ix->slots.in_use) use_spares(ix, false);
        }
        ~Back() { give(); }
    } back{ix};
    if (d_mask && k != 0 && nq != 0) {
        const int rc = gather_allowed(ix, d_mask, n_allowed, live, nq, std::min(std::min(k, ix->n), n_allowed));
        if (rc != TV_OK) return rc;
    }
    g_refused = false;
    const int rc = search_rows(ix, d_queries, nq, k, d_mask, n_allowed, live, d_out_scores, d_out_idx, out_k_eff);
    if (rc == TV_OK || !g_refused || !ix->slots.in_use) return rc;
    // no memory for the search beside its list and copy of rows, which are given up for it
    TV_HIP(hipStreamSynchronize(ix->stream));
    back.give();
    return search_rows(ix, d_queries, nq, k, d_mask, n_allowed, live, d_out_scores, d_out_idx, out_k_eff);
}

// ---- search calls, merged ----------------------------------------------------------------------
// The reference's search takes &self and runs on as many caller threads as there are
// (turbovec/src/lib.rs:22-52, tests/concurrent_search.rs); one GPU serves one launch at a time, and a
// launch costs the same for one query as for thirty-two.  So calls do not queue up one behind the
// other: a call registers itself, then waits for the index; whoever gets it next serves every
// registered call that is compatible with its own (same kind of buffers, same k, same mask) as one
// batch -- rows of a batch are scored independently, so each caller receives exactly what a call of
// its own would have returned -- and the others find their results ready when their turn comes.
constexpr size_t kMergeQueries = 4096;   // queries one merged batch may hold

}  // namespace

struct tv_request {
    bool host = true;              // tv_search (host buffers) or tv_search_dev (device buffers)
    const float *q = nullptr;
    size_t nq = 0, k = 0;
    const uint64_t *mask = nullptr;
    size_t mask_arg = 0;           // host: number of mask words; device: the mask's popcount
    float *out_s = nullptr;
    int64_t *out_i = nullptr;
    // host arrays that have been staged in pinned memory (q, out_s, out_i and staged_mask point into it): the device's addresses
    const uint64_t *staged_mask = nullptr;     // (mask stays the caller's: calls with one mask are told by its address)
    const float *dev_q = nullptr;  // or null: not staged
    float *dev_s = nullptr;
    int64_t *dev_i = nullptr;
    size_t k_eff = 0;
    int rc = TV_OK;
    std::string err;
    bool done = false;
};

namespace {

// The rows a mask allows, and the blocks of 32 with one.  For the 1.25 MB of 10M rows: 54 us with 256-bit vectors, which the
// build's flags do not ask for, and 150 without (120 for the rows alone).
typedef uint32_t HalfWord __attribute__((may_alias));
__attribute__((always_inline)) inline void count_words(const uint64_t *words, size_t n, size_t &rows, size_t &live) {
    for (size_t w = 0; w < n; w += 1024) {      // (from the first-level cache the second time)
        const uint64_t *x = words + w;
        const size_t m = std::min<size_t>(1024, n - w);
        uint64_t r = 0;
        uint32_t l = 0;
        for (size_t i = 0; i < m; ++i) r += uint64_t(__builtin_popcountll(x[i]));
        const HalfWord *h = reinterpret_cast<const HalfWord *>(x);      // (their order does not matter)
        for (size_t i = 0; i < 2 * m; ++i) l += uint32_t(h[i] != 0);
        rows += r;
        live += l;
    }
}
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
__attribute__((target("avx2"))) void count_words_avx2(const uint64_t *words, size_t n, size_t &rows, size_t &live) { count_words(words, n, rows, live); }
#endif
void count_mask(const uint64_t *words, size_t n, size_t &rows, size_t &live) {
    rows = live = 0;
    const uint64_t last = n % 64 ? words[n / 64] & ((uint64_t(1) << (n % 64)) - 1) : 0;
    count_words(&last, 1, rows, live);
#if defined(__x86_64__) && !defined(__HIP_DEVICE_COMPILE__)
    if (__builtin_cpu_supports("avx2")) return count_words_avx2(words, n / 64, rows, live);
#endif
    count_words(words, n / 64, rows, live);
}

// Serves the calls of `batch` (compatible with each other, at least one) as one search.  The index
// lock is held.  Returns the status every one of them gets.
int serve_batch(tv_index *ix, const std::vector<tv_request *> &batch, size_t *k_eff_out) {
    const tv_request &r0 = *batch[0];
    TV_HIP(hipSetDevice(ix->device));
    const size_t n = ix->n, dim = size_t(ix->geo.dim);
    size_t nq = 0;
    for (const tv_request *r : batch) nq += r->nq;
    if (!r0.host) {
        const size_t n_allowed = r0.mask ? r0.mask_arg : n;
        if (batch.size() == 1)
            return search_device(ix, r0.q, nq, r0.k, r0.mask, n_allowed, kLiveUnknown, r0.out_s, r0.out_i, k_eff_out);
        // several callers' device buffers: gathered into the staging allocation, results scattered back
        const size_t k_eff = std::min(std::min(r0.k, n), n_allowed);
        *k_eff_out = k_eff;
        if (k_eff == 0 || nq == 0) return TV_OK;
        const size_t q_bytes = round_up(nq * dim * sizeof(float), 256), s_bytes = round_up(nq * k_eff * sizeof(float), 256);
        const size_t i_bytes = round_up(nq * k_eff * sizeof(int64_t), 256);
        int rc = ensure_io(ix, q_bytes + s_bytes + i_bytes);
        if (rc != TV_OK) return rc;
        uint8_t *base = static_cast<uint8_t *>(ix->io);
        float *d_q = reinterpret_cast<float *>(base);
        float *d_s = reinterpret_cast<float *>(base + q_bytes);
        int64_t *d_i = reinterpret_cast<int64_t *>(base + q_bytes + s_bytes);
        size_t at = 0;
        for (const tv_request *r : batch) {
            if (r->nq) TV_HIP(hipMemcpyAsync(d_q + at * dim, r->q, r->nq * dim * sizeof(float), hipMemcpyDeviceToDevice, ix->stream));
            at += r->nq;
        }
        rc = search_device(ix, d_q, nq, r0.k, r0.mask, n_allowed, kLiveUnknown, d_s, d_i, nullptr);
        if (rc != TV_OK) return rc;
        at = 0;
        for (const tv_request *r : batch) {
            if (r->nq) {
                TV_HIP(hipMemcpyAsync(r->out_s, d_s + at * k_eff, r->nq * k_eff * sizeof(float), hipMemcpyDeviceToDevice, ix->stream));
                TV_HIP(hipMemcpyAsync(r->out_i, d_i + at * k_eff, r->nq * k_eff * sizeof(int64_t), hipMemcpyDeviceToDevice, ix->stream));
            }
            at += r->nq;
        }
        TV_HIP(hipStreamSynchronize(ix->stream));
        return TV_OK;
    }
    const uint64_t *mask_words = r0.staged_mask ? r0.staged_mask : r0.mask;
    const size_t n_mask_words = r0.mask_arg;
    size_t n_allowed = n, live = 0;
    if (mask_words) {
        if (n_mask_words != (n + 63) / 64) return TV_ERR_MASK_LENGTH_MISMATCH;
        count_mask(mask_words, n, n_allowed, live);  // search.rs:3222-3225; bits at or past n are ignored
    }
    const size_t k_eff = std::min(std::min(r0.k, n), n_allowed);
    *k_eff_out = k_eff;
    ix->last_scan_ms = 0.0f;
    ix->last_scan_launches = 0;
    if (k_eff == 0 || nq == 0) return TV_OK;
    // The device reads a staged caller's queries and writes its results where they lie (a large set of queries is
    // copied over first); several callers' are gathered on the device, as are arrays that are not staged, in an
    // allocation the index keeps between calls, apart from the per-chunk workspace, which is re-carved freely.
    const bool in_place = batch.size() == 1 && r0.dev_q != nullptr;
    const bool read_in_place = in_place && nq * dim * sizeof(float) <= kReadInPlace;
    const size_t q_bytes = read_in_place ? 0 : round_up(nq * dim * sizeof(float), 256), m_bytes = mask_words ? round_up(n_mask_words * 8, 256) : 0;
    const size_t s_bytes = in_place ? 0 : round_up(nq * k_eff * sizeof(float), 256), i_bytes = in_place ? 0 : round_up(nq * k_eff * sizeof(int64_t), 256);
    int rc = ensure_io(ix, q_bytes + s_bytes + i_bytes + m_bytes);
    if (rc != TV_OK) return rc;
    uint8_t *base = static_cast<uint8_t *>(ix->io);
    const float *d_q = read_in_place ? r0.dev_q : reinterpret_cast<float *>(base);
    float *d_s = in_place ? r0.dev_s : reinterpret_cast<float *>(base + q_bytes);
    int64_t *d_i = in_place ? r0.dev_i : reinterpret_cast<int64_t *>(base + q_bytes + s_bytes);
    uint64_t *d_m = mask_words ? reinterpret_cast<uint64_t *>(base + q_bytes + s_bytes + i_bytes) : nullptr;
    size_t at = 0;
    for (const tv_request *r : batch) {
        if (read_in_place) break;
        if (r->nq && hipMemcpyAsync(reinterpret_cast<float *>(base) + at * dim, r->q, r->nq * dim * sizeof(float), hipMemcpyHostToDevice, ix->stream) != hipSuccess) {
            g_last_error = "host to device copy failed";
            return TV_ERR_HIP;
        }
        at += r->nq;
    }
    if (mask_words && hipMemcpyAsync(d_m, mask_words, n_mask_words * 8, hipMemcpyHostToDevice, ix->stream) != hipSuccess) {
        g_last_error = "host to device copy failed";
        return TV_ERR_HIP;
    }
    // (an array that is not staged may change until it has been copied: the device counts what it got)
    rc = search_device(ix, d_q, nq, r0.k, d_m, n_allowed, r0.staged_mask ? live : kLiveUnknown, d_s, d_i, nullptr);
    if (rc != TV_OK || in_place) return rc;
    at = 0;
    for (const tv_request *r : batch) {
        if (r->nq && (hipMemcpyAsync(r->out_s, d_s + at * k_eff, r->nq * k_eff * sizeof(float), hipMemcpyDeviceToHost, ix->stream) != hipSuccess ||
                      hipMemcpyAsync(r->out_i, d_i + at * k_eff, r->nq * k_eff * sizeof(int64_t), hipMemcpyDeviceToHost, ix->stream) != hipSuccess)) {
            g_last_error = "device to host copy failed";
            return TV_ERR_HIP;
        }
        at += r->nq;
    }
    if (hipStreamSynchronize(ix->stream) != hipSuccess) {
        g_last_error = "device to host copy failed";
        return TV_ERR_HIP;
    }
    return TV_OK;
}

bool compatible(const tv_request &a, const tv_request &b) {
    if (a.host != b.host || a.k != b.k || a.mask != b.mask || a.mask_arg != b.mask_arg) return false;
    // (one array, but each call searches what was in it when it was made)
    const uint64_t *x = a.staged_mask ? a.staged_mask : a.mask, *y = b.staged_mask ? b.staged_mask : b.mask;
    return x == y || std::memcmp(x, y, a.mask_arg * sizeof(uint64_t)) == 0;
}

// How long a caller that is about to serve waits for the callers of the batch before to come back
// with their next call (they were all released at the same moment and are a few microseconds of
// host code away from asking again).  Only after a batch that did merge calls.
constexpr auto kGatherWait = std::chrono::microseconds(300);
constexpr auto kContendedWait = std::chrono::microseconds(20);

int search_merged(tv_index *ix, tv_request &r) {
    std::vector<tv_request *> batch;
    {
        std::unique_lock<std::mutex> reg(ix->waiting_mu);
        ix->waiting.push_back(&r);
        bool had_to_wait = false;
        ix->waiting_cv.notify_all();       // a serving caller gathering its batch may be waiting for this one
        for (;;) {
            if (r.done) {                  // served by another caller's launch
                if (r.rc != TV_OK) g_last_error = r.err;
                return r.rc;
            }
            if (!ix->serving) break;
            had_to_wait |= compatible(*ix->served, r);
            ix->waiting_cv.wait(reg);
        }
        ix->serving = true;
        ix->served = &r;
        // Callers in a loop come back together: when the batch before held several calls, give the
        // same number a moment to register again instead of serving this one alone and all of them
        // in the launch after.
        if (ix->last_batch_calls > 1) {
            const auto deadline = std::chrono::steady_clock::now() + kGatherWait;
            while (ix->waiting.size() < ix->last_batch_calls)
                if (ix->waiting_cv.wait_until(reg, deadline) == std::cv_status::timeout) break;
        }
        // A caller that had to wait is not the only one in a hurry: a search of a small index takes less time
        // than the callers' own work between two calls, and without a moment's pause they would line up one
        // behind the other.  (Only behind a search it could have shared: callers of other k or masks never can.)
        const auto pause = std::chrono::steady_clock::now() + kContendedWait;
        while (had_to_wait && ix->waiting.size() < 2 && std::chrono::steady_clock::now() < pause) {
            reg.unlock();
            std::this_thread::yield();
            reg.lock();
        }
        // this call first, then the compatible ones in order of arrival, up to the batch limit
        batch.push_back(&r);
        size_t total = r.nq;
        std::vector<tv_request *> rest;
        for (tv_request *w : ix->waiting) {
            if (w == &r) continue;
            if (compatible(*w, r) && total + w->nq <= kMergeQueries) { batch.push_back(w); total += w->nq; }
            else rest.push_back(w);
        }
        ix->waiting.swap(rest);
    }
    size_t k_eff = 0;
    int rc;
    {
        std::lock_guard<std::mutex> lock(ix->mu);   // against the entry points that change the index
        g_last_error.clear();
        rc = serve_batch(ix, batch, &k_eff);
        // (staged arrays go back to their pool: nothing may still be on its way from or to them)
        if (rc != TV_OK) (void)hipStreamSynchronize(ix->stream);
    }
    {
        std::lock_guard<std::mutex> reg(ix->waiting_mu);
        for (tv_request *w : batch) {
            w->rc = rc;
            w->k_eff = k_eff;
            if (rc != TV_OK) w->err = g_last_error;
            w->done = true;
        }
        ix->merged_calls += batch.size() - 1;
        ix->last_batch_calls = batch.size();
        ix->serving = false;
        ix->served = nullptr;
    }
    ix->waiting_cv.notify_all();
    return rc;
}

}  // namespace

extern "C" {

const char *tv_status_string(int status) {
    switch (status) {
        case TV_OK: return "ok";
        case TV_ERR_QUERY_BUFFER_NOT_MULTIPLE_OF_DIM: return "query buffer length not a multiple of dim";
        case TV_ERR_INVALID_QUERY_VALUE: return "invalid query value (must be finite and |value| < 1e16)";
        case TV_ERR_MASK_LENGTH_MISMATCH: return "mask length does not match index size";
        case TV_ERR_ALLOWLIST_EMPTY: return "allowlist is empty";
        case TV_ERR_UNKNOWN_ID: return "id in allowlist is not present in index";
        case TV_ERR_BAD_ARGUMENT: return "bad argument";
        case TV_ERR_HIP: return "HIP runtime error";
        case TV_ERR_NO_DEVICE: return "no usable GPU";
        case TV_ERR_INDEX_OUT_OF_RANGE: return "index out of range";
        case TV_ERR_BAD_IMAGE: return "invalid snapshot image";
        default: return "unknown status";
    }
}

const char *tv_last_error(void) { return g_last_error.c_str(); }

int tv_index_create(int dim, int bits, int device, tv_index **out) {
    if (!out) return TV_ERR_BAD_ARGUMENT;
    *out = nullptr;
    if (bits < 2 || bits > 4) { g_last_error = "bit_width must be 2, 3, or 4"; return TV_ERR_BAD_ARGUMENT; }
    if (dim <= 0 || dim % 8 != 0) { g_last_error = "dim must be a positive multiple of 8"; return TV_ERR_BAD_ARGUMENT; }
    if (dim > 16384) { g_last_error = "dim exceeds maximum 16384"; return TV_ERR_BAD_ARGUMENT; }
    int count = 0;
    if (hipGetDeviceCount(&count) != hipSuccess || count <= device || device < 0) {
        g_last_error = "no HIP device with that ordinal";
        return TV_ERR_NO_DEVICE;
    }
    if (device >= kMaxDevices) { g_last_error = "device ordinal beyond the scratch table"; return TV_ERR_NO_DEVICE; }
    TV_HIP(hipSetDevice(device));
    tv_index *ix = new (std::nothrow) tv_index();
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    ix->device = device;
    {
        DevicePool &pool = g_pool[device];
        std::lock_guard<std::mutex> lock(pool.mu);
        ++pool.indexes;
        ix->older = pool.newest;
        if (ix->older) ix->older->newer = ix;
        pool.newest = ix;
    }
    ix->geo.dim = dim;
    ix->geo.bits = bits;
    ix->geo.G = dim / (8 / bits);
    ix->geo.nch = (ix->geo.G + tv::kChunkGroups - 1) / tv::kChunkGroups;
    // 4-bit rows are padded with whole chunks of zero groups (their query weights are zero, so they
    // add nothing) up to a chunk count the all-queries-per-pass kernel has an instance for: even
    // from 9 chunks on, a multiple of 4 above 24, of 8 above 48 (to 96 chunks = 6144 dimensions).
    // The padding is part of the resident index on every path: at most 3 chunks (of 25: +12 %), 7
    // (of 49: +14 %), one in seven at worst; the device block is geo.block_bytes() = nch * 1024
    // bytes, not ceil(G / 32) * 1024.
    if (bits == 4 && ix->geo.nch >= 9) {
        if (ix->geo.nch > 48 && ix->geo.nch <= 96) ix->geo.nch = (ix->geo.nch + 7) / 8 * 8;
        else if (ix->geo.nch > 24 && ix->geo.nch <= 48) ix->geo.nch = (ix->geo.nch + 3) / 4 * 4;
        else if (ix->geo.nch <= 24) ix->geo.nch += ix->geo.nch & 1;
    }
    const auto tables = default_tables(dim);
    ix->cb = tv::make_codebook(bits, dim);
    int rc = TV_OK;
    do {
        if (hipStreamCreateWithFlags(&ix->stream, hipStreamNonBlocking) != hipSuccess) { rc = TV_ERR_HIP; break; }
        // One block (through device_alloc, which empties the pool before it refuses; too small for the pool itself): what upload_tables
        // copies, the TQ+ pair, the open floors.
        const size_t d = size_t(dim), words = 9 * d + 16 + kTauOpenInts;
        size_t got = 0;
        if (device_alloc(device, words * sizeof(uint32_t), reinterpret_cast<void **>(&ix->d_signs), &got) != hipSuccess) {
            rc = TV_ERR_HIP;
            break;
        }
        ix->d_perms = reinterpret_cast<uint32_t *>(ix->d_signs) + 2 * d;
        ix->d_packed = ix->d_perms + 2 * d;
        ix->d_centroids = reinterpret_cast<float *>(ix->d_packed + 2 * d);
        ix->d_tq_shift = ix->d_centroids + 16;
        ix->d_tq_scale = ix->d_tq_shift + d;
        ix->d_tau_open = reinterpret_cast<int *>(ix->d_tq_scale + 2 * d);
        const size_t flag_bytes = (kGroupQueries + kLevelFlagWords) * sizeof(uint32_t) + (tv::kStampsBefore + 1) * sizeof(uint64_t);
        if (hipHostMalloc(reinterpret_cast<void **>(&ix->h_flags), flag_bytes + (6 * d + 16) * sizeof(uint32_t), hipHostMallocMapped) != hipSuccess) {
            rc = TV_ERR_HIP;
            break;
        }
        ix->h_tables = reinterpret_cast<uint32_t *>(reinterpret_cast<uint8_t *>(ix->h_flags) + flag_bytes);
        if (hipHostGetDevicePointer(reinterpret_cast<void **>(&ix->d_flags_host), ix->h_flags, 0) != hipSuccess) {
            rc = TV_ERR_HIP;
            break;
        }
        static_assert((kGroupQueries + kLevelFlagWords) % 2 == 0, "the stamps behind the flags are 8-byte words");
        ix->h_stamps = reinterpret_cast<uint64_t *>(ix->h_flags + kGroupQueries + kLevelFlagWords);
        ix->d_stamps = reinterpret_cast<uint64_t *>(ix->d_flags_host + kGroupQueries + kLevelFlagWords);
        std::fill_n(ix->h_stamps, tv::kStampsBefore + 1, uint64_t(0));
        rc = upload_tables(ix, *tables);
        if (rc != TV_OK) break;
        rc = scratch_address(device, &ix->scratch);
        if (rc != TV_OK) break;
        ix->rot = tables->rot;      // (while the device reads)
        derive_levels(ix);
        if (hipStreamSynchronize(ix->stream) != hipSuccess) rc = TV_ERR_HIP;
    } while (0);
    if (rc != TV_OK) {
        if (g_last_error.empty()) g_last_error = "device allocation failed";
        tv_index_destroy(ix);
        return rc;
    }
    *out = ix;
    return TV_OK;
}

int tv_index_destroy(tv_index *ix) {
    if (!ix) return TV_OK;
    (void)hipSetDevice(ix->device);
    if (ix->stream) (void)hipStreamSynchronize(ix->stream);
    use_spares(ix, true);      // (from here on they are freed below)
    (void)device_free(ix->device, ix->d_codes, ix->codes_bytes);
    (void)device_free(ix->device, ix->d_scales, ix->scales_bytes);
    (void)device_free(ix->device, ix->ws, ix->ws_bytes);
    (void)device_free(ix->device, ix->io, ix->io_bytes);
    (void)device_free(ix->device, ix->slots.p, ix->slots.bytes);
    (void)device_free(ix->device, ix->gathered.p, ix->gathered.bytes);
    if (ix->d_signs) (void)hipFree(ix->d_signs);      // (the other tables too)
    {
        DevicePool &pool = g_pool[ix->device];
        std::unique_lock<std::mutex> lock(pool.mu);
        (ix->newer ? ix->newer->older : pool.newest) = ix->older;
        if (ix->older) ix->older->newer = ix->newer;
        pool.ahead -= ix->ahead;
        const bool last = --pool.indexes == 0;
        const auto blocks = last ? pool.empty() : decltype(pool.blocks){};
        void *staged[DevicePool::kStaged] = {};
        for (int i = 0; i < DevicePool::kStaged; ++i)
            if (last && !pool.staged[i].in_use) { staged[i] = pool.staged[i].p; pool.staged[i] = tv_spare{}; }
        uint8_t *pinned[DevicePool::kPinned];
        int n_pinned = 0;
        for (tv_pinned &b : pool.pinned)
            if (last && !b.lent && b.host) { pinned[n_pinned++] = b.host; b = tv_pinned{}; }
        lock.unlock();
        free_blocks(blocks);
        for (void *p : staged) if (p) (void)hipFree(p);
        for (int i = 0; i < n_pinned; ++i) (void)hipHostFree(pinned[i]);
    }
    if (ix->h_flags) (void)hipHostFree(ix->h_flags);
    if (ix->events_ready)
        for (int i = 0; i < tv::kTimedLaunches; ++i) {
            (void)hipEventDestroy(ix->ev_start[i]);
            (void)hipEventDestroy(ix->ev_stop[i]);
        }
    if (ix->stream) (void)hipStreamDestroy(ix->stream);
    delete ix;
    return TV_OK;
}

int tv_index_set_tables(tv_index *ix, const float *signs, const uint32_t *perms, const float *centroids) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    const size_t dim = size_t(ix->geo.dim);
    if (signs) ix->rot.signs.assign(signs, signs + 2 * dim);
    if (perms) {
        for (size_t i = 0; i < 2 * dim; ++i) if (perms[i] >= dim) return TV_ERR_BAD_ARGUMENT;
        ix->rot.perms.assign(perms, perms + 2 * dim);
    }
    if (centroids) {
        ix->cb.centroids.assign(centroids, centroids + (size_t(1) << ix->geo.bits));
        for (size_t i = 0; i + 1 < ix->cb.centroids.size(); ++i)
            ix->cb.boundaries[i] = (ix->cb.centroids[i] + ix->cb.centroids[i + 1]) * 0.5f;
        derive_levels(ix);
    }
    TableImage t;
    lay_out_tables(ix->rot, t);
    const int rc = upload_tables(ix, t);
    if (rc == TV_OK) TV_HIP(hipStreamSynchronize(ix->stream));
    return rc;
}

int tv_index_set_calibration(tv_index *ix, const float *shift, const float *scale) {
    if (!ix || (shift == nullptr) != (scale == nullptr)) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    const size_t dim = size_t(ix->geo.dim);
    if (!shift) { ix->tq_shift.clear(); ix->tq_scale.clear(); return TV_OK; }
    std::unique_ptr<float[]> inverse(new (std::nothrow) float[dim]);      // (the encoder's, behind the scales)
    if (!inverse) { g_last_error = "out of memory"; return TV_ERR_BAD_ARGUMENT; }
    for (size_t j = 0; j < dim; ++j) inverse[j] = 1.0f / scale[j];
    ix->tq_shift.assign(shift, shift + dim);
    ix->tq_scale.assign(scale, scale + dim);
    TV_HIP(hipMemcpyAsync(ix->d_tq_shift, shift, dim * sizeof(float), hipMemcpyHostToDevice, ix->stream));
    TV_HIP(hipMemcpyAsync(ix->d_tq_scale, scale, dim * sizeof(float), hipMemcpyHostToDevice, ix->stream));
    TV_HIP(hipMemcpyAsync(ix->d_tq_scale + dim, inverse.get(), dim * sizeof(float), hipMemcpyHostToDevice, ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    return TV_OK;
}

int tv_index_set_score_mode(tv_index *ix, int mode) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    if (mode != TV_SCORE_AUTO && mode != TV_SCORE_L_SCALAR && mode != TV_SCORE_L_CLASSIC && mode != TV_SCORE_L_U32 && mode != TV_SCORE_P)
        return TV_ERR_BAD_ARGUMENT;
    if (mode == TV_SCORE_P && ix->geo.bits != 4) { g_last_error = "score mode P needs 4-bit codes"; return TV_ERR_BAD_ARGUMENT; }
    std::lock_guard<std::mutex> lock(ix->mu);
    ix->score_mode = mode;
    return TV_OK;
}

int tv_index_get_tables(const tv_index *ix, float *signs, uint32_t *perms, float *centroids, float *boundaries) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    if (signs) std::memcpy(signs, ix->rot.signs.data(), ix->rot.signs.size() * sizeof(float));
    if (perms) std::memcpy(perms, ix->rot.perms.data(), ix->rot.perms.size() * sizeof(uint32_t));
    if (centroids) std::memcpy(centroids, ix->cb.centroids.data(), ix->cb.centroids.size() * sizeof(float));
    if (boundaries) std::memcpy(boundaries, ix->cb.boundaries.data(), ix->cb.boundaries.size() * sizeof(float));
    return TV_OK;
}

int tv_index_upload_seq(tv_index *ix, const uint8_t *seq_codes, size_t n_vectors, const float *scales) {
    if (!ix || (n_vectors && (!seq_codes || !scales))) return TV_ERR_BAD_ARGUMENT;
    if (n_vectors >= (size_t(1) << 31)) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    ix->n = 0;
    int rc = ensure_capacity(ix, n_vectors);
    if (rc != TV_OK) return rc;
    const tv::Geometry &g = ix->geo;
    const size_t n_blocks = (n_vectors + tv::kVecBlock - 1) / tv::kVecBlock;
    const size_t seq_block = size_t(g.G) * tv::kVecBlock;
    rc = clear_tail_blocks(ix, n_blocks);
    if (rc != TV_OK) return rc;
    // stage the sequential-blocked bytes through the workspace in slices
    const size_t slice_blocks = std::max<size_t>(1, (size_t(256) << 20) / seq_block);
    rc = ensure_workspace(ix, std::min(n_blocks, slice_blocks) * seq_block + 256);
    if (rc != TV_OK) return rc;
    for (size_t b0 = 0; b0 < n_blocks; b0 += slice_blocks) {
        const size_t nb = std::min(slice_blocks, n_blocks - b0);
        TV_HIP(hipMemcpyAsync(ix->ws, seq_codes + b0 * seq_block, nb * seq_block, hipMemcpyHostToDevice, ix->stream));
        TV_HIP(tv::launch_seq_to_native(static_cast<const uint8_t *>(ix->ws), ix->d_codes, g, b0, nb, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
    }
    if (n_vectors) {
        TV_HIP(hipMemsetAsync(ix->d_scales, 0, n_blocks * tv::kVecBlock * sizeof(float), ix->stream));
        TV_HIP(hipMemcpyAsync(ix->d_scales, scales, n_vectors * sizeof(float), hipMemcpyHostToDevice, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
    }
    ix->n = n_vectors;
    return TV_OK;
}

int tv_index_upload_seq_dev(tv_index *ix, const uint8_t *d_seq_codes, size_t n_vectors, const float *d_scales) {
    if (!ix || (n_vectors && (!d_seq_codes || !d_scales))) return TV_ERR_BAD_ARGUMENT;
    if (n_vectors >= (size_t(1) << 31)) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    ix->n = 0;
    int rc = ensure_capacity(ix, n_vectors);
    if (rc != TV_OK) return rc;
    const size_t n_blocks = (n_vectors + tv::kVecBlock - 1) / tv::kVecBlock;
    const size_t seq_block = size_t(ix->geo.G) * tv::kVecBlock;
    rc = clear_tail_blocks(ix, n_blocks);
    if (rc != TV_OK) return rc;
    const size_t slice_blocks = std::max<size_t>(1, (size_t(1) << 30) / seq_block);  // keeps each grid small
    for (size_t b0 = 0; b0 < n_blocks; b0 += slice_blocks) {
        const size_t nb = std::min(slice_blocks, n_blocks - b0);
        TV_HIP(tv::launch_seq_to_native(d_seq_codes + b0 * seq_block, ix->d_codes, ix->geo, b0, nb, ix->stream));
    }
    if (n_vectors) {
        TV_HIP(hipMemsetAsync(ix->d_scales, 0, n_blocks * tv::kVecBlock * sizeof(float), ix->stream));
        TV_HIP(hipMemcpyAsync(ix->d_scales, d_scales, n_vectors * sizeof(float), hipMemcpyDeviceToDevice, ix->stream));
    }
    TV_HIP(hipStreamSynchronize(ix->stream));
    ix->n = n_vectors;
    return TV_OK;
}

int tv_index_append_rows(tv_index *ix, const uint8_t *rows, const float *scales, size_t n_new) {
    if (!ix || (n_new && (!rows || !scales))) return TV_ERR_BAD_ARGUMENT;
    if (n_new == 0) return TV_OK;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    if (ix->n + n_new >= (size_t(1) << 31)) return TV_ERR_BAD_ARGUMENT;
    int rc = ensure_capacity(ix, ix->n + n_new);
    if (rc != TV_OK) return rc;
    const tv::Geometry &g = ix->geo;
    const size_t slice = std::max<size_t>(1, (size_t(64) << 20) / size_t(g.G));
    rc = ensure_workspace(ix, std::min(n_new, slice) * size_t(g.G) + 256);
    if (rc != TV_OK) return rc;
    for (size_t r0 = 0; r0 < n_new; r0 += slice) {
        const size_t nr = std::min(slice, n_new - r0);
        TV_HIP(hipMemcpyAsync(ix->ws, rows + r0 * g.G, nr * size_t(g.G), hipMemcpyHostToDevice, ix->stream));
        TV_HIP(tv::launch_append_rows(static_cast<const uint8_t *>(ix->ws), ix->d_codes, g, ix->n + r0, nr, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
    }
    TV_HIP(hipMemcpyAsync(ix->d_scales + ix->n, scales, n_new * sizeof(float), hipMemcpyHostToDevice, ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    ix->n += n_new;
    return TV_OK;
}

// lib.rs add -> encode.rs:1418-1476 on the device, then append_lanes (pack.rs:211-233).  The rows go to slots `at` and on, which
// the caller counts among the index's.
static int encode_rows(tv_index *ix, const float *d_vectors, size_t n_new, size_t at) {
    const tv::Geometry &g = ix->geo;
    const bool cal = !ix->tq_shift.empty();
    const size_t slice = size_t(1) << 20;
    for (size_t r0 = 0; r0 < n_new; r0 += slice) {
        const size_t nr = std::min(slice, n_new - r0);
        TV_HIP(tv::launch_encode(d_vectors + r0 * size_t(g.dim), nr, at + r0, ix->d_signs, ix->d_perms,
                                 ix->packed_ok ? ix->d_packed : nullptr, cal ? ix->d_tq_shift : nullptr, cal ? ix->d_tq_scale : nullptr,
                                 ix->cb.centroids.data(), ix->cb.boundaries.data(), g, ix->rot.block,
                                 ix->rot.inv_sqrt_block, ix->d_codes, ix->d_scales, nullptr, ix->device, ix->stream));
    }
    TV_HIP(hipStreamSynchronize(ix->stream));
    return TV_OK;
}

static int clear_slots(tv_index *ix, size_t end);

int tv_index_add_dev(tv_index *ix, const float *d_vectors, size_t n_new) {
    if (!ix || (n_new && !d_vectors)) return TV_ERR_BAD_ARGUMENT;
    if (n_new == 0) return TV_OK;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    if (ix->n + n_new >= (size_t(1) << 31)) return TV_ERR_BAD_ARGUMENT;
    Outgrown outgrown(ix);
    int rc = ensure_capacity(ix, ix->n + n_new, outgrown, ix->packed_ok);
    if (rc != TV_OK) return rc;
    rc = encode_rows(ix, d_vectors, n_new, ix->n);      // (waits for the stream)
    if (rc == TV_OK) {
        const hipError_t e = outgrown.release();
        if (e != hipSuccess) rc = fail_hip(e, "device_free(outgrown rows)");
    }
    if (rc == TV_OK) ix->n += n_new;      // (an add that fails adds nothing)
    else (void)clear_slots(ix, ix->n + n_new);
    return rc;
}

// Rows on their way to the device, checked as they pass through pinned memory, a few megabytes at a time: each of up
// to four threads fills its piece while the others' are copied (614 MB: 13 ms, at the rate of the bus; fresh pageable memory 20 to 39, and
// a pass over it for the check).  *bad: a value was refused; the rest need not have arrived.  Met with the index's lock held.
static int stage_rows(tv_index *ix, const float *rows, size_t values, float *d_rows, bool *bad) {
    constexpr size_t kPiece = (size_t(4) << 20) / sizeof(float), kThreads = 4;
    *bad = false;
    const size_t pieces = (values + kPiece - 1) / kPiece, threads = std::min<size_t>(kThreads, pieces);
    PinnedLoan loan(ix->device, threads * std::min(kPiece, values) * sizeof(float));
    if (!loan.b) {
        *bad = tv_validate_queries(rows, values, 1, nullptr) != TV_OK;
        if (!*bad) TV_HIP(hipMemcpyAsync(d_rows, rows, values * sizeof(float), hipMemcpyHostToDevice, ix->stream));
        return TV_OK;
    }
    std::atomic<size_t> next{0};
    std::atomic<bool> refused{false}, failed{false};
    in_parts(threads, 1, [&](size_t lo, size_t hi) {
        if (lo == hi) return;
        if (hipSetDevice(ix->device) != hipSuccess) { failed = true; return; }
        float *mine = reinterpret_cast<float *>(loan.b->host) + lo * kPiece;
        for (size_t p; !refused && !failed && (p = next.fetch_add(1)) < pieces;) {
            const size_t at = p * kPiece, m = std::min(kPiece, values - at);
            if (copy_checked(mine, rows + at, m)) { refused = true; break; }
            // (the wait is for whatever the threads have enqueued so far, this piece among it)
            if (hipMemcpyAsync(d_rows + at, mine, m * sizeof(float), hipMemcpyHostToDevice, ix->stream) != hipSuccess ||
                hipStreamSynchronize(ix->stream) != hipSuccess) failed = true;
        }
    });
    *bad = refused;
    if (failed) { g_last_error = "host to device copy failed"; return TV_ERR_HIP; }
    return TV_OK;
}

// Device bytes into fresh host memory, the other way round: threads share the copies out of pinned memory, whose
// page faults are most of the time (77 MB: one thread 18 ms, untouched; 4.4 with the pages touched by eight before).
static int fetch_bytes(tv_index *ix, const uint8_t *d_from, uint8_t *to, size_t bytes) {
    constexpr size_t kPiece = size_t(2) << 20;
    const size_t pieces = (bytes + kPiece - 1) / kPiece, threads = std::min(kMaxParts, pieces);
    PinnedLoan loan(ix->device, threads * std::min(kPiece, bytes));
    if (bytes == 0) return TV_OK;
    if (!loan.b) {
        touch_pages(to, bytes);
        TV_HIP(hipMemcpyAsync(to, d_from, bytes, hipMemcpyDeviceToHost, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
        return TV_OK;
    }
    std::atomic<size_t> next{0};
    std::atomic<bool> failed{false};
    in_parts(threads, 1, [&](size_t lo, size_t hi) {
        if (lo == hi) return;
        if (hipSetDevice(ix->device) != hipSuccess) { failed = true; return; }
        uint8_t *mine = loan.b->host + lo * kPiece;
        for (size_t p; !failed && (p = next.fetch_add(1)) < pieces;) {
            const size_t at = p * kPiece, m = std::min(kPiece, bytes - at);
            if (hipMemcpyAsync(mine, d_from + at, m, hipMemcpyDeviceToHost, ix->stream) != hipSuccess ||
                hipStreamSynchronize(ix->stream) != hipSuccess) { failed = true; break; }
            std::memcpy(to + at, mine, m);
        }
    });
    if (failed) { g_last_error = "device to host copy failed"; return TV_ERR_HIP; }
    return TV_OK;
}

// Slots from the index's last row up to `end` are cleared, as if no rows had ever gone there.
static int clear_slots(tv_index *ix, size_t end) {
    const tv::Geometry &g = ix->geo;
    const size_t first = ix->n, block = (first + tv::kVecBlock - 1) / tv::kVecBlock, end_block = (end + tv::kVecBlock - 1) / tv::kVecBlock;
    if (end <= first) return TV_OK;
    const size_t lanes = std::min(end, block * tv::kVecBlock) - first;      // in a block that holds earlier rows
    if (lanes) {
        int rc = ensure_workspace(ix, lanes * size_t(g.G) + 256);
        if (rc != TV_OK) return rc;
        TV_HIP(hipMemsetAsync(ix->ws, 0, lanes * size_t(g.G), ix->stream));
        TV_HIP(tv::launch_append_rows(static_cast<const uint8_t *>(ix->ws), ix->d_codes, g, first, lanes, ix->stream));
    }
    TV_HIP(hipMemsetAsync(ix->d_scales + first, 0, (end - first) * sizeof(float), ix->stream));
    if (end_block > block) TV_HIP(hipMemsetAsync(ix->d_codes + block * g.block_bytes(), 0, (end_block - block) * g.block_bytes(), ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    return TV_OK;
}

int tv_index_add(tv_index *ix, const float *vectors, size_t n_new) {
    if (!ix || (n_new && !vectors)) return TV_ERR_BAD_ARGUMENT;
    if (n_new == 0) return TV_OK;
    const size_t dim = size_t(ix->geo.dim);
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    if (ix->n + n_new >= (size_t(1) << 31)) return TV_ERR_BAD_ARGUMENT;
    int rc = ensure_capacity(ix, ix->n + n_new);
    if (rc != TV_OK) return rc;
    const size_t slice = std::max<size_t>(1, (size_t(256) << 20) / (dim * sizeof(float)));
    rc = ensure_workspace(ix, std::min(n_new, slice) * dim * sizeof(float) + 256);
    if (rc != TV_OK) return rc;
    for (size_t r0 = 0; r0 < n_new; r0 += slice) {
        const size_t nr = std::min(slice, n_new - r0);
        bool bad = false;
        rc = stage_rows(ix, vectors + r0 * dim, nr * dim, static_cast<float *>(ix->ws), &bad);
        if (rc == TV_OK && !bad) rc = encode_rows(ix, static_cast<const float *>(ix->ws), nr, ix->n + r0);
        if (rc != TV_OK || bad) {      // nothing is added: the index's rows are counted once the last slice is there
            const int cleared = clear_slots(ix, ix->n + r0 + (bad ? 0 : nr));
            if (rc == TV_OK) rc = cleared;
        }
        if (rc != TV_OK) return rc;
        if (bad) {      // the same predicate as for queries (encode.rs:76-83)
            size_t at = r0 * dim;
            (void)tv_validate_queries(vectors, n_new * dim, int(dim), &at);
            g_last_error = "vector " + std::to_string(at / dim) + " holds a non-finite or too large value";
            return TV_ERR_INVALID_QUERY_VALUE;
        }
    }
    ix->n += n_new;
    return TV_OK;
}

// TurboQuantIndex::calibrate (lib.rs:2599) on an empty index: rotate the normalised sample on
// the device (encode.rs:406-458), fit on the host (encode.rs:737-857), commit the pair.
int tv_index_calibrate(tv_index *ix, const float *sample, size_t n) {
    if (!ix || !sample) return TV_ERR_BAD_ARGUMENT;
    if (n < 2) { g_last_error = "calibration needs at least 2 rows"; return TV_ERR_BAD_ARGUMENT; }   // encode.rs:395
    const size_t dim = size_t(ix->geo.dim);
    size_t bad = 0;
    int rc = tv_validate_queries(sample, n * dim, ix->geo.dim, &bad);
    if (rc != TV_OK) {
        g_last_error = "sample row " + std::to_string(bad / dim) + " holds a non-finite or too large value";
        return rc;
    }
    std::vector<float> rotated(n * dim);
    {
        std::lock_guard<std::mutex> lock(ix->mu);
        if (ix->n != 0) {
            g_last_error = "calibrate on a populated index (re-encoding stored rows) is not supported";
            return TV_ERR_BAD_ARGUMENT;
        }
        TV_HIP(hipSetDevice(ix->device));
        const size_t slice = std::max<size_t>(1, (size_t(128) << 20) / (dim * sizeof(float)));
        rc = ensure_workspace(ix, 2 * std::min(n, slice) * dim * sizeof(float) + 512);
        if (rc != TV_OK) return rc;
        float *d_in = static_cast<float *>(ix->ws);
        float *d_out = d_in + std::min(n, slice) * dim;
        for (size_t r0 = 0; r0 < n; r0 += slice) {
            const size_t nr = std::min(slice, n - r0);
            TV_HIP(hipMemcpyAsync(d_in, sample + r0 * dim, nr * dim * sizeof(float), hipMemcpyHostToDevice, ix->stream));
            TV_HIP(tv::launch_encode(d_in, nr, 0, ix->d_signs, ix->d_perms, nullptr, nullptr, nullptr, ix->cb.centroids.data(),
                                     ix->cb.boundaries.data(), ix->geo, ix->rot.block, ix->rot.inv_sqrt_block,
                                     nullptr, nullptr, d_out, ix->device, ix->stream));
            TV_HIP(hipMemcpyAsync(rotated.data() + r0 * dim, d_out, nr * dim * sizeof(float), hipMemcpyDeviceToHost, ix->stream));
            TV_HIP(hipStreamSynchronize(ix->stream));
        }
    }
    std::vector<float> shift(dim), scale(dim);
    tv::fit_tqplus(rotated.data(), n, ix->geo.dim, ix->cb.centroids, shift.data(), scale.data());
    return tv_index_set_calibration(ix, shift.data(), scale.data());
}

int tv_index_get_calibration(const tv_index *ix, float *shift, float *scale, size_t *n_calib) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    if (n_calib) *n_calib = ix->tq_shift.size();
    if (shift && !ix->tq_shift.empty()) std::memcpy(shift, ix->tq_shift.data(), ix->tq_shift.size() * sizeof(float));
    if (scale && !ix->tq_scale.empty()) std::memcpy(scale, ix->tq_scale.data(), ix->tq_scale.size() * sizeof(float));
    return TV_OK;
}

int tv_index_swap_remove(tv_index *ix, size_t idx) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    if (idx >= ix->n) return TV_ERR_INDEX_OUT_OF_RANGE;
    TV_HIP(hipSetDevice(ix->device));
    TV_HIP(tv::launch_move_lane(ix->d_codes, ix->d_scales, ix->geo, ix->n - 1, idx, ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    ix->n -= 1;
    return TV_OK;
}

// The index's lock is held by the caller.
static int download_seq_locked(tv_index *ix, uint8_t *seq_out, float *scales_out) {
    TV_HIP(hipSetDevice(ix->device));
    const tv::Geometry &g = ix->geo;
    const size_t n_blocks = (ix->n + tv::kVecBlock - 1) / tv::kVecBlock;
    const size_t seq_block = size_t(g.G) * tv::kVecBlock;
    if (seq_out && n_blocks) {
        const size_t slice_blocks = std::max<size_t>(1, (size_t(256) << 20) / seq_block);
        int rc = ensure_workspace(ix, std::min(n_blocks, slice_blocks) * seq_block + 256);
        if (rc != TV_OK) return rc;
        for (size_t b0 = 0; b0 < n_blocks; b0 += slice_blocks) {
            const size_t nb = std::min(slice_blocks, n_blocks - b0);
            TV_HIP(tv::launch_native_to_seq(ix->d_codes, static_cast<uint8_t *>(ix->ws), g, b0, nb, seq_block, nullptr, ix->stream));
            TV_HIP(hipMemcpyAsync(seq_out + b0 * seq_block, ix->ws, nb * seq_block, hipMemcpyDeviceToHost, ix->stream));
            TV_HIP(hipStreamSynchronize(ix->stream));
        }
    }
    if (scales_out && ix->n) {
        TV_HIP(hipMemcpyAsync(scales_out, ix->d_scales, ix->n * sizeof(float), hipMemcpyDeviceToHost, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
    }
    return TV_OK;
}

int tv_index_download_seq(const tv_index *cix, uint8_t *seq_out, float *scales_out) {
    tv_index *ix = const_cast<tv_index *>(cix);
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    return download_seq_locked(ix, seq_out, scales_out);
}

size_t tv_index_len(const tv_index *ix) { return ix ? ix->n : 0; }
int tv_index_dim(const tv_index *ix) { return ix ? ix->geo.dim : 0; }
int tv_index_bits(const tv_index *ix) { return ix ? ix->geo.bits : 0; }

int tv_validate_queries(const float *queries, size_t len, int dim, size_t *bad_index) {
    if (dim <= 0 || len % size_t(dim) != 0) return TV_ERR_QUERY_BUFFER_NOT_MULTIPLE_OF_DIM;
    // A run of values at a time, without a branch per value: |x| < 1e16 and not NaN is an unsigned compare
    // of the bits without the sign.
    constexpr size_t kRun = 4096;
    std::atomic<size_t> first_bad{len};
    in_parts(len, size_t(1) << 20, [&](size_t lo, size_t hi) {
        for (size_t r = lo; r < hi && r < first_bad.load(std::memory_order_relaxed); r += kRun) {
            const size_t e = std::min(r + kRun, hi);
            auto bad = [&](size_t i) {
                uint32_t u;
                std::memcpy(&u, queries + i, 4);
                return (u & 0x7fffffffu) >= kTooLargeBits;
            };
            uint32_t any = 0;
            for (size_t i = r; i < e; ++i) any |= uint32_t(bad(i));
            if (!any) continue;
            size_t i = r;
            while (i < e && !bad(i)) ++i;
            if (i == e) continue;      // (the caller's array: another thread has overwritten the value since)
            size_t seen = first_bad.load();
            while (i < seen && !first_bad.compare_exchange_weak(seen, i)) {}
            return;
        }
    });
    if (first_bad.load() == len) return TV_OK;
    if (bad_index) *bad_index = first_bad.load();
    return TV_ERR_INVALID_QUERY_VALUE;
}

int tv_pack_mask(const uint8_t *mask_bytes, size_t n, uint64_t *words_out, size_t *n_allowed) {
    if ((n && !mask_bytes) || !words_out) return TV_ERR_BAD_ARGUMENT;
    size_t allowed = 0;
    for (size_t w = 0; w * 64 < n; ++w) {
        uint64_t word = 0;
        const size_t lim = std::min<size_t>(64, n - w * 64);
        size_t bit = 0;
        for (; bit + 8 <= lim; bit += 8) {      // eight bytes at a time: 1 where a byte is not zero, the ones gathered by a multiplication
            uint64_t x;
            std::memcpy(&x, mask_bytes + w * 64 + bit, 8);
            x = ((((x & 0x7f7f7f7f7f7f7f7full) + 0x7f7f7f7f7f7f7f7full) | x) >> 7) & 0x0101010101010101ull;
            word |= (x * 0x0102040810204080ull >> 56) << bit;
        }
        for (; bit < lim; ++bit) word |= uint64_t(mask_bytes[w * 64 + bit] != 0) << bit;
        allowed += size_t(__builtin_popcountll(word));
        words_out[w] = word;
    }
    if (n_allowed) *n_allowed = allowed;
    return TV_OK;
}

int tv_search_dev(tv_index *ix, const float *d_queries, size_t nq, size_t k, const uint64_t *d_mask_words,
                  size_t n_allowed, float *d_out_scores, int64_t *d_out_indices, size_t *out_k_eff) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    tv_request r;
    r.host = false;
    r.q = d_queries; r.nq = nq; r.k = k;
    r.mask = d_mask_words; r.mask_arg = d_mask_words ? n_allowed : 0;
    r.out_s = d_out_scores; r.out_i = d_out_indices;
    const int rc = search_merged(ix, r);
    if (out_k_eff) *out_k_eff = r.k_eff;
    return rc;
}

size_t tv_noalloc_scratch_bytes(void) { return kScratchBytes; }

int tv_search_dev_noalloc(tv_index *ix, const float *d_queries, size_t nq, size_t k, const uint64_t *d_mask_words,
                          size_t n_allowed, float *d_out_scores, int64_t *d_out_indices, size_t *out_k_eff) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    if (!d_mask_words) n_allowed = ix->n;
    const size_t k_eff = std::min(std::min(k, ix->n), n_allowed);
    // What the search may carve, worst case: the sampled path's chunk, and the exact path a query
    // falls back to when its candidates overflow.  Refused up front when that exceeds the array.
    // (The matrix-unit scan of u8-LUT batches pads a call to 32 queries, the sixteen-query passes to 16:
    // a call that only the smaller working set fits takes those.)
    auto carve = [&] {
        if (k_eff == 0 || nq == 0) return size_t(0);
        const size_t cq = std::min(nq, kChunkQueries);    // the exact path works in chunks of this size throughout
        const size_t exact = robust_need(ix, cq, k_eff);
        return k_eff <= size_t(tv::kMaxSampledK) && !ix->force_robust ? std::max(exact, sampled_need_worst(ix, nq)) : exact;
    };
    ix->ws_fixed = true;      // (what is carved depends on it)
    size_t need = carve();
    if (need > kScratchBytes) {
        ix->no_lut_mx = true;
        need = carve();
    }
    if (need > kScratchBytes) {
        ix->no_lut_mx = false;
        ix->ws_fixed = false;
        g_last_error = "tv_search_dev_noalloc: " + std::to_string(nq) + " queries, k=" + std::to_string(k) + " over " +
                       std::to_string(ix->n) + " rows may need " + std::to_string(need) +
                       " bytes of scratch; the fixed buffer holds " + std::to_string(kScratchBytes) +
                       " (fewer queries per call; k <= 32 on a large index)";
        return TV_ERR_BAD_ARGUMENT;
    }
    std::lock_guard<std::mutex> device_lock(g_scratch[ix->device].in_use);
    void *own_ws = ix->ws;
    const size_t own_bytes = ix->ws_bytes;
    ix->ws = ix->scratch;
    ix->ws_bytes = kScratchBytes;
    const int rc = search_device(ix, d_queries, nq, k, d_mask_words, n_allowed, kLiveUnknown, d_out_scores, d_out_indices, out_k_eff);
    ix->ws = own_ws;
    ix->ws_bytes = own_bytes;
    ix->ws_fixed = false;
    ix->no_lut_mx = false;
    return rc;
}

// bad_index: values are checked, on the snapshot of them that is searched (null: they are not).
static int search_host(tv_index *ix, const float *queries, size_t nq, size_t k, const uint64_t *mask_words,
                       size_t n_mask_words, float *out_scores, int64_t *out_indices, size_t *out_k_eff, size_t *bad_index) {
    if (!ix || (nq && !queries)) return TV_ERR_BAD_ARGUMENT;
    const size_t dim = size_t(ix->geo.dim), values = nq * dim;
    tv_request r;
    r.host = true;
    r.q = queries; r.nq = nq; r.k = k;
    r.mask = mask_words; r.mask_arg = mask_words ? n_mask_words : 0;
    r.out_s = out_scores; r.out_i = out_indices;
    size_t need = 0, s_at = 0, i_at = 0, m_at = 0;
    // (no product below overflows; a mask of another length is refused when the call is served, and not read)
    if (nq != 0 && k != 0 && nq <= (kPinnedLargest >> 2) && k <= (kPinnedLargest >> 2) &&
        (!mask_words || n_mask_words == (tv_index_len(ix) + 63) / 64)) {
        s_at = round_up(values * sizeof(float), 256);
        i_at = s_at + round_up(nq * k * sizeof(float), 256);
        m_at = i_at + round_up(nq * k * sizeof(int64_t), 256);
        need = m_at + r.mask_arg * sizeof(uint64_t);
    }
    if (need != 0) TV_HIP(hipSetDevice(ix->device));
    PinnedLoan loan(ix->device, need != 0 ? need : kPinnedLargest + 1);
    std::unique_ptr<float[]> own;      // where no block was lent, the snapshot of the values to be checked
    auto snapshot = [&](float *to) -> int {
        std::atomic<bool> bad{false};
        in_parts(values, size_t(1) << 18, [&](size_t lo, size_t hi) {
            if (copy_checked(to + lo, queries + lo, hi - lo)) bad.store(true, std::memory_order_relaxed);
        });
        r.q = to;
        return bad_index && bad.load() ? tv_validate_queries(to, values, int(dim), bad_index) : TV_OK;
    };
    int rc = TV_OK;
    if (loan.b) {
        rc = snapshot(reinterpret_cast<float *>(loan.b->host));
        if (rc != TV_OK) return rc;
        if (mask_words) {
            std::memcpy(loan.b->host + m_at, mask_words, r.mask_arg * sizeof(uint64_t));
            r.staged_mask = reinterpret_cast<uint64_t *>(loan.b->host + m_at);
        }
        r.out_s = reinterpret_cast<float *>(loan.b->host + s_at);
        r.out_i = reinterpret_cast<int64_t *>(loan.b->host + i_at);
        r.dev_q = reinterpret_cast<const float *>(loan.b->dev);
        r.dev_s = reinterpret_cast<float *>(loan.b->dev + s_at);
        r.dev_i = reinterpret_cast<int64_t *>(loan.b->dev + i_at);
    } else if (bad_index && values != 0) {
        own.reset(new (std::nothrow) float[values]);
        if (!own) { g_last_error = "no memory for a copy of the queries"; return TV_ERR_BAD_ARGUMENT; }
        rc = snapshot(own.get());
        if (rc != TV_OK) return rc;
    }
    rc = search_merged(ix, r);
    if (out_k_eff) *out_k_eff = r.k_eff;
    if (rc == TV_OK && loan.b && r.k_eff != 0) {
        std::memcpy(out_scores, r.out_s, nq * r.k_eff * sizeof(float));
        std::memcpy(out_indices, r.out_i, nq * r.k_eff * sizeof(int64_t));
    }
    return rc;
}

int tv_search(tv_index *ix, const float *queries, size_t nq, size_t k, const uint64_t *mask_words,
              size_t n_mask_words, float *out_scores, int64_t *out_indices, size_t *out_k_eff) {
    return search_host(ix, queries, nq, k, mask_words, n_mask_words, out_scores, out_indices, out_k_eff, nullptr);
}

int tv_search_checked(tv_index *ix, const float *queries, size_t nq, size_t k, const uint64_t *mask_words,
                      size_t n_mask_words, float *out_scores, int64_t *out_indices, size_t *out_k_eff, size_t *bad_index) {
    size_t unused = 0;
    return search_host(ix, queries, nq, k, mask_words, n_mask_words, out_scores, out_indices, out_k_eff, bad_index ? bad_index : &unused);
}

int tv_debug_scan(tv_index *ix, const float *queries, size_t nq, int32_t *acc_out, float *scores_out) {
    if (!ix || (nq && !queries)) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    const size_t n = ix->n;
    if (n == 0 || nq == 0) return TV_OK;
    const tv::Geometry &g = ix->geo;
    const int mode = effective_mode(ix);
    const bool mode_p = mode == TV_SCORE_P;
    const size_t tile_q = mode_p ? size_t(tv::kQTile) : size_t(lut_tile_q(ix, 1));
    for (size_t q0 = 0; q0 < nq; q0 += tile_q) {
        const size_t cq = std::min<size_t>(tile_q, nq - q0);
        size_t need = prepare_bytes(ix, cq) + round_up(cq * g.dim * 4, 256) + 2 * round_up(cq * n * 4, 256) + 65536;
        int rc = ensure_workspace(ix, need);
        if (rc != TV_OK) return rc;
        Arena ar;
        ar.base = static_cast<uint8_t *>(ix->ws);
        float *d_q = ar.take<float>(cq * g.dim);
        int32_t *d_acc = ar.take<int32_t>(cq * n);
        float *d_sc = ar.take<float>(cq * n);
        TV_HIP(hipMemcpyAsync(d_q, queries + q0 * g.dim, cq * g.dim * sizeof(float), hipMemcpyHostToDevice, ix->stream));
        Prepared pq;
        rc = prepare_queries(ix, ar, d_q, cq, pq);
        if (rc != TV_OK) return rc;
        tv::ScanArgs a;
        fill_scan_args(ix, a);
        a.tables = pq.d_tables;
        a.qscale = pq.d_qscale;
        a.qbias = pq.d_qbias;
        a.nq_tile = int(cq);
        a.k = 1;
        a.acc_out = d_acc;
        a.score_out = d_sc;
        const int grid = tv::scan_grid_blocks(ix->device, mode_p, g.nch, 1, int(tile_q));
        if (mode_p) TV_HIP(tv::launch_scan_p4(a, grid, tv::kModeDump, ix->stream));
        else TV_HIP(tv::launch_scan_lut(a, grid, tv::kModeDump, ix->stream));
        if (acc_out) TV_HIP(hipMemcpyAsync(acc_out + q0 * n, d_acc, cq * n * 4, hipMemcpyDeviceToHost, ix->stream));
        if (scores_out) TV_HIP(hipMemcpyAsync(scores_out + q0 * n, d_sc, cq * n * 4, hipMemcpyDeviceToHost, ix->stream));
        TV_HIP(hipStreamSynchronize(ix->stream));
    }
    return TV_OK;
}

int tv_debug_prepare(tv_index *ix, const float *queries, size_t nq, float *q_rot_out, float *scale_out,
                     float *bias_out) {
    if (!ix || (nq && !queries)) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    if (nq == 0) return TV_OK;
    const tv::Geometry &g = ix->geo;
    int rc = ensure_workspace(ix, prepare_bytes(ix, nq) + round_up(nq * g.dim * 4, 256) + 65536);
    if (rc != TV_OK) return rc;
    Arena ar;
    ar.base = static_cast<uint8_t *>(ix->ws);
    float *d_q = ar.take<float>(nq * g.dim);
    TV_HIP(hipMemcpyAsync(d_q, queries, nq * g.dim * sizeof(float), hipMemcpyHostToDevice, ix->stream));
    Prepared pq;
    rc = prepare_queries(ix, ar, d_q, nq, pq, true, true);
    if (rc != TV_OK) return rc;
    if (q_rot_out) TV_HIP(hipMemcpyAsync(q_rot_out, pq.d_qrot, nq * g.dim * 4, hipMemcpyDeviceToHost, ix->stream));
    if (scale_out) TV_HIP(hipMemcpyAsync(scale_out, pq.d_qscale, nq * 4, hipMemcpyDeviceToHost, ix->stream));
    if (bias_out) TV_HIP(hipMemcpyAsync(bias_out, pq.d_qbias, nq * 4, hipMemcpyDeviceToHost, ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    return TV_OK;
}

int tv_host_rotation_tables(int dim, float *signs, uint32_t *perms, int *block, float *inv_sqrt_block) {
    if (dim <= 0 || dim % 8 != 0 || dim > 16384) return TV_ERR_BAD_ARGUMENT;
    const tv::RotationTables t = tv::make_rotation_tables(dim);
    if (signs) std::memcpy(signs, t.signs.data(), t.signs.size() * sizeof(float));
    if (perms) std::memcpy(perms, t.perms.data(), t.perms.size() * sizeof(uint32_t));
    if (block) *block = t.block;
    if (inv_sqrt_block) *inv_sqrt_block = t.inv_sqrt_block;
    return TV_OK;
}

int tv_host_codebook(int bits, int dim, float *boundaries, float *centroids) {
    if (bits < 2 || bits > 4 || dim < 8 || dim > 16384) return TV_ERR_BAD_ARGUMENT;
    const tv::Codebook cb = tv::make_codebook(bits, dim);
    if (boundaries) std::memcpy(boundaries, cb.boundaries.data(), cb.boundaries.size() * sizeof(float));
    if (centroids) std::memcpy(centroids, cb.centroids.data(), cb.centroids.size() * sizeof(float));
    return TV_OK;
}

size_t tv_host_snapshot_len(int format, int dim, int bits, int kind, size_t n_calib, size_t n) {
    if (format != 6 && format != 7) return 0;
    return tv::snapshot_len(format, dim, bits, kind, n_calib, n);
}

int tv_host_snapshot_compose(int format, int dim, int bits, int kind, const float *boundaries, const float *centroids,
                             size_t n_calib, const float *shift, const float *scale,
                             const uint8_t *seq, size_t n, const float *scales, const uint64_t *ids,
                             uint8_t *out) {
    if (format != 6 && format != 7) return TV_ERR_BAD_ARGUMENT;
    if (bits < 2 || bits > 4 || dim <= 0 || dim % 8 != 0 || dim > 16384 || kind < 0 || kind > 1) return TV_ERR_BAD_ARGUMENT;
    if (!boundaries || !centroids || !out || (n && (!seq || !scales)) || (kind == 1 && n && !ids)) return TV_ERR_BAD_ARGUMENT;
    if ((n_calib != 0 && n_calib != size_t(dim)) || (n_calib && (!shift || !scale))) return TV_ERR_BAD_ARGUMENT;
    const tv::SnapshotParts s{kind, dim, bits, boundaries, centroids, n_calib, shift, scale, seq, n, scales, ids};
    tv::snapshot_compose(format, s, out);
    return TV_OK;
}

int tv_host_snapshot_info(const uint8_t *bytes, size_t len, int *format, int *kind, int *dim, int *bits,
                          size_t *n_calib, size_t *n) {
    if (!bytes) return TV_ERR_BAD_ARGUMENT;
    tv::SnapshotInfo info;
    const std::string why = tv::snapshot_parse(bytes, len, info);
    if (!why.empty()) { g_last_error = why; return TV_ERR_BAD_IMAGE; }
    if (format) *format = info.format;
    if (kind) *kind = info.kind;
    if (dim) *dim = info.dim;
    if (bits) *bits = info.bits;
    if (n_calib) *n_calib = info.n_calib;
    if (n) *n = info.n;
    return TV_OK;
}

int tv_host_snapshot_extract(const uint8_t *bytes, size_t len, float *boundaries, float *centroids,
                             float *shift, float *scale, uint8_t *seq, float *scales, uint64_t *ids) {
    if (!bytes) return TV_ERR_BAD_ARGUMENT;
    tv::SnapshotInfo info;
    const std::string why = tv::snapshot_parse(bytes, len, info);
    if (!why.empty()) { g_last_error = why; return TV_ERR_BAD_IMAGE; }
    const size_t nl = size_t(1) << info.bits;
    if (boundaries) std::memcpy(boundaries, bytes + info.boundaries_at, (nl - 1) * 4);
    if (centroids) std::memcpy(centroids, bytes + info.centroids_at, nl * 4);
    if (shift) std::memcpy(shift, bytes + info.shift_at, info.n_calib * 4);
    if (scale) std::memcpy(scale, bytes + info.scale_at, info.n_calib * 4);
    if (seq || scales || ids) {
        const size_t nb = (info.n + 31) / 32;
        std::vector<uint8_t> seq_tmp;
        std::vector<float> sc_tmp;
        if (!seq) { seq_tmp.resize(nb * info.row_bytes * 32); seq = seq_tmp.data(); }
        if (!scales) { sc_tmp.resize(nb * 32); scales = sc_tmp.data(); }
        tv::snapshot_extract(bytes, info, seq, scales, ids);
    }
    return TV_OK;
}

int tv_index_to_bytes(const tv_index *cix, const uint64_t *ids, int format, uint8_t *out, size_t cap, size_t *len) {
    tv_index *ix = const_cast<tv_index *>(cix);
    if (!ix || !len || (format != 6 && format != 7)) return TV_ERR_BAD_ARGUMENT;
    const int kind = ids ? 1 : 0;
    // one lock over size, download and compose: the image is of one state of the index
    std::lock_guard<std::mutex> lock(ix->mu);
    const size_t n = ix->n, n_calib = ix->tq_shift.size();
    *len = tv::snapshot_len(format, ix->geo.dim, ix->geo.bits, kind, n_calib, n);
    if (!out) return TV_OK;
    if (cap < *len) return TV_ERR_BAD_ARGUMENT;
    const size_t nb = (n + 31) / 32;
    if (format == 7) {
        // The device writes the units as the image holds them and they are copied straight to their place;
        // only the rows behind the last whole block pass through the host's composer.
        TV_HIP(hipSetDevice(ix->device));
        const tv::Geometry &g = ix->geo;
        const size_t whole = n / 32, unit = tv::snapshot_unit_len(g.dim, g.bits, kind), seq_block = size_t(g.G) * 32;
        std::vector<uint8_t> tail_seq(whole < nb ? seq_block : 0);
        float tail_scales[32] = {0};
        const size_t slice = std::max<size_t>(1, (size_t(256) << 20) / unit);
        int rc = ensure_workspace(ix, std::max(std::min(whole, slice) * unit, seq_block) + 256);
        if (rc != TV_OK) return rc;
        if (whole < nb) {
            TV_HIP(tv::launch_native_to_seq(ix->d_codes, static_cast<uint8_t *>(ix->ws), g, whole, 1, seq_block, nullptr, ix->stream));
            TV_HIP(hipMemcpyAsync(tail_seq.data(), ix->ws, seq_block, hipMemcpyDeviceToHost, ix->stream));
            TV_HIP(hipMemcpyAsync(tail_scales, ix->d_scales + whole * 32, (n - whole * 32) * sizeof(float), hipMemcpyDeviceToHost, ix->stream));
            TV_HIP(hipStreamSynchronize(ix->stream));
        }
        const tv::SnapshotParts s{kind, g.dim, g.bits, ix->cb.boundaries.data(), ix->cb.centroids.data(), n_calib,
                                  ix->tq_shift.data(), ix->tq_scale.data(), tail_seq.data(), n, tail_scales, ids ? ids + whole * 32 : nullptr};
        uint8_t *units = out + tv::snapshot_head(s, out);
        for (size_t b0 = 0; b0 < whole; b0 += slice) {
            const size_t m = std::min(slice, whole - b0);
            TV_HIP(tv::launch_native_to_seq(ix->d_codes, static_cast<uint8_t *>(ix->ws), g, b0, m, unit, ix->d_scales, ix->stream));
            rc = fetch_bytes(ix, static_cast<const uint8_t *>(ix->ws), units + b0 * unit, m * unit);
            if (rc != TV_OK) return rc;
        }
        if (ids)
            for (size_t b = 0; b < whole; ++b) std::memcpy(units + (b + 1) * unit - 32 * sizeof(uint64_t), ids + b * 32, 32 * sizeof(uint64_t));
        return TV_OK;
    }
    std::vector<uint8_t> seq(nb * size_t(ix->geo.G) * 32);
    std::vector<float> scales(n);
    int rc = download_seq_locked(ix, seq.data(), scales.data());
    if (rc != TV_OK) return rc;
    const tv::SnapshotParts s{kind, ix->geo.dim, ix->geo.bits, ix->cb.boundaries.data(), ix->cb.centroids.data(),
                              n_calib, ix->tq_shift.data(), ix->tq_scale.data(), seq.data(), n, scales.data(), ids};
    tv::snapshot_compose(format, s, out);
    return TV_OK;
}

int tv_index_from_bytes(const uint8_t *bytes, size_t len, int device, tv_index **out, uint64_t *ids_out) {
    if (!bytes || !out) return TV_ERR_BAD_ARGUMENT;
    *out = nullptr;
    tv::SnapshotInfo info;
    const std::string why = tv::snapshot_parse(bytes, len, info);
    if (!why.empty()) { g_last_error = why; return TV_ERR_BAD_IMAGE; }
    tv_index *ix = nullptr;
    int rc = tv_index_create(info.dim, info.bits, device, &ix);
    if (rc != TV_OK) return rc;
    const size_t nl = size_t(1) << info.bits;
    std::vector<float> cen(nl), sh(info.n_calib), sc(info.n_calib);
    std::memcpy(cen.data(), bytes + info.centroids_at, nl * 4);
    std::memcpy(sh.data(), bytes + info.shift_at, info.n_calib * 4);
    std::memcpy(sc.data(), bytes + info.scale_at, info.n_calib * 4);
    rc = tv_index_set_tables(ix, nullptr, nullptr, cen.data());
    if (rc == TV_OK && info.n_calib) rc = tv_index_set_calibration(ix, sh.data(), sc.data());
    if (rc == TV_OK && info.n) {
        const size_t nb = (info.n + 31) / 32;
        std::vector<uint8_t> seq(nb * info.row_bytes * 32);
        std::vector<float> scales(nb * 32);
        tv::snapshot_extract(bytes, info, seq.data(), scales.data(), ids_out);
        rc = tv_index_upload_seq(ix, seq.data(), info.n, scales.data());
    }
    if (rc != TV_OK) { tv_index_destroy(ix); return rc; }
    *out = ix;
    return TV_OK;
}

int tv_debug_stream_probe(tv_index *ix, const void *d_src, void *d_dst, size_t bytes, int reps, float *ms_per_rep) {
    if (!ix || !d_src || reps <= 0) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    int rc = ensure_events(ix);
    if (rc != TV_OK) return rc;
    rc = ensure_workspace(ix, 4096);
    if (rc != TV_OK) return rc;
    uint32_t *sink = static_cast<uint32_t *>(ix->ws);
    TV_HIP(tv::launch_probe(d_src, d_dst, bytes, d_dst != nullptr, sink, ix->stream));  // warm
    TV_HIP(hipEventRecord(ix->ev_start[0], ix->stream));
    for (int r = 0; r < reps; ++r) TV_HIP(tv::launch_probe(d_src, d_dst, bytes, d_dst != nullptr, sink, ix->stream));
    TV_HIP(hipEventRecord(ix->ev_stop[0], ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    float ms = 0.0f;
    TV_HIP(hipEventElapsedTime(&ms, ix->ev_start[0], ix->ev_stop[0]));
    if (ms_per_rep) *ms_per_rep = ms / float(reps);
    return TV_OK;
}

int tv_debug_mfma_probe(tv_index *ix, int iters, int reps, float *ms_per_rep, double *ops_per_rep) {
    if (!ix || iters <= 0 || reps <= 0) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    TV_HIP(hipSetDevice(ix->device));
    int rc = ensure_events(ix);
    if (rc != TV_OK) return rc;
    rc = ensure_workspace(ix, 4096);
    if (rc != TV_OK) return rc;
    uint32_t *sink = static_cast<uint32_t *>(ix->ws);
    double ops = 0.0;
    TV_HIP(tv::launch_probe_mfma(ix->device, iters, sink, &ops, ix->stream));  // warm
    TV_HIP(hipEventRecord(ix->ev_start[0], ix->stream));
    for (int r = 0; r < reps; ++r) TV_HIP(tv::launch_probe_mfma(ix->device, iters, sink, &ops, ix->stream));
    TV_HIP(hipEventRecord(ix->ev_stop[0], ix->stream));
    TV_HIP(hipStreamSynchronize(ix->stream));
    float ms = 0.0f;
    TV_HIP(hipEventElapsedTime(&ms, ix->ev_start[0], ix->ev_stop[0]));
    if (ms_per_rep) *ms_per_rep = ms / float(reps);
    if (ops_per_rep) *ops_per_rep = ops;
    return TV_OK;
}

int tv_debug_set_path(tv_index *ix, int force_full_lists) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    ix->force_robust = (force_full_lists & 1) != 0;
    ix->no_batched = (force_full_lists & 2) != 0;
    ix->no_wide = (force_full_lists & 4) != 0;
    ix->no_lut16 = (force_full_lists & 8) != 0;
    ix->no_direct = (force_full_lists & 16) != 0;
    ix->force_gather = (force_full_lists & 64) != 0;
    ix->force_near = (force_full_lists & 128) != 0;
    ix->no_gather = !ix->force_gather && force_full_lists != 0;     // (a call that names its kernels means them with the mask)
    return TV_OK;
}

int tv_debug_sampling_plan(const tv_index *cix, size_t nq, size_t k, uint32_t *strides, uint32_t *repeat_offsets, size_t cap,
                           size_t *count) {
    tv_index *ix = const_cast<tv_index *>(cix);
    if (!ix || !count) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    *count = 0;
    const size_t k_eff = std::min(k, ix->n);
    if (k_eff == 0 || nq == 0 || k_eff > size_t(tv::kMaxSampledK) || ix->force_robust) return TV_OK;   // no ladder
    const size_t n_blocks = (ix->n + tv::kVecBlock - 1) / tv::kVecBlock;
    if (direct_serves(ix, nq, k_eff, n_blocks, false)) return TV_OK;
    const SampledPlan plan = sampled_plan(ix, chunk_len(ix, nq));
    if (near_takes(ix, chunk_len(ix, nq), k_eff, n_blocks, ix->n)) return TV_OK;
    const SamplingSteps steps = level_strides(ix, plan, n_blocks, n_blocks, std::max<size_t>(k_eff, 16), false, false);
    *count = steps.size();
    for (size_t i = 0; i < steps.size() && i < cap; ++i) {
        if (strides) strides[i] = steps[i];
        if (repeat_offsets) repeat_offsets[i] = repeat_offset(steps[i]);
    }
    return TV_OK;
}

int tv_debug_level_repeats(tv_index *ix, int track, size_t *count) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    if (track >= 0) ix->track_levels = track;
    if (count) *count = ix->level_repeats;
    return TV_OK;
}

int tv_debug_workspace_bytes(const tv_index *cix, size_t *workspace, size_t *staging) {
    tv_index *ix = const_cast<tv_index *>(cix);
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> lock(ix->mu);
    std::lock_guard<std::mutex> kept(g_pool[ix->device].mu);
    if (workspace) *workspace = ix->ws_bytes + ix->slots.bytes + ix->gathered.bytes;
    if (staging) *staging = ix->io_bytes;
    return TV_OK;
}

int tv_debug_overflow_redos(const tv_index *ix, size_t *count) {
    if (!ix || !count) return TV_ERR_BAD_ARGUMENT;
    *count = ix->overflow_redos;
    return TV_OK;
}

int tv_debug_exact_redos(const tv_index *ix, size_t *count) {
    if (!ix || !count) return TV_ERR_BAD_ARGUMENT;
    *count = ix->exact_redos;
    return TV_OK;
}

int tv_debug_gathered_searches(const tv_index *ix, size_t *count, size_t *in_place) {
    if (!ix || !count) return TV_ERR_BAD_ARGUMENT;
    *count = ix->gathered_searches;
    if (in_place) *in_place = ix->in_place_searches;
    return TV_OK;
}

int tv_debug_merged_calls(const tv_index *cix, size_t *count) {
    tv_index *ix = const_cast<tv_index *>(cix);
    if (!ix || !count) return TV_ERR_BAD_ARGUMENT;
    std::lock_guard<std::mutex> reg(ix->waiting_mu);
    *count = ix->merged_calls;
    return TV_OK;
}

int tv_debug_queries_per_launch(const tv_index *ix, int *queries) {
    if (!ix || !queries) return TV_ERR_BAD_ARGUMENT;
    *queries = ix->last_queries_per_launch;
    return TV_OK;
}

int tv_last_scan_ms(const tv_index *ix, float *ms, int *launches) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    if (ms) *ms = ix->last_scan_ms;
    if (launches) *launches = ix->last_scan_launches;
    return TV_OK;
}

int tv_index_device_ptrs(const tv_index *ix, void **d_codes, void **d_scales, size_t *code_bytes) {
    if (!ix) return TV_ERR_BAD_ARGUMENT;
    if (d_codes) *d_codes = ix->d_codes;
    if (d_scales) *d_scales = ix->d_scales;
    if (code_bytes) *code_bytes = (ix->n + tv::kVecBlock - 1) / tv::kVecBlock * ix->geo.block_bytes();
    return TV_OK;
}

}  // extern "C"
