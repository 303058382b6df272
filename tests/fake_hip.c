/* A HIP runtime without a device, for tests of the library's host side: device memory is host memory with a limit,
 * launches do nothing (but the one whose counts the host waits for), and the test decides how long a wait takes.  Loaded with RTLD_GLOBAL before the library, whose
 * references then resolve here. */
#define _GNU_SOURCE
#include <pthread.h>
#include <stdatomic.h>
#include <stddef.h>
#include <stdint.h>
#include <stdlib.h>
#include <string.h>
#include <time.h>
#include <unistd.h>

enum { ok = 0, out_of_memory = 2 };
typedef struct { uint32_t x, y, z; } dim3_t;

/* ---- what a test sets and reads ---- */
atomic_size_t fake_limit = (size_t)1 << 34, fake_used;
atomic_int fake_large_alloc_us;       /* how long an allocation of 256 MiB and more takes */
atomic_int fake_stream_wait_us;       /* how long a stream's wait takes ... */
atomic_int fake_stream_waits;         /* ... and how many there were */
atomic_int fake_stream_waits_refused; /* so many of the next ones report an error */
atomic_int fake_frees_refused;        /* so many of the next frees of device memory report an error */
atomic_int fake_device_busy;          /* the device's wait does not end while this is set ... */
atomic_int fake_device_waits;         /* ... and this many threads are in one */
atomic_long fake_clock_reads;         /* std::chrono::steady_clock::now() */
atomic_int fake_cus = 256;            /* compute units the device says it has */
atomic_int fake_largest_grid;         /* workgroups of the largest launch */
atomic_int fake_launches;             /* kernels launched */
atomic_int fake_pinned_blocks;        /* blocks of pinned memory of 64 KiB and more allocated so far ... */
atomic_size_t fake_pinned, fake_pinned_peak;      /* ... and their bytes now, and at most */
uint32_t fake_marker;                 /* when not 0: copies to the device are searched for this word ... */
atomic_int fake_marker_copies;        /* ... and those that hold it counted */

int hipGetDeviceCount(int *n) { *n = 1; return ok; }
int hipSetDevice(int d) { (void)d; return ok; }
int hipDeviceGetAttribute(int *v, int attr, int d) { (void)attr; (void)d; *v = fake_cus; return ok; }
const char *hipGetErrorString(int e) { return e == ok ? "ok" : "out of memory"; }
static _Thread_local int last;
int hipGetLastError(void) { const int e = last; last = ok; return e; }

static int take(void **p, size_t n) {
    size_t used = fake_used;
    do {
        if (used + n > fake_limit) return last = out_of_memory;
    } while (!atomic_compare_exchange_weak(&fake_used, &used, used + n));
    size_t *at = calloc(1, n + 256);
    at[0] = n;
    *p = (char *)at + 256;
    return ok;
}
static int give(void *p) {
    if (p) { size_t *at = (size_t *)((char *)p - 256); fake_used -= at[0]; free(at); }
    return ok;
}
int hipDeviceSynchronize(void) {
    ++fake_device_waits;
    while (fake_device_busy) usleep(100);
    --fake_device_waits;
    return ok;
}
int hipMalloc(void **p, size_t n) {
    if (n >= (size_t)256 << 20 && fake_large_alloc_us) usleep(fake_large_alloc_us);
    return take(p, n);
}
int hipFree(void *p) {
    if (p) hipDeviceSynchronize();
    give(p);
    if (p && fake_frees_refused > 0) { --fake_frees_refused; return last = out_of_memory; }
    return ok;
}
int hipHostMalloc(void **p, size_t n, unsigned flags) {
    (void)flags;
    const size_t counted = n >= 65536 ? n : 0;
    size_t *at = calloc(1, n + 256);
    at[0] = counted;
    *p = (char *)at + 256;
    fake_pinned_blocks += counted != 0;
    const size_t now = atomic_fetch_add(&fake_pinned, counted) + counted;
    for (size_t peak = fake_pinned_peak; now > peak && !atomic_compare_exchange_weak(&fake_pinned_peak, &peak, now);) {}
    return ok;
}
int hipHostFree(void *p) {
    if (p) { size_t *at = (size_t *)((char *)p - 256); fake_pinned -= at[0]; free(at); }
    return ok;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned flags) { (void)flags; *d = h; return ok; }
int hipGetSymbolAddress(void **p, const void *symbol) { (void)symbol; static char *at; if (!at) at = calloc(1, 64 << 20); *p = at; return ok; }
int hipMemcpyAsync(void *to, const void *from, size_t n, int kind, void *s) {
    (void)s;
    if (fake_marker != 0 && kind == 1 /* host to device */) {
        const uint32_t *w = from;
        size_t i = 0;
        while (i < n / 4 && w[i] != fake_marker) ++i;
        fake_marker_copies += i < n / 4;
    }
    memmove(to, from, n);
    return ok;
}
int hipMemsetAsync(void *p, int v, size_t n, void *s) { (void)s; memset(p, v, n); return ok; }
int hipStreamCreateWithFlags(void **s, unsigned flags) { (void)flags; *s = &last; return ok; }
int hipStreamDestroy(void *s) { (void)s; return ok; }
int hipStreamSynchronize(void *s) {
    (void)s;
    ++fake_stream_waits;
    if (fake_stream_wait_us) usleep(fake_stream_wait_us);
    if (fake_stream_waits_refused > 0) { --fake_stream_waits_refused; return last = out_of_memory; }
    return ok;
}
int hipEventCreate(void **e) { *e = &last; return ok; }
int hipEventDestroy(void *e) { (void)e; return ok; }
int hipEventRecord(void *e, void *s) { (void)e; (void)s; return ok; }
int hipEventElapsedTime(float *ms, void *a, void *b) { (void)a; (void)b; *ms = 0.0f; return ok; }
int hipFuncSetAttribute(const void *f, int attr, int v) { (void)f; (void)attr; (void)v; return ok; }
/* tv_filter.hip's count of a mask's rows and of the blocks they lie in */
atomic_int fake_counts;               /* launches of it that the host waits for */
static const void *mask_count;
/* tv_kernels.hip's selection by four threads a segment */
atomic_int fake_parted;               /* launches of it */
static const void *parted;
/* every kernel by its mangled name */
enum { most_kernels = 2048 };
static struct { const void *host; const char *name; atomic_int launches; size_t lds; } kernels[most_kernels];
static int n_kernels;
/* launches of those whose name has `part` in it, and the dynamic LDS of their last ones, at most */
int fake_launched(const char *part) {
    int n = 0;
    for (int i = 0; i < n_kernels; ++i) if (strstr(kernels[i].name, part)) n += kernels[i].launches;
    return n;
}
size_t fake_lds(const char *part) {
    size_t most = 0;
    for (int i = 0; i < n_kernels; ++i) if (strstr(kernels[i].name, part) && kernels[i].lds > most) most = kernels[i].lds;
    return most;
}
void __hipRegisterFunction(void **modules, const void *host, char *device, const char *name, unsigned limit, void *a, void *b, void *c, void *d, int *e) {
    (void)modules; (void)device; (void)limit; (void)a; (void)b; (void)c; (void)d; (void)e;
    if (n_kernels < most_kernels) {
        kernels[n_kernels].host = host;
        kernels[n_kernels++].name = strdup(name);
    }
    if (strstr(name, "k_mask_count")) mask_count = host;
    if (strstr(name, "k_finalILj1024ELj4E")) parted = host;
}
int hipLaunchKernel(const void *f, dim3_t g, dim3_t b, void **args, size_t lds, void *s) {
    (void)g; (void)b; (void)s;
    ++fake_launches;
    for (int i = 0; i < n_kernels; ++i)
        if (kernels[i].host == f) { ++kernels[i].launches; kernels[i].lds = lds; }
    fake_parted += f == parted;
    if (f == mask_count && *(uint64_t **)args[5] != NULL) {
        ++fake_counts;
        const uint32_t *mask = *(const uint32_t **)args[0];
        const uint32_t n = *(uint32_t *)args[1];
        const uint32_t pieces = *(uint32_t *)args[3];
        uint64_t *totals = *(uint64_t **)args[5], rows = 0, live = 0;
        for (uint32_t w = 0; w * 32 < n; ++w) {
            const uint32_t x = n - w * 32 < 32 ? mask[w] & ((1u << (n - w * 32)) - 1u) : mask[w];
            rows += (uint32_t)__builtin_popcount(x);
            live += x != 0;
        }
        for (uint32_t i = 1; i < (pieces + 3) / 4 && i < 256; ++i) totals[i] = (uint64_t)1 << 63;
        totals[0] = (uint64_t)1 << 63 | live << 31 | rows;
    }
    return ok;
}
static _Thread_local size_t pushed_lds;
int __hipPushCallConfiguration(dim3_t g, dim3_t b, size_t lds, void *s) {
    (void)b; (void)s;
    pushed_lds = lds;
    const int n = (int)(g.x * g.y * g.z);
    if (n > fake_largest_grid) fake_largest_grid = n;
    return ok;
}
int __hipPopCallConfiguration(dim3_t *g, dim3_t *b, size_t *lds, void **s) {
    *g = *b = (dim3_t){1, 1, 1};
    *lds = pushed_lds;
    *s = NULL;
    return ok;
}

/* std::chrono::steady_clock::now() */
int64_t _ZNSt6chrono3_V212steady_clock3nowEv(void) {
    struct timespec t;
    ++fake_clock_reads;
    clock_gettime(CLOCK_MONOTONIC, &t);
    return (int64_t)t.tv_sec * 1000000000 + t.tv_nsec;
}
