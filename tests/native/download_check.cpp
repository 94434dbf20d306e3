// csrc/download.hpp on the CPU: the HIP calls it makes are stood in for by a
// queue that copies when an event or the stream is waited for, and the n-th
// memory allocation of a call fails.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <functional>
#include <new>

#include "download.hpp"

static std::atomic<long> fail_at{-1};   // allocations until one fails, < 0: none
void *operator new(size_t n) {
    if (fail_at >= 0 && fail_at-- == 0) throw std::bad_alloc();
    if (void *p = malloc(n ? n : 1)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

// The stream: copies in order, carried out up to what is waited for.
struct Copy {
    void *dst;
    const void *src;
    size_t n;
};
static std::mutex mx;
static Copy copies[1 << 16];
static size_t enqueued = 0, done = 0;
static size_t marks[64];
static int events = 0;
static void upto(size_t k) {
    std::lock_guard<std::mutex> l(mx);
    for (; done < k; done++) memcpy(copies[done].dst, copies[done].src, copies[done].n);
}
extern "C" {
hipError_t hipHostMalloc(void **p, size_t n, unsigned) { *p = malloc(n); return hipSuccess; }
hipError_t hipHostFree(void *p) { free(p); return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = (hipEvent_t)(uintptr_t)(++events); return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
    std::lock_guard<std::mutex> l(mx);
    if (enqueued == sizeof copies / sizeof copies[0]) abort();
    copies[enqueued++] = Copy{d, s, n};
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    std::lock_guard<std::mutex> l(mx);
    marks[(uintptr_t)e % 64] = enqueued;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    size_t k;
    {
        std::lock_guard<std::mutex> l(mx);
        k = marks[(uintptr_t)e % 64];
    }
    upto(k);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
    size_t k;
    {
        std::lock_guard<std::mutex> l(mx);
        k = enqueued;
    }
    upto(k);
    return hipSuccess;
}
}

using ssa::Download;
using ssa::PinnedRing;

static int fail(const char *what, size_t n) {
    printf("%s: %zu\n", what, n);
    return 1;
}

// n elements and n particles through the ring (or, for a small total, without)
static int round_trip(size_t n, size_t total) {
    std::vector<unsigned> a(n), b(n);
    std::vector<double> s(3 * n), p(3 * n);
    for (size_t i = 0; i < n; i++) a[i] = (unsigned)i * 2654435761u;
    for (size_t i = 0; i < 3 * n; i++) s[i] = (double)i + 0.25;
    PinnedRing ring;
    {
        Download out(nullptr, ring, total);
        out.put(b.data(), a.data(), n);
        out.put3(p.data(), s.data(), n);
        out.put(b.data(), a.data(), n);
        out.finish();
    }
    enqueued = done = 0;
    if (a != b) return fail("put", n);
    for (size_t i = 0; i < n; i++)
        for (int c = 0; c < 3; c++)
            if (p[3 * i + c] != s[c * n + i]) return fail("put3", n);
    return 0;
}

int main(int argc, char **argv) {
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "sizes") {
        // elements and particles of a slot, and one less and more; all slots
        // once, and again
        const size_t e = PinnedRing::SLOT / 4, q = PinnedRing::SLOT / 24;
        for (size_t n : {(size_t)0, (size_t)1, e - 1, e, e + 1, q - 1, q, q + 1, 3 * q + 1, PinnedRing::SLOTS * q,
                         PinnedRing::SLOTS * q + 1, PinnedRing::SLOTS * e + 1})
            for (size_t total : {(size_t)1, ssa::DOWNLOAD_MIN})
                if (round_trip(n, total)) return 1;
        return 0;
    }
    // every allocation of a download failing in turn: an exception or a result
    const size_t n = PinnedRing::SLOT / 2;
    std::vector<unsigned> a(n, 7u), b(n);
    PinnedRing ring;
    bool whole = false;
    for (long k = 0; !whole; k++) {
        fail_at = k;
        try {
            Download out(nullptr, ring, ssa::DOWNLOAD_MIN);
            out.put(b.data(), a.data(), n);
            out.finish();
            whole = fail_at >= 0;
            fail_at = -1;
            if (a != b) return fail("after a failed allocation", (size_t)k);
        } catch (const std::bad_alloc &) {
        }
        fail_at = -1;
        enqueued = done = 0;
        std::fill(b.begin(), b.end(), 0u);
        if (k > 1000) return fail("allocations", (size_t)k);
    }
    return 0;
}
