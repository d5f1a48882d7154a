// Host build of the copy ring (photons-on-mt3000_amd/csrc/host_pipe.h) for
// tests/test_host_pipe.py, over a stand-in for the few runtime calls it makes:
// copies are queued and done when an event or the stream is waited for, so that
// a slot filled again too early shows in the data.  No device is used.
#include "../../photons-on-mt3000_amd/csrc/host_pipe.h"

#include <cstdlib>
#include <deque>
#include <map>

namespace {

struct Op {
    void *dst;
    const void *src;
    size_t n;
    long long mark;             // > 0: an event's record
};
std::deque<Op> g_queue;
std::map<const char *, size_t> g_pinned;
long long g_copies, g_allocs, g_alloc_bytes, g_mark, g_done, g_last_error;
bool g_no_pinning;              // pinned allocations fail
const char *g_user;             // copies to or from the caller's own array
size_t g_user_n;
long long g_user_copies;

void run_until(long long mark)
{
    while (!g_queue.empty() && g_done < mark) {
        const Op o = g_queue.front();
        g_queue.pop_front();
        if (o.mark)
            g_done = o.mark;
        else
            std::memcpy(o.dst, o.src, o.n);
    }
}

bool in_user(const void *p) { return p >= g_user && p < g_user + g_user_n; }

bool pinned(const void *p)
{
    auto it = g_pinned.upper_bound(static_cast<const char *>(p));
    return it != g_pinned.begin() && static_cast<const char *>(p) < (--it)->first + it->second;
}

}  // namespace

extern "C" {

hipError_t hipMemcpyAsync(void *dst, const void *src, size_t n, hipMemcpyKind, hipStream_t)
{
    ++g_copies;
    g_user_copies += in_user(dst) || in_user(src);
    g_queue.push_back({dst, src, n, 0});
    // pageable memory is read or written before the call returns
    if ((in_user(dst) && !pinned(dst)) || (in_user(src) && !pinned(src)))
        run_until(1ll << 62);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t)
{
    run_until(1ll << 62);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    *e = reinterpret_cast<hipEvent_t>(new long long(0));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    delete reinterpret_cast<long long *>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    *reinterpret_cast<long long *>(e) = ++g_mark;
    g_queue.push_back({nullptr, nullptr, 0, g_mark});
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    run_until(*reinterpret_cast<long long *>(e));
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    ++g_allocs;
    if (g_no_pinning) {
        g_last_error = hipErrorOutOfMemory;
        return hipErrorOutOfMemory;
    }
    g_alloc_bytes += (long long)n;
    *p = std::malloc(n);
    g_pinned[static_cast<char *>(*p)] = n;
    return hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    g_pinned.erase(static_cast<char *>(p));
    std::free(p);
    return hipSuccess;
}
// as the runtime answers: memory that it does not know is an error, kept as the last one
hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    std::memset(a, 0, sizeof(*a));
    if (pinned(p)) {
        a->type = hipMemoryTypeHost;
        return hipSuccess;
    }
    g_last_error = hipErrorInvalidValue;
    return hipErrorInvalidValue;
}
hipError_t hipGetLastError(void)
{
    const hipError_t e = static_cast<hipError_t>(g_last_error);
    g_last_error = 0;
    return e;
}

// One context's copies: to the device and back for each of count sizes, from
// pageable or pinned arrays (shift bytes into their allocation).  0 when all data
// arrived; out = {copies, copies that touch the caller's arrays, pinned
// allocations of the ring, their bytes}.
int pipe_copies(const long long *sizes, int count, int pin, size_t shift, long long *out)
{
    pp2p::HostPipe pipe;
    int bad = 0;
    long long copies = 0, user = 0, allocs = 0, bytes = 0;
    for (int c = 0; c < count; ++c) {
        const size_t n = (size_t)sizes[c];
        char *dev = static_cast<char *>(std::calloc(n + 1, 1)), *host = nullptr;
        if (pin)
            (void)hipHostMalloc(reinterpret_cast<void **>(&host), n + shift, 0);
        else
            host = static_cast<char *>(std::malloc(n + shift));
        char *at = host + shift;
        for (size_t i = 0; i < n; ++i)
            at[i] = (char)(i * 2654435761u >> 13);
        g_user = at;
        g_user_n = n;
        g_copies = g_user_copies = g_allocs = g_alloc_bytes = 0;
        bad |= pipe.to_device(dev, at, n, nullptr) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess;
        bad |= std::memcmp(dev, at, n) != 0;
        std::memset(at, 1, n);
        bad |= pipe.to_host(at, dev, n, nullptr) != hipSuccess;
        bad |= std::memcmp(dev, at, n) != 0 || hipGetLastError() != hipSuccess;
        copies += g_copies;
        user += g_user_copies;
        allocs += g_allocs;
        bytes += g_alloc_bytes;
        g_user = nullptr;
        g_user_n = 0;
        if (pin)
            (void)hipHostFree(host);
        else
            std::free(host);
        std::free(dev);
    }
    pipe.release();
    out[0] = copies;
    out[1] = user;
    out[2] = allocs;
    out[3] = bytes;
    return bad;
}

// Ordinary arrays and records of 40 bytes (their first 12 packed) where nothing
// can be pinned.  0 when all data arrived and no error stayed behind.
int pipe_without_pinning(long long n)
{
    pp2p::HostPipe pipe;
    g_no_pinning = true;
    const size_t bytes = 12 * (size_t)n;
    char *rec = static_cast<char *>(std::malloc(40 * (size_t)n)), *dev = static_cast<char *>(std::calloc(bytes + 1, 1));
    char *flat = static_cast<char *>(std::malloc(bytes));
    for (size_t i = 0; i < 40 * (size_t)n; ++i)
        rec[i] = (char)(i * 2654435761u >> 13);
    for (size_t i = 0; i < (size_t)n; ++i)
        std::memcpy(flat + 12 * i, rec + 40 * i, 12);
    int bad = pipe.to_device_filled(dev, bytes, 12, nullptr, [&](char *at, size_t b, size_t m) {
                  for (size_t i = 0; i < m / 12; ++i)
                      std::memcpy(at + 12 * i, rec + 40 * (b / 12 + i), 12);
              }) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess;
    bad |= std::memcmp(dev, flat, bytes) != 0;
    std::memset(dev, 1, bytes);
    g_user = flat;
    g_user_n = bytes;
    bad |= pipe.to_device(dev, flat, bytes, nullptr) != hipSuccess || hipStreamSynchronize(nullptr) != hipSuccess;
    bad |= std::memcmp(dev, flat, bytes) != 0;
    std::memset(flat, 1, bytes);
    bad |= pipe.to_host(flat, dev, bytes, nullptr) != hipSuccess;
    bad |= std::memcmp(dev, flat, bytes) != 0 || hipGetLastError() != hipSuccess;
    pipe.release();
    g_user = nullptr;
    g_user_n = 0;
    g_no_pinning = false;
    std::free(rec);
    std::free(dev);
    std::free(flat);
    return bad;
}

}  // extern "C"
