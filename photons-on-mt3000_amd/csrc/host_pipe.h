// Copies between pageable host memory and the device through a small ring of
// pinned slots: the DMA engine moves one piece while a few host threads fill or
// empty the others (internal to the library).  Memory that the DMA engine
// reaches by itself (pinned by the caller) is copied straight, with no thread.
//
// A copy straight from pageable memory runs at half the pinned rate, and one
// into memory that the caller has just allocated at 4 GB/s, since a single
// thread takes every page fault; here up to twelve threads share the faults,
// ahead of the copy and a 2 MiB block each (with large pages, threads that fault
// in one block wait for each other).
// The threads and the ring (four slots of 2 MiB) belong to one context; both start
// with its first large copy and end with it.  That copy pays for them: 0.15 ms for
// the threads, about 0.3 ms for pinning the ring and 0.1 ms for each MiB of it that
// is used.  The threads sleep
// between copies; within one they wait for the next piece for some tens of
// microseconds before they sleep (spinning throughout took the processor time of
// the caller's own threads: passes of ten times the usual length now and then).
// Measured: 230 MB into fresh pages 21.4 -> 6.5 ms, 36 MB 3.2 -> 0.8 ms, 4.3 MB
// 0.28 -> 0.20 ms; two 10 MB lists up 1.40 -> 0.82 ms, 306 MB of positions and tags up
// as before (57 GB/s pinned).
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <functional>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace pp2p {

// A few threads that run one function over slices, together with the caller.
class Crew {
public:
    ~Crew()
    {
        {
            std::lock_guard<std::mutex> l(m_);
            quit_ = true;
            gen_.fetch_add(1);
        }
        wake_.notify_all();
        for (auto &t : th_)
            t.join();
    }

    // fn(k) for k in [0, slices), each once, on any of the threads
    void run(int slices, const std::function<void(int)> &fn)
    {
        if (slices <= 1) {
            if (slices == 1)
                fn(0);
            return;
        }
        start(slices - 1);
        if (!th_.empty()) {
            std::lock_guard<std::mutex> l(m_);
            fn_ = &fn;
            slices_ = slices;
            next_.store(0, std::memory_order_relaxed);
            open_ = true;
            gen_.fetch_add(1, std::memory_order_release);
        }
        if (th_.empty()) {
            for (int k = 0; k < slices; ++k)
                fn(k);
            return;
        }
        wake_.notify_all();
        for (int k; (k = next_.fetch_add(1)) < slices;)
            fn(k);
        // a thread that wakes up later finds the job closed; those in it end
        // their slices
        {
            std::lock_guard<std::mutex> l(m_);
            open_ = false;
        }
        while (inside_.load(std::memory_order_acquire) > 0)
            std::this_thread::yield();
    }

private:
    // at least `want` threads, as far as there are processors
    void start(int want)
    {
        const unsigned hw = std::thread::hardware_concurrency();
        want = std::min(want, (int)std::min<unsigned>(hw > 1 ? hw - 1 : 0, 11));
        if ((int)th_.size() >= want || full_)
            return;
        try {
            th_.reserve(want);
            while ((int)th_.size() < want)
                th_.emplace_back([this] { work(); });
        } catch (const std::exception &) {           // fewer threads, or none: the caller copies
            full_ = true;
        }
    }

    void work()
    {
        for (unsigned seen = 0;;) {
            for (int spin = 0; spin < 200 && gen_.load(std::memory_order_acquire) == seen; ++spin)
                std::this_thread::yield();
            {
                std::unique_lock<std::mutex> l(m_);
                wake_.wait(l, [&] { return gen_.load(std::memory_order_relaxed) != seen; });
                seen = gen_.load(std::memory_order_relaxed);
                if (quit_)
                    return;
                if (!open_)
                    continue;
                inside_.fetch_add(1, std::memory_order_relaxed);
            }
            for (int k; (k = next_.fetch_add(1)) < slices_;)
                (*fn_)(k);
            inside_.fetch_sub(1, std::memory_order_release);
        }
    }

    std::vector<std::thread> th_;
    std::mutex m_;
    std::condition_variable wake_;
    std::atomic<unsigned> gen_{0};
    std::atomic<int> next_{0}, inside_{0};
    const std::function<void(int)> *fn_ = nullptr;
    int slices_ = 0;
    bool full_ = false, quit_ = false, open_ = false;
};

class HostPipe {
public:
    // Smaller copies go through the runtime: 2.6 MB arrays measured the same
    // either way once the threads and the ring are there, and 1.4 ms longer the first
    // time.
    static constexpr size_t kLeast = 4 << 20;

    // Whether a copy from or to p goes through the ring: not a small one, and not
    // where the runtime knows the memory (both ends asked).
    static bool staged(const void *p, size_t bytes)
    {
        return bytes >= kLeast && !(known(p) && known(static_cast<const char *>(p) + bytes - 1));
    }

    // bytes from src to dst; the caller may reuse a pageable src when it returns,
    // a pinned one when the stream has passed the copy.
    hipError_t to_device(void *dst, const void *src, size_t bytes, hipStream_t st)
    {
        hipError_t e = hipSuccess;
        if (!staged(src, bytes) || ((e = open(piece_of(bytes))) == hipSuccess && !ring_))
            return bytes ? hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st) : hipSuccess;
        if (e != hipSuccess)
            return e;
        const char *s = static_cast<const char *>(src);
        return to_device_filled(dst, bytes, 1, st, [s](char *at, size_t b, size_t n) { std::memcpy(at, s + b, n); });
    }

    // bytes that fill(at, b, n) writes to at: those from byte b on, n of them,
    // both multiples of `unit`.  fill runs on several threads.
    template <class Fill>
    hipError_t to_device_filled(void *dst, size_t bytes, size_t unit, hipStream_t st, Fill fill)
    {
        if (!bytes)
            return hipSuccess;
        hipError_t e = open(piece_of(bytes));
        const size_t piece = piece_of(bytes) / unit * unit;
        std::unique_ptr<char[]> plain;               // one piece where nothing can be pinned
        if (e == hipSuccess && !ring_) {
            plain.reset(new (std::nothrow) char[piece]);
            if (!plain)
                return hipErrorOutOfMemory;
        }
        for (size_t b = 0, k = 0; b < bytes && e == hipSuccess; b += piece, ++k) {
            const size_t n = std::min(piece, bytes - b);
            char *at = plain ? plain.get() : slot(k);
            e = hipEventSynchronize(ev_[k % kSlots]);            // the copy that last used the slot
            if (e != hipSuccess)
                break;
            const int s = slices_of(n);
            const size_t each = (n / unit + s - 1) / s * unit;
            crew_->run(s, [&](int q) {
                const size_t o = q * each;
                if (o < n)
                    fill(at + o, b + o, std::min(each, n - o));
            });
            e = hipMemcpyAsync(static_cast<char *>(dst) + b, at, n, hipMemcpyHostToDevice, st);
            if (e == hipSuccess)
                e = plain ? hipStreamSynchronize(st) : hipEventRecord(ev_[k % kSlots], st);
        }
        return e;
    }

    // bytes from src to dst; complete when it returns.
    hipError_t to_host(void *dst, const void *src, size_t bytes, hipStream_t st)
    {
        const size_t piece = piece_of(bytes), pieces = (bytes + piece - 1) / piece;
        hipError_t e = hipSuccess;
        if (!staged(dst, bytes) || ((e = open(piece)) == hipSuccess && !ring_)) {
            e = bytes ? hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st) : hipSuccess;
            return e == hipSuccess ? hipStreamSynchronize(st) : e;
        }
        size_t issued = 0, touched = 0;
        for (size_t k = 0; k < pieces && e == hipSuccess; ++k) {
            for (; issued < pieces && issued < k + kSlots && e == hipSuccess; ++issued) {      // into the emptied slots
                const size_t b = issued * piece;
                e = hipMemcpyAsync(slot(issued), static_cast<const char *>(src) + b, std::min(piece, bytes - b),
                                   hipMemcpyDeviceToHost, st);
                if (e == hipSuccess)
                    e = hipEventRecord(ev_[issued % kSlots], st);
            }
            // the pages of the next pieces, a dozen blocks at a time
            if (touched < bytes && touched < (k + 2) * piece) {
                const size_t to = std::min(bytes, touched + 12 * kBlock);
                touch(static_cast<char *>(dst), touched, to);
                touched = to;
            }
            if (e == hipSuccess)
                e = hipEventSynchronize(ev_[k % kSlots]);
            if (e != hipSuccess)
                break;
            const size_t b = k * piece, n = std::min(piece, bytes - b);
            const int s = slices_of(n);
            const size_t each = (n + s - 1) / s;
            crew_->run(s, [&](int q) {
                const size_t o = q * each;
                if (o < n)
                    std::memcpy(static_cast<char *>(dst) + b + o, slot(k) + o, std::min(each, n - o));
            });
        }
        return e;
    }

    // fn(b, n) over slices of [0, bytes), their starts multiples of 64, on several
    // threads from kLeast on
    template <class Fn>
    void each(size_t bytes, Fn fn)
    {
        if (bytes < kLeast) {
            fn((size_t)0, bytes);
            return;
        }
        if (!crew_)
            crew_.reset(new Crew());
        const int s = slices_of(bytes);
        const size_t part = ((bytes + s - 1) / s + 63) / 64 * 64;
        crew_->run(s, [&](int q) {
            const size_t b = q * part;
            if (b < bytes)
                fn(b, std::min(part, bytes - b));
        });
    }

    void release()
    {
        for (auto &v : ev_) {
            if (v)
                (void)hipEventDestroy(v);
            v = nullptr;
        }
        if (ring_)
            (void)hipHostFree(ring_);
        ring_ = nullptr;
        slot_ = 0;
        crew_.reset();
    }

private:
    static constexpr size_t kSlot = 2 << 20, kSmallSlot = 256 << 10;
    static constexpr int kSlots = 4;
    static constexpr size_t kBlock = 2 << 20;

    // pinned, managed or device memory; pageable memory is an error to some
    // versions of the runtime, which must not stay behind as the last one
    static bool known(const void *p)
    {
        hipPointerAttribute_t a;
        if (hipPointerGetAttributes(&a, p) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        return a.type != hipMemoryTypeUnregistered;
    }

    // about four pieces of a copy below 8 MiB, so that it overlaps itself too
    static size_t piece_of(size_t bytes)
    {
        const size_t p = (bytes / kSlots + 4095) / 4096 * 4096;
        return std::min(kSlot, std::max(p, (size_t)64 << 10));
    }
    static int slices_of(size_t n) { return (int)std::max<size_t>(n >> 17, 1); }        // 128 KiB and more

    // one byte of every page of [p + b, p + e) written, a block of 2 MiB per slice
    // (the range is about to be overwritten)
    void touch(char *p, size_t b, size_t e)
    {
        const size_t base = reinterpret_cast<size_t>(p), first = (base + b) / kBlock, last = (base + e - 1) / kBlock;
        crew_->run((int)(last - first + 1), [&](int q) {
            const size_t lo = std::max((first + q) * kBlock, base + b), hi = std::min((first + q + 1) * kBlock, base + e);
            for (size_t a = lo; a < hi; a = (a / 4096 + 1) * 4096)
                *reinterpret_cast<volatile char *>(a) = 0;
        });
    }

    char *slot(size_t k) const { return ring_ + (k % kSlots) * slot_; }

    // the threads, and slots of at least `slot` bytes with no copy in flight, or no
    // ring where none can be pinned (the copies are then the runtime's).  A ring
    // has small slots or full ones, nothing between: pinning it takes about 0.3 ms
    // whatever its size, and the first touch of its pages (0.4 ms per MiB on one
    // thread) comes with the pieces that use them; a ring that grew with the longest
    // copy so far was pinned and touched twice when a program's lists are longer than
    // its positions (1 ms of its first pass).
    hipError_t open(size_t slot)
    {
        slot = slot <= kSmallSlot ? kSmallSlot : kSlot;
        if (!crew_)
            crew_.reset(new Crew());
        for (auto &v : ev_) {
            // an upload's last copies may still be in flight
            hipError_t e = v ? hipEventSynchronize(v) : hipEventCreateWithFlags(&v, hipEventDisableTiming);
            if (e != hipSuccess)
                return e;
        }
        if (slot <= slot_)
            return hipSuccess;
        if (ring_)
            (void)hipHostFree(ring_);
        ring_ = nullptr;
        slot_ = 0;
        void *p = nullptr;
        if (hipHostMalloc(&p, kSlots * slot, hipHostMallocDefault) == hipSuccess) {
            ring_ = static_cast<char *>(p);
            slot_ = slot;
        } else {
            (void)hipGetLastError();
        }
        return hipSuccess;
    }

    char *ring_ = nullptr;
    size_t slot_ = 0;
    hipEvent_t ev_[kSlots] = {nullptr, nullptr, nullptr, nullptr};
    std::unique_ptr<Crew> crew_;
};

}  // namespace pp2p
