// hostcopy.cpp — see hostcopy.hpp.
#include "hostcopy.hpp"

#include <algorithm>
#include <cstring>
#include <exception>

namespace ptk {

void CopyTeam::part(const Job& j, int i) const {
    const size_t parts = threads_.size() + 1;
    const size_t len = (j.n / parts + 63) / 64 * 64;
    const size_t lo = std::min(j.n, len * (size_t)i), hi = (size_t)i + 1 == parts ? j.n : std::min(j.n, lo + len);
    if (hi > lo) std::memcpy(j.dst + lo, j.src + lo, hi - lo);
}

void CopyTeam::work(int i) {
    unsigned seen = 0;
    while (true) {
        // the next chunk of a copy follows within microseconds; between copies, sleep
        for (int k = 0; k < 4000 && turn_.load(std::memory_order_acquire) == seen; ++k) __builtin_ia32_pause();
        if (turn_.load(std::memory_order_acquire) == seen) {
            std::unique_lock<std::mutex> lock(mu_);
            cv_.wait(lock, [&] { return turn_.load(std::memory_order_acquire) != seen; });
        }
        if (stop_.load()) return;
        ++seen;  // no copy starts before every helper has ended the one before
        part(job_, i);
        left_.fetch_sub(1, std::memory_order_release);
    }
}

void CopyTeam::copy(void* dst, const void* src, size_t n) {
    if (n < ((size_t)64 << 10)) {
        std::memcpy(dst, src, n);
        return;
    }
    if (!started_) {
        started_ = true;
        try {
            threads_.reserve(kWorkers);
            const int cores = (int)std::thread::hardware_concurrency();
            for (int i = 0; i < std::min(kWorkers, cores - 1); ++i) threads_.emplace_back([this, i] { work(i + 1); });
        } catch (const std::exception&) {
            // no more threads to be had: those there are share the work
        }
    }
    const Job j{static_cast<char*>(dst), static_cast<const char*>(src), n};
    if (threads_.empty()) {
        part(j, 0);
        return;
    }
    {
        std::lock_guard<std::mutex> lock(mu_);
        job_ = j;
        left_.store((int)threads_.size(), std::memory_order_relaxed);
        turn_.fetch_add(1, std::memory_order_release);
    }
    cv_.notify_all();
    part(j, 0);
    while (left_.load(std::memory_order_acquire) != 0) __builtin_ia32_pause();
}

CopyTeam::~CopyTeam() {
    {
        std::lock_guard<std::mutex> lock(mu_);
        stop_.store(true);
        turn_.fetch_add(1, std::memory_order_release);
    }
    cv_.notify_all();
    for (std::thread& t : threads_) t.join();
}

HostCopy::~HostCopy() {
    for (Slot& s : ring_) {
        (void)wait(s);
        if (s.done) (void)hipEventDestroy(s.done);
        if (s.p) (void)hipHostFree(s.p);
    }
}

// Whether the first `slots` ring buffers are there. Their events are made on the device of
// the stream they will be recorded on, which need not be the caller's current one.
bool HostCopy::ready(int slots, hipStream_t st) {
    if (ring_[slots - 1].p) return true;  // they are made in order
    int current = 0;
    hipDevice_t device = 0;
    if (hipGetDevice(&current) != hipSuccess || hipStreamGetDevice(st, &device) != hipSuccess ||
        (device != current && hipSetDevice(device) != hipSuccess)) {
        (void)hipGetLastError();
        return false;
    }
    bool ok = true;
    for (int i = 0; i < slots && ok; ++i) {
        Slot& s = ring_[i];
        if (s.p) continue;
        if (!s.done && hipEventCreateWithFlags(&s.done, hipEventDisableTiming) != hipSuccess) {
            s.done = nullptr;
            ok = false;
        }
        void* p = nullptr;
        if (ok && hipHostMalloc(&p, kChunk, hipHostMallocDefault) != hipSuccess) ok = false;
        if (ok) s.p = static_cast<char*>(p);
    }
    if (!ok) (void)hipGetLastError();
    if (device != current) (void)hipSetDevice(current);
    return ok;
}

hipError_t HostCopy::wait(Slot& s) {
    if (!s.busy) return hipSuccess;
    s.busy = false;
    return hipEventSynchronize(s.done);
}

// Whether p is the caller's pageable memory. What the runtime knows (page-locked memory
// moves at PCIe speed by itself; managed and device memory is not for the copying threads)
// is its own to copy: 33 MB back into page-locked memory take 0.59 ms, through the ring 0.75.
static bool pageable(const void* p) {
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();  // not an address of the runtime's
        return true;
    }
    return a.type == hipMemoryTypeUnregistered;
}

// Bytes per chunk of a copy of n. A chunk costs about 20 us of calls and waits, so up
// to 2 MB go in one and up to 8 MB in two (1 / 2 / 4 / 8 chunks at least: 1.9 MB back
// in 66 / 79 / 123 / 176 us, 4.2 MB in 149 / 127 / 176 / 222 us; from 15 MB on, where
// 4 MB chunks follow one another, no difference). The runtime's pageable copies take
// 105 us for 1.9 MB, 235 for 4.2, 1.85 ms for 33 MB back (now 0.76).
static size_t chunk_of(size_t n, size_t most) {
    return std::min(most, std::max((size_t)2 << 20, (n / 2 + 65535) / 65536 * 65536));
}

hipError_t HostCopy::to_host(void* dst, const void* src, size_t n, hipStream_t st) {
    const size_t chunk = chunk_of(n, kChunk);
    const size_t chunks = (n + chunk - 1) / chunk;
    const int slots = (int)std::min<size_t>(kRing, chunks);
    if (n < kLeast || !pageable(dst) || !ready(slots, st)) {
        hipError_t e = hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, st);
        const hipError_t es = hipStreamSynchronize(st);
        return e != hipSuccess ? e : es;
    }
    auto len = [&](size_t c) { return std::min(chunk, n - c * chunk); };
    auto start = [&](size_t c) -> hipError_t {
        Slot& s = ring_[c % slots];
        hipError_t e = wait(s);
        if (e == hipSuccess)
            e = hipMemcpyAsync(s.p, static_cast<const char*>(src) + c * chunk, len(c), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipEventRecord(s.done, st);
        s.busy = e == hipSuccess;
        return e;
    };
    hipError_t e = hipSuccess;
    for (size_t c = 0; c < (size_t)slots && e == hipSuccess; ++c) e = start(c);
    for (size_t c = 0; c < chunks && e == hipSuccess; ++c) {
        Slot& s = ring_[c % slots];
        e = wait(s);
        if (e != hipSuccess) break;
        team_.copy(static_cast<char*>(dst) + c * chunk, s.p, len(c));
        if (c + slots < chunks) e = start(c + slots);
    }
    const hipError_t es = hipStreamSynchronize(st);
    return e != hipSuccess ? e : es;
}

hipError_t HostCopy::to_device(void* dst, const void* src, size_t n, hipStream_t st) {
    const size_t chunk = chunk_of(n, kChunk);
    const size_t chunks = (n + chunk - 1) / chunk;
    const int slots = (int)std::min<size_t>(kRing, chunks);
    if (n < kLeast || !pageable(src) || !ready(slots, st)) return hipMemcpyAsync(dst, src, n, hipMemcpyHostToDevice, st);
    for (size_t c = 0; c < chunks; ++c) {
        Slot& s = ring_[c % slots];
        const size_t len = std::min(chunk, n - c * chunk);
        hipError_t e = wait(s);
        if (e != hipSuccess) return e;
        team_.copy(s.p, static_cast<const char*>(src) + c * chunk, len);
        e = hipMemcpyAsync(static_cast<char*>(dst) + c * chunk, s.p, len, hipMemcpyHostToDevice, st);
        if (e == hipSuccess) e = hipEventRecord(s.done, st);
        if (e != hipSuccess) {
            // the ring buffers may still be read: nothing is left in flight
            (void)hipStreamSynchronize(st);
            return e;
        }
        s.busy = true;
    }
    return hipSuccess;
}

}  // namespace ptk
