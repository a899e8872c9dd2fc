// hostcopy.hpp — copies between pageable host memory and the device through pinned
// staging buffers.
//
// The C ABI takes and fills the caller's own buffers. The runtime copies pageable
// memory at 27 GB/s to the device and 17 GB/s back here (100 MB, measured), where
// pinned memory moves at 57 GB/s each way and one core copies 25 GB/s: a 1920x1080
// denoise spent 4.8 of its 5.9 ms there. A HostCopy moves a copy in chunks through a
// ring of pinned buffers, with several threads copying a chunk between the ring and
// the caller's memory while the next ones are in flight. Memory that is page-locked
// already, or otherwise known to the runtime, is copied by it in one piece.
#pragma once

#include <hip/hip_runtime.h>

#include <atomic>
#include <condition_variable>
#include <mutex>
#include <thread>
#include <vector>

namespace ptk {

// memcpy by the calling thread and up to kWorkers helpers, which sleep between copies.
class CopyTeam {
public:
    ~CopyTeam();
    void copy(void* dst, const void* src, size_t n);

private:
    static constexpr int kWorkers = 3;
    // one copy: each thread takes part `i` of the workers + 1 parts
    struct Job {
        char* dst = nullptr;
        const char* src = nullptr;
        size_t n = 0;
    };
    void part(const Job& j, int i) const;
    void work(int i);
    std::vector<std::thread> threads_;
    std::mutex mu_;
    std::condition_variable cv_;
    Job job_;
    std::atomic<unsigned> turn_{0};    // copies started
    std::atomic<int> left_{0};         // helpers still at the current one
    std::atomic<bool> stop_{false};
    bool started_ = false;
};

class HostCopy {
public:
    ~HostCopy();
    // dst (host) <- src (device) after the stream's work so far; waits for it.
    hipError_t to_host(void* dst, const void* src, size_t n, hipStream_t s);
    // dst (device) <- src (host), in stream order; a page-locked src may still be read until
    // the stream has been waited for.
    hipError_t to_device(void* dst, const void* src, size_t n, hipStream_t s);

private:
    static constexpr int kRing = 4;
    static constexpr size_t kChunk = (size_t)4 << 20;    // bytes of a ring buffer
    static constexpr size_t kLeast = (size_t)128 << 10;  // smaller copies go to the runtime
    struct Slot {
        char* p = nullptr;
        hipEvent_t done = nullptr;
        bool busy = false;  // `done` has been recorded and not waited for
    };
    bool ready(int slots, hipStream_t st);
    hipError_t wait(Slot& s);
    Slot ring_[kRing];
    CopyTeam team_;
};

}  // namespace ptk
