// Runs the pinned-ring copies (pathtracer_amd/csrc/hostcopy.cpp) on the CPU against
// stand-ins for the HIP calls they make: "device" memory is host memory, copies happen
// at once, and the stand-ins note which addresses the runtime was given.
//
// Usage: hostcopy_sim kind n [stream_device]    kind: pageable | pinned | device | managed
// Checks the bytes both ways, and how they went: pageable memory through the ring (the
// runtime never sees the caller's address), anything the runtime knows in one copy of
// its own. As in HIP, an event belongs to the device that was current when it was made and
// can be recorded only on that device's streams; the stream here is one of stream_device,
// the current device 0, which the copies must leave so. Prints "ok" or the first violation, and exits 0 or 1.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "hostcopy.hpp"

static const char* g_known = nullptr;  // the caller's buffer, when the runtime knows it
static size_t g_len = 0;
static hipMemoryType g_type = hipMemoryTypeUnregistered;
static int g_current = 0, g_stream_device = 0;
static std::vector<std::pair<const void*, size_t>> g_host_side;  // host addresses given to the runtime

extern "C" {
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::memset(a, 0, sizeof *a);
    a->type = hipMemoryTypeUnregistered;
    if (g_known && p >= g_known && p < g_known + g_len) a->type = g_type;
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind kind, hipStream_t) {
    g_host_side.emplace_back(kind == hipMemcpyDeviceToHost ? dst : src, n);
    std::memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new int(g_current));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<int*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
    return *reinterpret_cast<int*>(e) == g_stream_device ? hipSuccess : hipErrorInvalidHandle;
}
hipError_t hipGetDevice(int* d) {
    *d = g_current;
    return hipSuccess;
}
hipError_t hipSetDevice(int d) {
    g_current = d;
    return hipSuccess;
}
hipError_t hipStreamGetDevice(hipStream_t, hipDevice_t* d) {
    *d = g_stream_device;
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = std::malloc(n);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    std::free(p);
    return hipSuccess;
}
hipError_t hipGetLastError(void) { return hipSuccess; }
}

static int fail(const char* what) {
    std::printf("FAIL %s\n", what);
    return 1;
}

int main(int argc, char** argv) {
    if (argc != 3 && argc != 4) return 2;
    if (argc == 4) g_stream_device = std::atoi(argv[3]);
    const std::string kind = argv[1];
    const size_t n = (size_t)std::atoll(argv[2]);
    std::vector<char> caller(n + 1), dev(n + 1);
    for (size_t i = 0; i < n; ++i) caller[i] = (char)(i * 2654435761u >> 24);
    const std::vector<char> want = caller;
    if (kind != "pageable") {
        g_known = caller.data();
        g_len = n;
        g_type = kind == "pinned" ? hipMemoryTypeHost : kind == "device" ? hipMemoryTypeDevice : hipMemoryTypeManaged;
    }
    const bool ring = kind == "pageable" && n >= ((size_t)128 << 10);
    auto direct_once = [&] { return g_host_side.size() == 1 && g_host_side[0].first == caller.data() && g_host_side[0].second == n; };
    auto sees_caller = [&] {
        for (auto& h : g_host_side)
            if (h.first >= caller.data() && h.first < caller.data() + n) return true;
        return false;
    };
    ptk::HostCopy hc;
    for (int round = 0; round < 2; ++round) {
        g_host_side.clear();
        if (hc.to_device(dev.data(), caller.data(), n, nullptr) != hipSuccess) return fail("to_device");
        if (std::memcmp(dev.data(), want.data(), n)) return fail("to_device: bytes");
        if (ring ? sees_caller() : !direct_once()) return fail("to_device: wrong way");
        std::memset(caller.data(), 0, n);
        g_host_side.clear();
        if (hc.to_host(caller.data(), dev.data(), n, nullptr) != hipSuccess) return fail("to_host");
        if (std::memcmp(caller.data(), want.data(), n)) return fail("to_host: bytes");
        if (ring ? sees_caller() : !direct_once()) return fail("to_host: wrong way");
    }
    if (g_current != 0) return fail("the current device changed");
    std::printf("ok\n");
    return 0;
}
