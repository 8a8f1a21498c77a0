// CPU stand-in for the part of the HIP runtime that host_copy.hip uses, with
// entries that tests/test_host_copy.py calls.  Copies happen at once; a
// stream marked busy holds back whoever waits for it or for an event on it.
#include <atomic>
#include <chrono>
#include <cstdlib>
#include <cstring>
#include <mutex>
#include <set>
#include <thread>

#include "host_copy.h"

namespace {
std::atomic<bool> g_busy[2];
std::atomic<int> g_waiting[2];
std::atomic<long> g_direct;  // copies whose destination is not pinned memory of hipHostMalloc
std::mutex g_m;
std::set<const char*> g_known;  // caller's memory that the runtime knows
char* g_pinned = nullptr;
size_t g_pinned_bytes = 0;

void wait_for(int s) {
    g_waiting[s]++;
    while (g_busy[s].load()) std::this_thread::sleep_for(std::chrono::milliseconds(1));
    g_waiting[s]--;
}
int index_of(hipStream_t s) { return (int)((size_t)s) - 1; }
}  // namespace

struct ihipEvent_t {
    int stream = -1;
};

extern "C" {
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError(void) { return hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
    *p = g_pinned = (char*)malloc(n);
    g_pinned_bytes = n;
    return g_pinned ? hipSuccess : hipErrorOutOfMemory;
}
hipError_t hipHostFree(void* p) {
    free(p);
    g_pinned = nullptr;
    g_pinned_bytes = 0;
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = new ihipEvent_t;
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    e->stream = index_of(s);
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
    wait_for(e->stream);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) {
    wait_for(index_of(s));
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t n, hipMemcpyKind, hipStream_t) {
    if ((char*)dst < g_pinned || (char*)dst >= g_pinned + g_pinned_bytes) g_direct++;
    memcpy(dst, src, n);
    return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
    std::lock_guard<std::mutex> lock(g_m);
    memset(a, 0, sizeof(*a));
    a->type = g_known.count((const char*)p) ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
    return hipSuccess;
}

// stream 0 or 1
int hc_read(void* dst, const void* src, size_t bytes, int stream) {
    return (int)desalm::host_read(dst, src, bytes, (hipStream_t)(size_t)(stream + 1), 0);
}
void hc_users(int change) { desalm::host_read_users(change); }
void hc_busy(int stream, int on) { g_busy[stream].store(on != 0); }
int hc_waiting(int stream) { return g_waiting[stream].load(); }
long hc_direct(void) { return g_direct.exchange(0); }
void hc_know(const void* p) {
    std::lock_guard<std::mutex> lock(g_m);
    g_known.insert((const char*)p);
}
}
