// host_copy.hip -- device-to-host copies into pageable memory.
//
// A plain copy of a field into a caller's array runs at 10 GB/s into fresh
// pages and 18 GB/s into resident ones: the runtime moves it through pinned
// memory with one thread, which also takes the page faults.  host_read moves
// it in chunks through a pinned ring instead; the DMA of the next chunks runs
// while several threads copy the chunks that have arrived.  128 MB (q of a
// 193x129x129 block) into fresh pages: 11.9 -> 3.7 ms with four threads (two: 5.9,
// eight: 3.4; 3.3 is the link).  The count does not follow the caller's CPU
// affinity: the four threads of a process held to two CPUs take 6.1 ms, to one
// 10.1 ms (resident pages 4.2 and 5.0), a plain copy there 12.4 ms (7.4).
// Host-to-device copies are left to the runtime (30 GB/s).
//
// The ring is the process's: kSlots chunks of pinned memory, allocated by the
// first large read, used by one read at a time (a mutex, taken once the read's
// stream is idle), and freed when the last context is finalized (a program
// without contexts, which may read through desalm_gtsv_batch, keeps its 16 MiB
// until it ends).
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

#include "host_copy.h"

namespace desalm {

namespace {

constexpr size_t kChunk = (size_t)2 << 20;
constexpr int kWorkers = 4;
constexpr int kSlots = 2 * kWorkers;           // chunk c uses slot c % kSlots, and worker c % kWorkers alone
constexpr size_t kSmall = (size_t)4 << 20;     // below: one plain copy

std::mutex g_mutex;
char* g_ring = nullptr;
int g_users = 0;  // contexts

// chunks w, w + kWorkers, ... of a read: wait for the chunk's DMA, copy it
// out, start the DMA that reuses its slot
void copy_chunks(int w, int device, char* dst, const char* src, size_t bytes, hipStream_t s, hipEvent_t* ev,
                 std::atomic<int>* status) {
    if (hipSetDevice(device) != hipSuccess) {
        status->store((int)hipErrorInvalidDevice);
        return;
    }
    const size_t n = (bytes + kChunk - 1) / kChunk;
    for (size_t c = (size_t)w; c < n && status->load() == (int)hipSuccess; c += kWorkers) {
        const int slot = (int)(c % kSlots);
        hipError_t e = hipEventSynchronize(ev[slot]);
        if (e == hipSuccess) {
            memcpy(dst + c * kChunk, g_ring + slot * kChunk, std::min(kChunk, bytes - c * kChunk));
            const size_t next = c + kSlots;
            if (next < n) {
                e = hipMemcpyAsync(g_ring + slot * kChunk, src + next * kChunk,
                                   std::min(kChunk, bytes - next * kChunk), hipMemcpyDeviceToHost, s);
                if (e == hipSuccess) e = hipEventRecord(ev[slot], s);
            }
        }
        if (e != hipSuccess) status->store((int)e);
    }
}

// Pinned, managed or device memory: the DMA writes it in place (128 MB into
// pinned memory 2.36 ms, through the ring 3.28).
bool known_to_runtime(const void* p) {
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
        (void)hipGetLastError();
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t host_read(void* dst, const void* src, size_t bytes, hipStream_t s, int device) {
    auto plain = [&] {
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    };
    if (bytes < kSmall || known_to_runtime(dst)) return plain();
    // the stream's earlier work is waited for outside the lock, which then
    // covers the copy alone: a read behind pending kernels does not hold up
    // reads of other contexts or the end of one
    const hipError_t before = hipStreamSynchronize(s);
    if (before != hipSuccess) return before;
    std::lock_guard<std::mutex> lock(g_mutex);
    if (!g_ring && hipHostMalloc((void**)&g_ring, kSlots * kChunk, hipHostMallocPortable) != hipSuccess) {
        g_ring = nullptr;
        (void)hipGetLastError();
        return plain();
    }
    hipEvent_t ev[kSlots] = {};
    std::atomic<int> status{(int)hipSuccess};
    for (int k = 0; k < kSlots && status.load() == (int)hipSuccess; k++)
        status.store((int)hipEventCreateWithFlags(&ev[k], hipEventDisableTiming));
    const size_t n = (bytes + kChunk - 1) / kChunk;
    for (size_t c = 0; c < n && c < (size_t)kSlots && status.load() == (int)hipSuccess; c++) {
        hipError_t e = hipMemcpyAsync(g_ring + c * kChunk, (const char*)src + c * kChunk,
                                      std::min(kChunk, bytes - c * kChunk), hipMemcpyDeviceToHost, s);
        if (e == hipSuccess) e = hipEventRecord(ev[c], s);
        status.store((int)e);
    }
    // a class of chunks whose thread cannot be started is copied here
    std::thread t[kWorkers];
    bool here[kWorkers] = {true};
    for (int w = 1; w < kWorkers; w++) {
        here[w] = false;
        try {
            t[w] = std::thread(copy_chunks, w, device, (char*)dst, (const char*)src, bytes, s, ev, &status);
        } catch (...) {
            here[w] = true;
        }
    }
    for (int w = 0; w < kWorkers; w++)
        if (here[w]) copy_chunks(w, device, (char*)dst, (const char*)src, bytes, s, ev, &status);
    for (int w = 1; w < kWorkers; w++)
        if (t[w].joinable()) t[w].join();
    // after an error a DMA into the ring may still be under way
    if (status.load() != (int)hipSuccess) (void)hipStreamSynchronize(s);
    for (int k = 0; k < kSlots; k++)
        if (ev[k]) (void)hipEventDestroy(ev[k]);
    return (hipError_t)status.load();
}

void host_read_users(int change) {
    std::lock_guard<std::mutex> lock(g_mutex);
    g_users += change;
    if (g_users == 0 && g_ring) {
        (void)hipHostFree(g_ring);
        g_ring = nullptr;
    }
}

}  // namespace desalm
