// Device-to-host copies into pageable memory (host_copy.hip).
#pragma once
#include <hip/hip_runtime_api.h>
#include <stddef.h>

namespace desalm {

// copy from device memory to host memory, after the work on s, complete on
// return; and the number of contexts that keep its pinned ring alive
hipError_t host_read(void* dst, const void* src, size_t bytes, hipStream_t s, int device);
void host_read_users(int change);

}  // namespace desalm
