// Device memory. The blocks of closed contexts and of their calls' transient staging are kept for later allocations of
// about their size, up to kDevCacheBytes per process: a context of 29079 nodes per partition with k = 100 holds 125
// blocks (450 MB), whose hipMalloc and hipFree took 2.4 and 9.5 ms of a 37 ms detection when graphs are worked on one
// after another. The cache is emptied with the last live context and by mmsb_release (release_device_cache), and before
// any allocation of the library fails: all of them come through dev_alloc or dev_malloc. An allocator of the calling
// program does not see the kept blocks as free. What a live context gives up to save memory is not kept (dev_release).
#pragma once

#include <hip/hip_runtime_api.h>

#include <cstddef>

namespace mmsb {

constexpr size_t kDevCacheBytes = (size_t)1 << 30;

// hipMalloc on the current device. The contents are undefined.
hipError_t dev_alloc(void** p, size_t bytes);
// Gives back a block of dev_alloc (null: nothing). No work that uses it may be in flight on any stream: it may be
// handed to another context, thread or stream at once.
void dev_free(void* p);
// Gives a block of dev_alloc back to the device (hipFree).
void dev_release(void* p);
// hipMalloc on the current device, for blocks that are freed with hipFree.
hipError_t dev_malloc(void** p, size_t bytes);
template <typename T>
hipError_t dev_malloc(T** p, size_t bytes) { return dev_malloc(reinterpret_cast<void**>(p), bytes); }
// Bytes kept for the current device, part of what a new allocation can use beyond hipMemGetInfo's free bytes.
size_t dev_cached_bytes();
void release_device_cache();

}  // namespace mmsb
