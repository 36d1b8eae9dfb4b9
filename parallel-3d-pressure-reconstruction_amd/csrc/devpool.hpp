// Device memory of the library's buffers: blocks given up by one buffer serve
// the next one, within a bound.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace omni3d {

// A block of at least `bytes` on the current device; *cap its size, *dev the
// device.  Contents undefined, as hipMalloc's.
hipError_t device_alloc(void** p, size_t bytes, size_t* cap, int* dev);
// Gives a block up.  Work queued on any stream may still use it: it serves
// again only after the device has been waited for.
void device_free(void* p, size_t cap, int dev);
// Returns the unused blocks of every device to the driver; bytes returned.
size_t device_release_unused();

}  // namespace omni3d
