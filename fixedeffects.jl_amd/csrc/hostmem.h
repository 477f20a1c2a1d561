// hostmem.h -- memory a handle takes and gives back (a bounded pool of device
// blocks shared by the handles of a process).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace fehip {

// A block of at least `bytes` on the current device, and its real size and
// device (for pool_put).  Its contents are undefined.  Blocks come from those
// given back before where one of the same size class is there, else from
// hipMalloc (after emptying the pool if that fails).
hipError_t pool_get(size_t bytes, void **ptr, size_t *size, int *device);

// Gives a block back.  No work that uses it may be pending on any stream.
// The pool keeps at most kPoolBytes per device and frees the rest.
void pool_put(void *ptr, size_t size, int device);

constexpr size_t kPoolBytes = size_t(4) << 30;

}  // namespace fehip
