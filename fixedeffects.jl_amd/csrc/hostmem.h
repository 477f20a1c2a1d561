// hostmem.h -- memory a handle takes and gives back (a bounded pool of device
// blocks shared by the handles of a process), and copies between the caller's
// pageable memory and the device.
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>
#include <cstdint>

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

// FEHIP_DEVICE_MB in the environment limits what blocks may come to per device,
// in MB; beyond it a call fails as it does where the device has no room.  Read
// here, once a call of the C-ABI.
void pool_read_limit();

// Frees the blocks the pool keeps, of every device.
void pool_trim();

// Pageable host memory to the device: the source has been read when the call
// returns, the device has it in stream order.  Large copies go through pinned
// buffers filled by a few threads (see hostmem.hip).
hipError_t copy_in(void *dst, const void *src, size_t bytes, hipStream_t st);

// Device to pageable host memory: written when the call returns.
hipError_t copy_out(void *dst, const void *src, size_t bytes, hipStream_t st);

// 1-based refs to 0-based int32 on the device, narrowed on the way; *bad is
// set when one lies outside 1..nlev.  False (nothing done) for arrays small
// enough that the runtime's copy and a kernel take less time.
bool copy_in_refs(int32_t *dst, const int64_t *src, int64_t n, int64_t nlev, bool *bad, hipStream_t st,
                  hipError_t *err);
inline bool copy_in_refs(int32_t *, const int32_t *, int64_t, int64_t, bool *, hipStream_t, hipError_t *) {
    return false;  // 4-byte refs: nothing to narrow
}

}  // namespace fehip
