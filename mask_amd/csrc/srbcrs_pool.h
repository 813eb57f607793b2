// Device memory of plans and conversions, kept for reuse.
//
// hipMalloc and hipFree of the arrays of one conversion (2.5 GB for a graph
// of 11.7 M edges) cost more than its kernels: 8 ms at best, 40 ms where the
// freed pages are not handed out again at once.  Freed blocks are therefore
// kept, up to kPoolBytes per process, and given back when that is exceeded
// (the ones unused longest first), when an allocation of this library fails,
// and by pool_release.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace srbcrs {

constexpr size_t kPoolBytes = size_t(4) << 30;

// Device memory on the current device, at least `bytes`; null: none left.
// A block taken from the pool is idle: no queued work uses it.  fresh: always
// through hipMalloc, which graph capture refuses, and of just this size.  why
// receives HIP's reason where it is null.
void* pool_alloc(size_t bytes, bool fresh = false, hipError_t* why = nullptr);
// Give a block back.  No queued work may still use it, on any stream.
void pool_free(void* p);
// hipFree of a block from pool_alloc.
void pool_drop(void* p);
// hipFree of all kept blocks of a device (-1: of all devices).
void pool_release(int device);

}  // namespace srbcrs
