// sfv_transfer.hpp — device-to-host copies into pageable memory
// (sfv_transfer.hip).
#pragma once

#include <hip/hip_runtime.h>

#include <cstddef>

namespace sfv {

// Copy n bytes from the current device to dst after the work queued on st;
// returns when they are there.  dst may be any memory a plain copy could write,
// pinned and device memory included.  Any number of threads may copy at once.
hipError_t copy_to_host(void* dst, const void* src, size_t n, hipStream_t st);

// Each handle and each server holds the staging memory; what the last of them leaves is one
// lane at most (sfv_transfer.hip).
void staging_retain();
void staging_release();
// Lanes that hold memory at present.
int staging_lanes();

}  // namespace sfv
