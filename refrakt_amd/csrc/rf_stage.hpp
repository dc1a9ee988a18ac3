// Device-to-host copies into ordinary (pageable) memory.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>

namespace rfh {

// Copies n bytes of device memory to `host` behind everything on stream s and
// returns when they are there.
hipError_t download(void* host, const void* device, size_t n, hipStream_t s);

// Contexts hold the staging buffers and copying threads alive: each context
// calls stage_hold once and stage_release when it goes; the last one to go
// frees them.
void stage_hold();
void stage_release();

}  // namespace rfh
