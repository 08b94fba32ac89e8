// Copies between device memory and ordinary (pageable) host memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace aslhip {

// Every object that transfers (lattice, trainer) holds one reference; the
// staging buffers go back with the last one.
void transfer_hold();
void transfer_drop();

// Copies n bytes after the work queued on s; returns when dst holds them.
// launches: those queued since the host last waited for s, 0 after this call has.
hipError_t to_host(void *dst, const void *src, size_t n, hipStream_t s, int *launches = nullptr);
// Copies n bytes; returns when src may change (wait false: once s has been
// waited for, which is the caller's to do), work queued on s afterwards sees dst.
hipError_t to_device(void *dst, const void *src, size_t n, hipStream_t s, bool wait = true);

}  // namespace aslhip
