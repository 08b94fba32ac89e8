// Device memory.
#pragma once
#include <hip/hip_runtime.h>

#include <cstddef>

namespace aslhip {

// A buffer that one call of a lattice needs, kept between calls (allocating and
// freeing 45 MB took 0.4 ms of a read of 1.6): at most KEEP bytes each and
// KEEP_ALL in the process, given back when an allocation fails.
struct Scratch {
  void *p = nullptr;
  size_t bytes = 0;
  bool busy = false;             // a call has it
  hipEvent_t used = nullptr;     // the end of the last call's work, if the call did not wait for it
  Scratch *prev = nullptr, *next = nullptr;  // those that hold a buffer
};
constexpr size_t KEEP = 256u << 20, KEEP_ALL = 512u << 20;

// A buffer of n bytes, from s or allocated.
hipError_t scratch_take(Scratch &s, size_t n, void **p);
// Ends the call's use of it; pending: work on this stream still uses it.
hipError_t scratch_give(Scratch &s, size_t n, void *p, hipStream_t pending = nullptr);
void scratch_drop(Scratch &s);

// A failed allocation gives the kept buffers back and tries once more; then it is
// reported by its return value alone: the runtime would also keep it as the
// thread's last error, which the next launch on this thread would report as its own.
hipError_t device_alloc_bytes(void **p, size_t n);
template <class T>
hipError_t device_alloc(T **p, size_t n) {
  return device_alloc_bytes(reinterpret_cast<void **>(p), n);
}

}  // namespace aslhip
