#include "memory.hpp"

#include <mutex>

namespace aslhip {
namespace {

std::mutex keep_mu;       // the list and all of every Scratch
Scratch *kept = nullptr;  // the buffers, those kept last first
size_t kept_bytes = 0;

// Under keep_mu.  (Waits for an event, not for the stream, which another thread
// may be capturing.)
void release(Scratch &s) {
  if (s.used) (void)hipEventSynchronize(s.used);
  (void)hipFree(s.p);
  kept_bytes -= s.bytes;
  s.p = nullptr;
  s.bytes = 0;
  (s.prev ? s.prev->next : kept) = s.next;
  if (s.next) s.next->prev = s.prev;
  s.prev = s.next = nullptr;
}

bool release_idle() {
  std::lock_guard<std::mutex> lock(keep_mu);
  bool any = false;
  for (Scratch *s = kept, *next; s; s = next) {
    next = s->next;
    if (s->busy) continue;
    release(*s);
    any = true;
  }
  return any;
}

}  // namespace

hipError_t device_alloc_bytes(void **p, size_t n) {
  hipError_t e = hipMalloc(p, n);
  if (e == hipErrorOutOfMemory && release_idle()) {
    (void)hipGetLastError();
    e = hipMalloc(p, n);
  }
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
  }
  return e;
}

hipError_t scratch_take(Scratch &s, size_t n, void **p) {
  {
    std::lock_guard<std::mutex> lock(keep_mu);
    if (s.p && !s.busy && s.bytes >= n) {
      s.busy = true;
      *p = s.p;
      return hipSuccess;
    }
  }
  return device_alloc_bytes(p, n);
}

hipError_t scratch_give(Scratch &s, size_t n, void *p, hipStream_t pending) {
  std::unique_lock<std::mutex> lock(keep_mu);
  const bool had = p == s.p;
  bool keep = had || (!s.p && n <= KEEP && kept_bytes + n <= KEEP_ALL);
  hipError_t e = hipSuccess;
  if (keep && pending) {
    if (!s.used) e = hipEventCreateWithFlags(&s.used, hipEventDisableTiming);
    if (e == hipSuccess) e = hipEventRecord(s.used, pending);
    if (e != hipSuccess) {  // wait instead
      (void)hipGetLastError();
      e = hipStreamSynchronize(pending);
    }
  }
  if (had) {
    s.busy = false;
  } else if (keep) {
    s.p = p;
    s.bytes = n;
    s.next = kept;
    if (kept) kept->prev = &s;
    kept = &s;
    kept_bytes += n;
  }
  lock.unlock();
  if (keep) return e;
  if (pending) e = hipStreamSynchronize(pending);
  const hipError_t f = hipFree(p);
  return e != hipSuccess ? e : f;
}

void scratch_drop(Scratch &s) {
  std::lock_guard<std::mutex> lock(keep_mu);
  if (s.p) release(s);
  if (s.used) (void)hipEventDestroy(s.used);
  s.used = nullptr;
}

}  // namespace aslhip
